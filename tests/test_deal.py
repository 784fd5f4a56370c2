"""The numbers behind the work order of a launch (csrc/omni_attn_deal.hpp, compiled alone): a division by a
multiplication gives the quotient for every n < 2^31, and the last group of an XCD has the slabs that are left."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "omni-attention_amd", "csrc")

PROGRAM = r"""
#include "omni_attn_deal.hpp"
#include <cstdio>
#include <random>
using namespace omni_attn;
static long long wrong = 0;
static void check(uint32_t n, uint32_t d) {
  if (divide(n, fast_div(d)) != n / d) {
    if (wrong++ < 5) printf("%u / %u = %u\n", n, d, divide(n, fast_div(d)));
  }
}
int main() {
  const uint32_t top = 0x7fffffff;
  std::mt19937_64 gen(1);
  auto around = [&](uint32_t d) {
    for (uint32_t m : {1u, 2u, 3u, 1000u, top / d}) {
      const uint64_t p = uint64_t(m) * d;
      for (long long n : {(long long)p - 1, (long long)p, (long long)p + 1})
        if (n >= 0 && n <= top) check(uint32_t(n), d);
    }
    check(0, d);
    check(top, d);
    for (int i = 0; i < 50; ++i) check(uint32_t(gen() & top), d);
  };
  for (uint32_t d = 1; d < 5000; ++d) around(d);
  for (int b = 0; b < 31; ++b)
    for (long long d : {(1LL << b) - 1, 1LL << b, (1LL << b) + 1})
      if (d > 0) around(uint32_t(d));
  for (int i = 0; i < 5000; ++i) around(uint32_t(gen() & top) | 1);
  around(top);
  for (int slabs = 1; slabs <= 70; ++slabs)
    for (int xcds : {1, 8})
      for (int parts : {1, 2, 8})
        for (int group : {1, 2, 3, 5, 8, 100}) {
          const DealPlan d = plan_deal(slabs, parts, xcds, group, 13, 5);
          long long all = 0;
          for (int x = 0; x < xcds; ++x) {
            const int here = d.slabs + (x < d.one_more);
            all += here;
            int left = here;
            while (left > group) left -= group;
            if (left > 0)  // the workgroups of the last group, in ranks of `left`
              for (uint32_t n = 0; n < 3u * left; ++n) wrong += divide(n, left == group ? d.group : d.last[x < d.one_more]) != n / left;
          }
          wrong += all != slabs * parts || (1 << d.part_shift) != parts || d.part_tiles != (13 + parts - 1) / parts;
        }
  printf("wrong %lld\n", wrong);
  return wrong != 0;
}
"""


def test_divisions_of_the_work_order(tmp_path):
    source, program = tmp_path / "deal.cpp", tmp_path / "deal"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", CSRC, str(source), "-o", str(program)], check=True)
    run = subprocess.run([str(program)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
