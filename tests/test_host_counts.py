"""The pieces of host memory behind the mask builder's counts (csrc/omni_attn_host_counts.hpp, compiled alone with a stream
that is played by the host): what calls take is given back, also by calls that fail, and never handed out while a kernel may
write it."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "omni-attention_amd", "csrc")

PROGRAM = r"""
#include "omni_attn_host_counts.hpp"
#include <cstdio>
#include <cstdlib>
#include <memory>
#include <set>
struct Host {
  struct Stream { bool ends = true, fails = false; };
  static inline int held = 0, drains = 0;
  static inline std::set<void*> stuck;
  static void* allocate(size_t n) { ++held; return std::malloc(n); }
  static void release(void* p) { --held; std::free(p); }
  static bool running(Stream s) { if (s.fails) throw std::runtime_error("stream"); return !s.ends; }
  static bool drain(Stream s) { ++drains; return s.ends && !s.fails; }
};
typedef omni_attn::HostCounts<Host, 20> Counts;
#define CHECK(x) if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; }
static void post(Counts& c, int tag, int n) {
  for (int i = 0; i < n; ++i) c.memory()[i] = uint32_t(Counts::word_of(tag)) | uint32_t(i);
}
int main() {
  for (int i = 0; i < 9000; ++i) {  // counts and totals in turn (the tags begin again twice); one piece does for all
    Counts c;
    const int tag = c.next_tag({});
    CHECK(tag > 0 && tag < 4096);
    if (i % 3 == 0) {
      c.memory()[0] = uint32_t(Counts::word_of(tag % 4095 + 1)) | 5u;  // (a total may look like a later call's count)
      c.memory()[1] = uint32_t(Counts::word_of(tag));
      CHECK(uint32_t(c.wait_total(tag)) == (uint32_t(Counts::word_of(tag % 4095 + 1)) | 5u));
    } else {
      for (int w = 0; w < 7; ++w) CHECK(int(c.memory()[w] >> 20) != tag);
      post(c, tag, 7);
      CHECK(c.wait(tag, 7) == 21);
    }
  }
  CHECK(Host::held == 1 && Host::drains == 0);
  for (int i = 0; i < 5000; ++i) {  // calls that fail while the kernel runs, in the wait, and refused ones
    try {
      Counts c;
      const int tag = c.next_tag({});
      for (int w = 0; w < 7; ++w) CHECK(int(c.memory()[w] >> 20) != tag);
      post(c, tag, i % 3);
      if (i % 2) throw std::runtime_error("no memory for the lists");
      c.wait(tag, 7);
      CHECK(false);
    } catch (const std::runtime_error&) {
    }
    CHECK(Host::held == 1 && Host::drains == i + 1);
  }
  for (int i = 0; i < 3; ++i) {  // a stream that cannot be waited for keeps its memory; it is not handed out again
    Host::Stream s;
    s.fails = i == 0;
    s.ends = false;
    Counts c;
    CHECK(Host::stuck.insert(c.memory()).second);
    c.next_tag(s);
  }
  CHECK(Host::held == 3);
  {
    std::vector<std::unique_ptr<Counts>> many;  // calls of many threads at once: at most kKeep pieces stay
    for (int i = 0; i < 40; ++i) {
      many.emplace_back(new Counts);
      CHECK(Host::stuck.count(many.back()->memory()) == 0);
      for (int j = 0; j < i; ++j) CHECK(many[j]->memory() != many[i]->memory());
    }
    CHECK(Host::held == 43);
  }
  CHECK(Host::held == 3 + int(Counts::kKeep));
}
"""


def test_pieces_are_given_back(tmp_path):
    source, program = tmp_path / "counts.cpp", tmp_path / "counts"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(source), "-o", str(program), "-lpthread"], check=True)
    run = subprocess.run([str(program)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
