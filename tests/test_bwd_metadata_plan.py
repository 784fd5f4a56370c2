"""How the dK/dV kernel divides a compute unit's LDS between a slab's metadata and its table of steps (host
arithmetic of csrc/omni_attn_bwd_plan.hpp, compiled alone): the table never costs a workgroup that the metadata
alone would leave room for, and what is planned fits."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "omni-attention_amd", "csrc")

PROGRAM = r"""
#include "omni_attn_bwd_plan.hpp"
#include <cstdio>
#include <cstdlib>
int main(int argc, char** argv) {
  const size_t fixed = size_t(atol(argv[1]));
  const int fit = atoi(argv[2]), steps = atoi(argv[3]);
  const long long many[] = {16384, 100001, 0x7fffffff};
  for (long long i = 1; i < 9003; ++i) {
    const long long n = i < 9000 ? i : many[i - 9000];
    const auto p = omni_attn::dkdv_plan(fixed, fit, n, steps);
    printf("%lld %d %d %zu\n", n, p.words, p.steps, p.bytes);
  }
}
"""


def shapes():
    """(LDS of tiles, hand-over and row offsets; workgroups per compute unit by registers; steps per query block)
    of every instance: key groups x groups x rows per step at each head dimension."""
    for D in (32, 64, 128):
        for key_groups, groups, step in ((4, 1, 64 if D == 128 else 32), (2, 1, 32), (2, 2, 32), (1, 4, 32)):
            if (key_groups, groups) == (1, 4) and D == 128:
                continue
            fixed = groups * (6 * step * D * 2 + 2 * key_groups * (step // 32) * 2 * 64 * 16 + 6 * step * 4)
            fit = {128: 2, 64: 4, 32: 5}[D] * 256 // (key_groups * 128 * groups)
            for QB in (64, 128):
                yield pytest.param(fixed, fit, QB // step, id=f"D{D}-{key_groups}x{groups}-QB{QB}")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, "-o", str(d / "plan"), str(d / "plan.cpp")], check=True)
    return str(d / "plan")


@pytest.mark.parametrize("fixed,fit,steps_per_block", shapes())
def test_table_takes_what_the_metadata_leaves(program, fixed, fit, steps_per_block):
    lds, unit = 160 * 1024, 1280
    resident = lambda size: min(fit, lds // (-(-size // unit) * unit))
    out = subprocess.run([program, str(fixed), str(fit), str(steps_per_block)], check=True, capture_output=True, text=True)
    rows = [tuple(map(int, line.split())) for line in out.stdout.splitlines()]
    assert len(rows) == 9002
    for n_words, words, steps, size in rows:
        assert size <= lds and size >= fixed + 12 * words + 8 * steps + 12
        # as many workgroups as metadata alone (12 bytes per word, at most 4096 words or what fits) allow
        alone = fixed + 12 * min(n_words, 4096, (lds - fixed) // 12)
        assert resident(size) >= resident(alone), (n_words, words, steps)
        # a window has all words where they fit, and about equal windows otherwise
        windows = -(-n_words // words)
        assert words >= min(n_words, 250) and (windows == 1 or words <= n_words // windows + 2)
        assert min(128, words * steps_per_block) <= steps <= max(128, words * steps_per_block)
