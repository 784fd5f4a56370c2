"""The rules that split the walks of launches with few rows (csrc/omni_attn_split_rules.hpp, compiled alone).  The
reason for a split is few rows and long lists: a launch with fewer rows of the same length, or with longer
lists of as many rows, is split too wherever this one is.  No line is drawn around a size."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "omni-attention_amd", "csrc")

PROGRAM = r"""
#include "omni_attn_split_rules.hpp"
#include <cstdio>
using namespace omni_attn;
int main() {
  for (int kind = 0; kind < 6; ++kind)    // forward: busiest XCD of 20, 34 and 60 tiles; dQ; dK/dV, soft-capped
    for (int D = 32; D <= 128; D *= 2)
      for (int block = 64; block <= 128; block += 64)
        for (int S = 64; S <= 16384; S += 64) {
          printf("%d %d %d %d ", kind, D, block, S);
          for (long long rows = 16; rows <= 4096; rows += 16) {
            bool split;
            if (kind < 3)
              split = fwd_choose_split(D, block, rows, S, kind == 0 ? 20 : (kind == 1 ? 34 : 60), 32) != FwdSplit::kNone;
            else if (kind == 3)
              split = bwd_choose_dq_split(D, block, rows, S) != FwdSplit::kNone;
            else
              split = bwd_choose_dkdv_split(D, kind == 5, rows, S) != DkdvSplit::kNone;
            putchar(split ? '1' : '0');
          }
          putchar('\n');
        }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, "-o", str(d / "rules"), str(d / "rules.cpp")], check=True)
    out = subprocess.run([str(d / "rules")], check=True, capture_output=True, text=True).stdout
    table = {}
    for line in out.splitlines():
        kind, D, block, S, bits = line.split()
        table.setdefault((int(kind), int(D), int(block)), []).append((int(S), bits))
    return table


@pytest.mark.parametrize("kind", range(6), ids=["fwd-one-round", "fwd-a-little-more", "fwd-more", "dq", "dkdv", "dkdv-capped"])
def test_fewer_rows_and_longer_lists_stay_split(rules, kind):
    for (k, D, block), by_length in rules.items():
        if k != kind:
            continue
        shortest = None  # rows (in steps of 16) up to which the shorter lists are split
        for S, bits in sorted(by_length):
            upto = bits.find("0") if "0" in bits else len(bits)
            assert "1" not in bits[upto:], (D, block, S, "rows")
            assert shortest is None or upto >= shortest, (D, block, S, "length")
            shortest = upto
        assert 0 < upto < len(bits)  # (with the longest lists: some, and not all)


def test_lengths_that_end_inside_a_block(tmp_path):
    """What is split for a length that fills its blocks is split the same way for one that does not; beyond that, fewer
    rows of the same length are split too, and so are one batch element's where a batch's are."""
    source, program = tmp_path / "ragged.cpp", tmp_path / "ragged"
    source.write_text(r"""
#include "omni_attn_split_rules.hpp"
using namespace omni_attn;
int main() {
  for (int D = 32; D <= 128; D *= 2)
    for (int S = 128; S <= 16384; S += 128)
      for (int batched = 0; batched < 2; ++batched) {
        bool all = false;  // from many rows to few: once split, always
        for (long long rows = 4096; rows >= 16; rows -= 16) {
          const long long busiest = (rows / 4 + 7) / 8;
          const FwdSplit plain = fwd_choose_split(D, 128, rows, S, busiest, 32);
          const FwdSplit ragged = fwd_choose_split(D, 128, rows, S, busiest, 32, true, true, batched);
          if (plain != FwdSplit::kNone && plain != ragged) return 1;
          const FwdSplit plain64 = fwd_choose_split(D, 64, rows, S, busiest, 32);
          if (plain64 != FwdSplit::kNone && plain64 != fwd_choose_split(D, 64, rows, S, busiest, 32, true, true, batched)) return 5;
          if (batched && ragged != FwdSplit::kNone && fwd_choose_split(D, 128, rows, S, busiest, 32, true, true, false) == FwdSplit::kNone) return 2;
          if (ragged != FwdSplit::kNone) all = true;
          else if (all && !batched && S >= 1152) return 3;
          if (bwd_choose_dq_split(D, 128, rows, S) != FwdSplit::kNone &&
              bwd_choose_dq_split(D, 128, rows, S) != bwd_choose_dq_split(D, 128, rows, S, true, batched)) return 4;
        }
      }
}
""")
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(source), "-o", str(program)], check=True)
    assert subprocess.run([str(program)]).returncode == 0


def test_order_line_of_a_form(tmp_path):
    """Workgroups from which on long lists go first: what two waves per SIMD make (one workgroup per compute unit for lone
    waves at head_dim 128), and never more than the LDS holds: per group K and V rows of a step, twice unless the group
    is one wave, and a mask byte per row and key."""
    source, program = tmp_path / "line.cpp", tmp_path / "line"
    source.write_text(r"""
#include "omni_attn_split_rules.hpp"
#include <cstdio>
using namespace omni_attn;
int main() {
  for (int s = 0; s < 5; ++s)
    for (int D = 32; D <= 128; D *= 2)
      for (int QB = 64; QB <= 128; QB += 64) printf("%d %d %d %d\n", s, D, QB, fwd_order_line(FwdSplit(s), D, QB, 32));
}
""")
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(source), "-o", str(program)], check=True)
    out = subprocess.run([str(program)], check=True, capture_output=True, text=True).stdout
    for line in out.splitlines():
        split, D, QB, workgroups = map(int, line.split())
        rows, groups = [(QB, 1), (32, 4), (64, 2), (64, 4), (128, 2)][split]
        step = 32 if D == 128 and rows != 128 else 64
        tiles = groups * ((1 if rows == 32 else 2) * 2 * step * D * 2 + rows * step)
        by_waves = 8 // (groups * rows // 32)
        assert by_waves * tiles <= 160 * 1024, (split, D, QB)
        assert workgroups == 32 * (1 if (split, D) == (1, 128) else by_waves), (split, D, QB)


# The launches of tests/test_gpu_split_walk.py's test of lengths that end inside a block: D, B, slabs per element, S, block,
# and the splits that it runs: of the forward, and of dQ (0 none, 2 and 4: 64- and 128-row groups).  The launch without
# any is one that the rule leaves whole.
RAGGED_LAUNCHES = [
    (128, 1, 32, 1160, 128, 2, 0), (128, 1, 24, 1610, 128, 4, 0), (128, 1, 16, 2700, 128, 4, 0),
    (128, 3, 8, 1630, 128, 2, 0), (64, 2, 16, 1500, 128, 2, 2), (64, 1, 16, 4400, 128, 2, 2), (32, 2, 24, 1300, 128, 0, 0),
    (32, 2, 20, 1300, 128, 2, 0), (64, 1, 37, 1300, 64, 0, 2), (32, 1, 32, 2950, 128, 2, 2), (128, 1, 32, 1170, 64, 2, 0),
    (128, 2, 12, 1500, 64, 2, 0), (64, 2, 12, 1500, 64, 2, 2), (32, 1, 32, 1900, 64, 2, 2)]


def test_keys_per_step_of_dq(tmp_path):
    """32 keys for 64-row blocks at head_dim 128 alone, in launches of many rows: more rows of the same length keep them, and so
    does a length that fills its blocks.  And the launches that a GPU test runs for their steps have them."""
    source, program = tmp_path / "step.cpp", tmp_path / "step"
    source.write_text(r"""
#include "omni_attn_split_rules.hpp"
using namespace omni_attn;
int main() {
  for (int S = 64; S <= 32768; S += 64) {
    int before[2] = {64, 64};
    for (long long rows = 16; rows <= 8192; rows += 16) {
      for (int ragged = 0; ragged < 2; ++ragged) {
        const int step = bwd_dq_step(128, 64, rows, S, ragged);
        if (step != 64 && step != 32) return 1;
        if (step > before[ragged]) return 2;
        before[ragged] = step;
        if (ragged && step == 32 && bwd_dq_step(128, 64, rows, S, false) != 32) return 3;
        if (bwd_dq_step(128, 128, rows, S, ragged) != 64 || bwd_dq_step(64, 64, rows, S, ragged) != 64) return 4;
        if (rows <= 1536 && step != 64) return 5;  // (two workgroups on a compute unit, and half as many again)
      }
    }
    if (before[0] != 32 || before[1] != 32) return 6;
  }
  for (int ragged = 0; ragged < 2; ++ragged)  // tests/test_gpu_whole_blocks.py
    if (bwd_dq_step(128, 64, 960, 256, ragged) != 64 || bwd_dq_step(128, 64, 2240, 256, ragged) != 32 ||
        bwd_choose_dq_split(128, 64, 960, 256, ragged, false) != FwdSplit::kNone) return 7;
}
""")
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(source), "-o", str(program)], check=True)
    assert subprocess.run([str(program)]).returncode == 0


def test_dealing_and_the_rules_that_look_at_it(tmp_path):
    """Uneven launches and soft-capped ones: what is split for a length that fills its blocks stays split; with 64-row
    blocks the forward is split for a length inside a block in even launches only, dQ in both (and where the even forward is);
    soft-capped dQ wherever the plain one is.  And the launches that a GPU test runs for their split have it."""
    source, program = tmp_path / "dealing.cpp", tmp_path / "dealing"
    launches = ",".join("{%s}" % ",".join(map(str, l)) for l in RAGGED_LAUNCHES)
    source.write_text(r"""
#include "omni_attn_split_rules.hpp"
#include <cstdio>
using namespace omni_attn;
int main() {
  const FwdSplit none = FwdSplit::kNone;
  bool uneven_dq = false;
  for (int D = 32; D <= 128; D *= 2)
    for (int QB = 64; QB <= 128; QB += 64)
      for (int S = QB; S <= 8192; S += QB)
        for (int slabs = 1; slabs <= 96; ++slabs)
          for (int batched = 0; batched < 2; ++batched) {
            const Dealing d = fwd_dealing(slabs, S, 8);
            const long long rows = (long long)slabs * (S / 32);
            const FwdSplit whole = fwd_choose_split(D, QB, rows, S, d.busiest, 32, false, d.even, batched);
            const FwdSplit ragged = fwd_choose_split(D, QB, rows, S, d.busiest, 32, true, d.even, batched);
            const FwdSplit if_even = fwd_choose_split(D, QB, rows, S, d.busiest, 32, true, true, batched);
            if (whole != none && whole != ragged) return 1;
            if (QB == 64 && !d.even && ragged != whole) return 2;
            const FwdSplit dq = bwd_choose_dq_split(D, QB, rows, S, true, batched, false);
            if (bwd_choose_dq_split(D, QB, rows, S) != none && dq == none) return 3;
            if (D == 64 && if_even != none && whole == none && dq != FwdSplit::kRows64x2) return 4;
            if (dq != none && bwd_choose_dq_split(D, QB, rows, S, true, batched, true) == none) return 5;
            if (D == 64 && QB == 64 && !d.even && ragged == none && dq != none && bwd_choose_dq_split(D, QB, rows, S) == none)
              uneven_dq = true;
          }
  if (!uneven_dq) return 6;
  const int launches[][7] = {""" + launches + r"""};
  for (const auto& l : launches) {
    const int D = l[0], slabs = l[1] * l[2], QB = l[4], S = (l[3] + QB - 1) / QB * QB;
    const Dealing d = fwd_dealing(slabs, S, 8);
    const long long rows = (long long)slabs * (S / 32);
    const int f = int(fwd_choose_split(D, QB, rows, S, d.busiest, 32, true, d.even, l[1] > 1));
    const int q = int(bwd_choose_dq_split(D, QB, rows, S, true, l[1] > 1));
    const int f0 = int(fwd_choose_split(D, QB, rows, S, d.busiest, 32, false, d.even, l[1] > 1));
    if (f != l[5] || q != l[6] || f0 != 0) {
      printf("D=%d slabs=%d S=%d: %d %d, without the length %d\n", D, slabs, l[3], f, q, f0);
      return 7;
    }
  }
}
""")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(source), "-o", str(program)], check=True)
    run = subprocess.run([str(program)], capture_output=True, text=True)
    assert run.returncode == 0, (run.returncode, run.stdout)
