"""Where the generic forward's steps find their rows (csrc/omni_attn_generic_rows.hpp, compiled alone)."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "omni-attention_amd", "csrc")


def run_program(tmp_path, text):
    source, program = tmp_path / "rows.cpp", tmp_path / "rows"
    source.write_text("#include \"omni_attn_generic_rows.hpp\"\n#include <cstdio>\n#include <initializer_list>\nusing namespace omni_attn;\n"
                      "#define CHECK(x) if (!(x)) { printf(\"line %d: %s\\n\", __LINE__, #x); return 1; }\n" + text)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fsanitize=undefined", "-fno-sanitize-recover=all", "-I", CSRC,
                    str(source), "-o", str(program)], check=True)
    run = subprocess.run([str(program)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout + run.stderr


def test_halves_never_begin_behind_the_end_of_their_buffer(tmp_path):
    """The check of a buffer's range takes the uniform offset off its size first: it may not be larger.  A lane reads
    where its row is one of the sequence, and nothing else."""
    run_program(tmp_path, r"""
int main() {
  for (int D = 8; D <= 256; D += 8)
    for (int pitch : {D, D + 8, 40 * D})
      for (int seqlen = 1; seqlen <= 70; ++seqlen)
        for (int row0 = 0; row0 < seqlen + 16; row0 += 16) {
          const uint32_t end = rows_end(seqlen, pitch, D, kBack), bytes = uint32_t(pitch) * 2;
          const HalfAt at = half_at(row0 < seqlen, row0, bytes, end);
          for (uint32_t i = 0; i < 4; ++i) {  // loads of a run: 1024 i in the instruction, off the uniform offset
            CHECK(at.offset >= 1024 * i);
            const uint32_t uniform = at.offset - 1024 * i;
            CHECK(uniform <= at.size);
            for (int r = 0; r < 16; ++r)
              for (int d0 : {0, D - 8}) {
                const uint32_t lane = uint32_t(r) * bytes + uint32_t(d0) * 2 + 1024 * i;
                CHECK((lane + 16 <= at.size - uniform) == (row0 + r < seqlen));
                CHECK((lane < at.size - uniform) == (row0 + r < seqlen));
                CHECK(row0 + r >= seqlen || lane + uniform == kBack + uint32_t(row0 + r) * bytes + uint32_t(d0) * 2);
              }
          }
        }
}
""")


def test_positions_in_lists_of_the_largest_blocks(tmp_path):
    """One column passes the check of sizes with as many rows as an int holds: nothing wraps around, and a walk ends."""
    run_program(tmp_path, r"""
int main() {
  const int most = 0x7fffffff;
  for (int S : {1, 15, 16, 17, 31, 32, 33, 4096, most - 33, most - 32, most - 31, most - 30, most - 16, most - 15, most - 1, most})
    for (int unit : {1, 16, 32})
      for (int KB : {1, 16, 31, 32, 48, 4096, most / 8, most - 257, most - 31, most - 1, most}) {
        const long long end = (S + (unit - 1LL)) / unit * unit;
        const int keys = walked_keys(KB, S, unit);
        CHECK(keys > 0 && keys == (KB < end ? KB : end));
        CHECK(blocks_of(S, KB) == (S + (KB - 1LL)) / KB);
        for (int step : {128, 256}) {  // the first and the last positions of a walk over two blocks
          const int adv_slot = step / keys, adv_off = step % keys;
          for (long long pos : {0LL, 31LL, keys - 1LL, keys - 32LL, keys - 256LL, 2LL * keys - 1}) {
            if (pos < 0) continue;
            int slot = int(pos / keys), off = int(pos % keys);
            for (int n = 1; n < 4; ++n) {
              int slot_of_int = slot, off_of_int = off;
              move_on<uint32_t>(slot, off, adv_slot, adv_off, keys);
              const long long to = pos + (long long)n * step;
              CHECK(slot == to / keys && off == to % keys);
              if (keys > most - 257) continue;
              move_on<int>(slot_of_int, off_of_int, adv_slot, adv_off, keys);
              CHECK(slot == slot_of_int && off == off_of_int);
            }
          }
        }
      }
}
""")
