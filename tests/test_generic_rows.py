"""Positions in the lists of the generic forward (csrc/omni_attn_generic_rows.hpp, compiled alone)."""
import os
import subprocess

import omni_attn_capi

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "omni-attention_amd", "csrc")


def run_program(tmp_path, text):
    source, program = tmp_path / "rows.cpp", tmp_path / "rows"
    source.write_text("#include \"omni_attn_generic_rows.hpp\"\n#include <cstdio>\n#include <initializer_list>\nusing namespace omni_attn;\n"
                      "#define CHECK(x) if (!(x)) { printf(\"line %d: %s\\n\", __LINE__, #x); return 1; }\n" + text)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fsanitize=undefined", "-fno-sanitize-recover=all", "-I", CSRC,
                    str(source), "-o", str(program)], check=True)
    run = subprocess.run([str(program)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout + run.stderr


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


def test_query_blocks_beyond_the_largest_int_are_refused():
    """Rows are ints, also those of the last query block that lie behind the sequence."""
    lib = omni_attn_capi.load_library()
    one = 4096  # any non-null value: validation fails before it would be dereferenced
    def call(S, QB, KB=32, D=1):
        return lib.omni_attn_fwd_generic_gfx950(one, one, one, one, 0, one, one, one, 0, 0, 1, 1, S, D, -(-S // QB), 1, QB, KB,
                                                0, 0, 0, 0.0, 0)
    most = 2 ** 31 - 1
    for S, QB in ((most, 2), (most, 64), (most, most), (most - 30, 32), (100, most), (most - 46, 48)):
        assert call(S, QB) == 2, (S, QB)
    assert call(most - 1, 1, D=2) == 7  # too large, not a bad shape
