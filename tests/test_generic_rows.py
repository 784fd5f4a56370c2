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
