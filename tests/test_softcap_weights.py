"""Weights and slopes of soft-capped scores in the backward (csrc/omni_attn_softcap.hpp, compiled alone) against 64 bits: no
further off than the textbook's form in 32 bits, exp2(cap tanh log2(e) - LSE log2(e)) and 1 - tanh^2."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "omni-attention_amd", "csrc")

PROGRAM = r"""
#include "omni_attn_softcap.hpp"
#include <cstdio>
#include <random>
#include <vector>
using namespace omni_attn;
int main() {
  std::mt19937_64 gen(7);
  const double log2e = 1.4426950408889634;
  for (double cap : {10., 15., 20., 30., 50., 100., 300.})
    for (double spread : {0.3, 1., 3., 10., 60.}) {
      std::normal_distribution<double> normal(0, spread);
      double ours = 0, plain = 0, slope_ours = 0, slope_plain = 0;
      const double D = 64;
      const float c2 = float(2 * log2e / (std::sqrt(D) * cap)), cap_l2 = float(log2e * cap);
      for (int row = 0; row < 200; ++row) {
        std::vector<float> s(300);
        double sum = 0;
        for (float& x : s) {
          x = float(normal(gen) * std::sqrt(D));
          sum += std::exp(cap * std::tanh(double(x) / std::sqrt(D) / cap));
        }
        const float lse = float(std::log(sum)), off = lse * -1.4426950408889634f;
        for (float x : s) {
          const double tanh = std::tanh(double(x) / std::sqrt(D) / cap);
          const double w = std::exp(cap * tanh - double(lse)), slope = 1 / std::pow(std::cosh(double(x) / std::sqrt(D) / cap), 2);
          if (w < 1e-30 || slope < 1e-30) continue;
          const float d = capped_d(x, c2), t = 1.f - d;
          const double got = exp2f(capped_exponent(t, cap_l2, off)), got_slope = capped_slope(d, t);
          const float t0 = fmaf(1.f / (exp2f(x * c2) + 1.f), -2.f, 1.f);
          const double ref = exp2f(fmaf(t0, float(cap) * 1.4426950408889634f, off)), ref_slope = fmaf(-t0, t0, 1.f);
          ours += std::pow(got / w - 1, 2);
          plain += std::pow(ref / w - 1, 2);
          slope_ours += std::pow(got_slope / slope - 1, 2);
          slope_plain += std::pow(ref_slope / slope - 1, 2);
        }
      }
      printf("cap %g spread %g: weight %.3f slope %.3f of the plain form's error\n", cap, spread, std::sqrt(ours / plain),
             std::sqrt(slope_ours / slope_plain));
    }
  // the ends: tanh is -1 and 1, the slope 0, the weight of a row without a key 0
  for (float s : {-INFINITY, -1e30f, 1e30f, INFINITY}) {
    const float d = capped_d(s, 0.01f), t = 1.f - d;
    if (t != (s < 0 ? -1.f : 1.f) || capped_slope(d, t) != 0.f || exp2f(capped_exponent(t, 72.f, -INFINITY)) != 0.f) printf("end %g\n", s);
  }
}
"""


def test_capped_weights_against_64_bits(tmp_path):
    source, program = tmp_path / "softcap.cpp", tmp_path / "softcap"
    source.write_text("#include <cmath>\n" + PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-I", CSRC, str(source), "-o", str(program)], check=True)
    lines = subprocess.run([str(program)], check=True, capture_output=True, text=True).stdout.splitlines()
    assert len(lines) == 35
    for line in lines:
        words = line.split()
        assert float(words[words.index("weight") + 1]) <= 1.02, line  # (6e4 weights: the ratio is good to about 1 %)
        assert float(words[words.index("slope") + 1]) <= 1.02, line
