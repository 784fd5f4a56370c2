// Soft-capped scores in the backward.  (Compiles for the host as well.)
#pragma once

#include <math.h>

#include "omni_attn_deal.hpp"

namespace omni_attn {

// A score s stands for x = s / sqrt(D) and counts as cap * tanh(x / cap).  With d = 2 / (exp(2 x / cap) + 1) the tanh is 1 - d
// and its derivative d (2 - d) = d + d (1 - d), which keeps its bits where the tanh is near 1.
OMNI_ATTN_HOST_DEVICE float capped_d(float s, float c2) {  // c2: 2 log2(e) / (sqrt(D) cap)
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rcpf(__builtin_fmaf(__builtin_amdgcn_exp2f(s * c2), 0.5f, 0.5f));
#else
  return 1.f / fmaf(exp2f(s * c2), 0.5f, 0.5f);
#endif
}
// Exponent (base 2) of its weight.  cap_l2: cap log2(e); off: -LSE log2(e).  (As off + cap_l2 - 2 cap_l2 / (exp(2 x / cap) + 1), the
// first two added up per row, it is an instruction less, but a larger number is rounded: the error of a weight against
// 64 bits, 1e-6 - 5e-6, is larger by up to 7 % at a cap of 20, 15 % at 30, 21 % at 100.)
OMNI_ATTN_HOST_DEVICE float capped_exponent(float tanh, float cap_l2, float off) { return __builtin_fmaf(tanh, cap_l2, off); }
OMNI_ATTN_HOST_DEVICE float capped_slope(float d, float tanh) { return __builtin_fmaf(d, tanh, d); }

}  // namespace omni_attn
