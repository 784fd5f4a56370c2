// One translation unit per (element type, head_dim): compiled several times with
// -DOMNI_INST_BF16={0,1} -DOMNI_INST_D={32,64,128}; each object defines the four
// (QB, KB) instances of the forward kernel and its split forms for that pair behind one C++ symbol.
#include "omni_attn_fwd_kernel.hpp"

#ifndef OMNI_INST_BF16
#error "compile with -DOMNI_INST_BF16=0|1"
#endif
#ifndef OMNI_INST_D
#error "compile with -DOMNI_INST_D=32|64|128"
#endif

namespace omni_attn {

template <bool BF16, int D>
int launch_fwd_blocks(const FwdParams& p, int QB, int KB, hipStream_t stream);

template <>
int launch_fwd_blocks<OMNI_INST_BF16 != 0, OMNI_INST_D>(const FwdParams& p, int QB, int KB,
                                                        hipStream_t stream) {
  constexpr bool BF = OMNI_INST_BF16 != 0;
  constexpr int D = OMNI_INST_D;
  switch (p.split) {
    case FwdSplit::kRows32x4: return launch_fwd_ksplit<BF, D, 32, 4, D == 128 ? 32 : 64>(p, stream);
    case FwdSplit::kRows64x2: return launch_fwd_ksplit<BF, D, 64, 2, D == 128 ? 32 : 64>(p, stream);
#if OMNI_INST_D == 128
    case FwdSplit::kRows64x4: return launch_fwd_ksplit<BF, D, 64, 4, 32>(p, stream);
    case FwdSplit::kRows128x2: return launch_fwd_ksplit<BF, D, 128, 2, 64>(p, stream);
#endif
    default: break;
  }
  if (QB == 128 && KB == 128) return launch_fwd<BF, D, 128, 128>(p, stream);
  if (QB == 128 && KB == 64) return launch_fwd<BF, D, 128, 64>(p, stream);
  if (QB == 64 && KB == 128) return launch_fwd<BF, D, 64, 128>(p, stream);
  if (QB == 64 && KB == 64) return launch_fwd<BF, D, 64, 64>(p, stream);
  return int(hipErrorInvalidValue);
}

}  // namespace omni_attn
