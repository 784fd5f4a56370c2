// Positions in the lists of the generic forward.  (Nothing here needs a GPU compiler.)
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define OMNI_ATTN_ROWS_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define OMNI_ATTN_ROWS_HOST_DEVICE inline
#endif

namespace omni_attn {

// Blocks of n rows (0 < n) that S rows take, and keys of a block of KB that are walked: all of them, or no more than S rows take
// in whole units of a step (32), half a step (16) or keys (1).  (S and a block may be as large as an int.)
OMNI_ATTN_ROWS_HOST_DEVICE int blocks_of(int S, int n) { return int((int64_t(S) + n - 1) / n); }
OMNI_ATTN_ROWS_HOST_DEVICE int walked_keys(int KB, int S, int unit) {
  const int64_t end = int64_t(blocks_of(S, unit)) * unit;
  return KB < end ? KB : int(end);
}
// Moves the position (slot, off) of a list on by adv_slot blocks and adv_off <= 256 keys.  T: int where a block has at most
// 2^31 - 257 keys (eight columns and more: S * D is an int), uint32_t otherwise.  (uint32_t everywhere: 40x40 blocks, B=1 H=8
// S=2000 D=96 bf16 40.1 -> 40.6 us, S=720 D=256 fp16 20.6 -> 21.1.)
template <class T>
OMNI_ATTN_ROWS_HOST_DEVICE void move_on(int& slot, int& off, int adv_slot, int adv_off, int keys) {
  slot += adv_slot;
  T to = T(off) + T(adv_off);
  if (to >= T(keys)) {
    to -= T(keys);
    ++slot;
  }
  off = int(to);
}

}  // namespace omni_attn
