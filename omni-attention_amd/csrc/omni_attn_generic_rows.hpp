// Where the generic forward's steps find their rows.  (Nothing here needs a GPU compiler.)
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define OMNI_ATTN_ROWS_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define OMNI_ATTN_ROWS_HOST_DEVICE inline
#endif

namespace omni_attn {

// Buffers that are read in halves of 16 keys begin this far before the slab (nothing is read there): a run of loads takes
// up to this much off its uniform offset again (buffer_to_lds_in_a_row).
constexpr uint32_t kBack = 3072;

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

// Bytes of a buffer that ends with the last column of the last row of the sequence.
OMNI_ATTN_ROWS_HOST_DEVICE uint32_t rows_end(int seqlen, int64_t pitch, int D, uint32_t back) {
  return uint32_t((int64_t(seqlen) - 1) * pitch + D) * 2u + back;
}

// Uniform offset and size of the buffer for half a step.  A load is checked as lane offset + offset in the instruction against
// size - uniform offset, and that difference must not be negative: a half that is not `live` (it begins behind the sequence, or
// no row attends to it) has a buffer that ends where the half begins, all of its lanes are outside, write zeros and touch no
// memory.
struct HalfAt {
  uint32_t offset, size;
};
OMNI_ATTN_ROWS_HOST_DEVICE HalfAt half_at(bool live, int row0, uint32_t pitch_bytes, uint32_t end) {
  return {live ? kBack + uint32_t(row0) * pitch_bytes : kBack, live ? end : kBack};
}

}  // namespace omni_attn
