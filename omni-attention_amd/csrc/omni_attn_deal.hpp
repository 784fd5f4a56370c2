// The numbers behind the work order of a launch (deal_slab in the forward's header says what the order is),
// worked out on the host.  (Nothing here needs a GPU compiler.)
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define OMNI_ATTN_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define OMNI_ATTN_HOST_DEVICE inline
#endif

namespace omni_attn {

// Division of n < 2^31 by a number that the host knows: three scalar instructions, where a division by a kernel
// argument is 25 - 30 with a trip to the vector unit and back.  A workgroup made seven of them, 150 of the 400
// instructions before it could ask for its list, one after the other (a lone wave issues one in about five cycles).
// Without them: B=1 H=8 S=512 D=64 causal 6.55 -> 6.31 us, B=1 H=16 S=1024 D=64 10.2 -> 9.5, unaligned spans of
// 1237 rows 29.8 -> 29.3.
// mul = floor(2^(31 + shift) / d) + 1 with 2^shift >= d exceeds 2^(31 + shift) / d by less than 2^shift / d, so
// n * mul / 2^(31 + shift) exceeds n / d by less than 1 / d: the floors are the same.
struct FastDiv {
  uint32_t mul, shift;
};
inline FastDiv fast_div(uint32_t d) {  // 0 < d < 2^31
  uint32_t shift = 0;
  while ((1u << shift) < d) ++shift;
  return {uint32_t((uint64_t(1) << (31 + shift)) / d + 1), shift};
}
OMNI_ATTN_HOST_DEVICE uint32_t divide(uint32_t n, const FastDiv& by) {
  return uint32_t((uint64_t(n << 1) * by.mul) >> 32) >> by.shift;
}

struct DealPlan {
  FastDiv xcd;         // by the number of XCDs
  FastDiv per_group;   // by the workgroups of a group of slabs
  FastDiv group;       // by the slabs of a group,
  FastDiv last[2];     // and of the last group of an XCD: of those with the fewest slabs, and with one more
  FastDiv heads;       // by H
  int slabs;           // slabs (or parts) of the XCDs that have fewest
  int one_more;        // XCDs with one more
  int part_tiles;      // tiles of a part
  int part_shift;      // log2 of the parts per slab
};
// slabs in all, parts per slab (a power of two), XCDs, slabs that are walked together, tiles per slab, heads.
inline DealPlan plan_deal(int n_slabs, int parts, int n_xcd, int slab_group, int tiles, int H) {
  DealPlan d;
  const int all = n_slabs * parts;
  d.slabs = all / n_xcd;
  d.one_more = all % n_xcd;
  d.part_shift = 0;
  while ((1 << d.part_shift) < parts) ++d.part_shift;
  d.part_tiles = (tiles + parts - 1) / parts;
  d.xcd = fast_div(uint32_t(n_xcd));
  d.group = fast_div(uint32_t(slab_group));
  // (a group of more workgroups than a launch can have is never left)
  const uint64_t per_group = uint64_t(slab_group) * uint64_t(d.part_tiles);
  d.per_group = fast_div(per_group < 0x7fffffffu ? uint32_t(per_group) : 0x7fffffffu);
  for (int i = 0; i < 2; ++i) {
    const int rest = (d.slabs + i) % slab_group;
    d.last[i] = fast_div(uint32_t(rest != 0 ? rest : slab_group));
  }
  d.heads = fast_div(uint32_t(H));
  return d;
}

}  // namespace omni_attn
