// The forward for shapes the tuned kernel has no instance for.
//
// The reference's correctness kernel omni_attn_simple_kernel_impl
// (omni-attn-mma/mma/attn_naive.cu:21-302, launcher :305-408) takes any Q_BLOCK / KV_BLOCK and
// any head_dim up to 256 (`float out[256]`, :189-190); its MMA kernels take only
// {64, 128}^2 x {32, 64, 128}.  This kernel keeps that generality and the slot rules, on the matrix
// cores, at the precision of a scalar kernel: products of 16-bit operands summed in fp32, and fp32
// weights that enter the second product with all their bits.
//
// One workgroup owns up to 32 query rows of one query block; its waves share the keys of the
// block's list: the listed keys are one sequence of positions, slot * KB + offset; step n is the
// positions 32 n .. 32 n + 31 (of one block or of several, for any KB) and wave w takes the steps
// w, w + waves, ...  A wave has its own running maximum, sum and O^T accumulators; they are merged
// through LDS at the end.  No workgroup barrier until then.
//
// S^T = K.Q^T and O^T = V^T.P^T with v_mfma_f32_32x32x16 as in the tuned forward: a lane owns a query
// row; the K and V rows of a step go to tiles of the wave in LDS, straight from global memory where rows
// lie on 16-byte boundaries.  Up to 128 columns a wave has a tile for each, and the rows of the next step are
// requested as soon as the products have read it; beyond, it has one tile, which V takes over from K and the next step's
// K from V, and the other wave of its SIMD works meanwhile.  A weight is a sum of three 16-bit parts with one
// product each.  fp16 has few exponents: weights are scaled by 2^11 first, and those below 2^-12 of the
// reference (scores of a peaked row) leave a rest that goes through two more products of the steps that have any.
//
// A key that a row may not attend to never reaches it, whatever its V row holds (0 * infinity would):
// a wave whose sums end up infinite or NaN walks its list once more and leaves out the zero weights.
//
// Bound by the instructions of a step (softmax, split of the weights and bookkeeping on the vector pipe: about 3000
// cycles of a wave against 770 of its products at D=96) times the steps of the longest list over the waves.  So rows
// that go to LDS directly have their offsets laid out once, their fragments are fetched in groups (K, and V under the
// weights; three ahead beyond 128 columns), and a weight's part is taken off without being converted first.  B=1 H=8
// S=2048 D=96, causal in 32x32 blocks, launches back to back: fp16 23.8 us, bf16 23.0 (28.7 and 26.9 without); spans in
// 64x64 blocks at B=1 H=4 S=1500 bf16: D=136 22.4, D=208 26.9, D=256 29.2; rows at any alignment, D=101 35.3, D=131 37.0,
// D=165 41.9.  33 us (37) at D=96 where queries are four times as large (every row peaked, a rest in most steps).  Two parts per
// weight, cut off after 22 bits and at 2^-32 of the reference, gain 2 us, but are
// not the scalar kernel's sum.  One wave per row with vector arithmetic: 1934 us.
#include "../../include/omni_attn_gfx950.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <cmath>
#include <type_traits>
#include <utility>

#include "omni_attn_deal.hpp"
#include "omni_attn_generic_rows.hpp"

namespace omni_attn {
// Keeps the hipError_t behind an OMNI_ATTN_ERR_LAUNCH for omni_attn_last_hip_error() (defined
// beside that function).
void record_hip_error(int hip_error);
}  // namespace omni_attn

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2_t;
typedef __attribute__((ext_vector_type(4))) short s16x4_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) int32_t i32x4_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;

enum : int { kMasked = 0, kCausal = 1, kFull = 2, kPartial = 3 };
constexpr int kMaxD = 256;

struct GenericParams {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  omni_attn_strides q_at, k_at, v_at;  // (o is contiguous, S rows per slab)
  uint16_t* o;
  float* lse;
  const int32_t* kv_num_blocks;
  const int32_t* kv_indices;
  const int32_t* types;
  const int32_t* partial_idx;
  const uint8_t* partial_masks;
  int num_partial;
  int S, D, H, Tq, Tk, max_blocks, QB, KB, seqlen;
  int kb_eff;         // keys of a block that can be inside the sequence: min(KB, S)
  int adv_slot, adv_off;  // 32 positions per wave = adv_slot blocks of kb_eff keys + adv_off keys
  int q_tiles;        // 32-row tiles per query block
  int o_vec;          // rows of o start on 8-byte boundaries and D is a multiple of 8
  int mask_words;     // four keys of a tile row may be read as one 32-bit word
  int whole;          // a step never crosses a block (blocks of 32 n keys, mask_words)
  unsigned n_slabs;   // B * H
  omni_attn::FastDiv by_slabs, by_tiles, by_heads;  // by n_slabs, q_tiles, H
  float scale, sl2, softcap;
};

// Columns are worked in chunks of 8, chunk i at columns 8 i .. 8 i + 7.  Where D is not a multiple of
// 8 the last chunk holds the columns D - 8 .. D - 1 instead, and so do the chunks beyond it: every
// read is 16 bytes inside its row (at any alignment), Q is zero where a chunk repeats a column, and
// the repeated columns of the result are not stored.
__device__ __forceinline__ int chunk_start(int d0, int D) { return d0 + 8 <= D ? d0 : D - 8; }

// How rows are read: straight to LDS (rows of k and v on 16-byte boundaries, D a multiple of 8), by
// 16-byte loads at any alignment, or element by element (head dimensions below 8).
// A step straight to LDS is two halves of 16 keys.  kWhole (blocks of 32 n keys) has both in one block, kHalves (16 n keys)
// each in one: what a step needs to know (first key row, mode, tile) is one or two sets of scalars, and the offsets of
// 16 rows are laid out once.  kKeys takes other block sizes: every key is followed by a lane of its own.  B=1 H=8, us,
// 16 n keys by key -> in halves: S=715 48x48 spans D=40 11.3 -> 10.0, D=96 14.1 -> 11.4; S=2048 causal D=96 48x48
// 37.0 -> 33.4, 16x16 49.7 -> 45.3; 32x32, one kernel for all -> kWhole, bf16 23.5 -> 23.0, fp16 24.5 -> 24.4.
enum class Rows : int { kWhole, kWide, kSmall, kHalves, kKeys };

// The chunk of `row` at column d0 (kSmall: zeros behind the row).
template <Rows R>
__device__ __forceinline__ u32x4_t load8(const uint16_t* row, int d0, int D) {
  u32x4_t r;
  if constexpr (R == Rows::kSmall) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = d0 + 2 * i;
      const uint32_t lo = row[d < D ? d : 0], hi = row[d + 1 < D ? d + 1 : 0];
      r[i] = (d < D ? lo : 0u) | (d + 1 < D ? hi << 16 : 0u);
    }
  } else {
    __builtin_memcpy(&r, row + chunk_start(d0, D), 16);
  }
  return r;
}

// 16 bytes per lane from a buffer straight into LDS, at lds_base + 16 * lane; a lane whose offset lies
// beyond the buffer writes zeros.  (Inline asm, so that reads of other tiles are not ordered behind it;
// completion is waited for explicitly.)
__device__ __forceinline__ void buffer_to_lds(i32x4_t rsrc, uint32_t lane_off, uint32_t uniform_off,
                                              uint32_t lds_base) {
  i32x4_t r;
  r[0] = __builtin_amdgcn_readfirstlane(rsrc[0]);
  r[1] = __builtin_amdgcn_readfirstlane(rsrc[1]);
  r[2] = __builtin_amdgcn_readfirstlane(rsrc[2]);
  r[3] = __builtin_amdgcn_readfirstlane(rsrc[3]);
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %1, %2, %3 offen lds"
      :
      : "s"(__builtin_amdgcn_readfirstlane(lds_base)), "v"(lane_off), "s"(r),
        "s"(__builtin_amdgcn_readfirstlane(uniform_off))
      : "memory", "m0");
}
// N such loads from one uniform offset, 1 KiB of LDS apart.  (The offset in the instruction counts for both addresses, and
// is taken off the uniform one again, which is at least kBack: the check of the range does not take a negative one.  A load by
// itself takes three scalar instructions more.  With scores that are masked in place and weights that are split without
// copies, fp16 B=1 H=8 S=2048 causal 32x32 D=96 24.3 -> 23.8 us, D=120 29.3 -> 28.8, D=256 S=1024 21.9 -> 21.3.)
constexpr uint32_t kBack = 3072;
template <int N>
__device__ __forceinline__ void buffer_to_lds_in_a_row(i32x4_t rsrc, const uint32_t* lane_off, uint32_t uniform_off,
                                                       uint32_t lds_base) {
  static_assert(N >= 1 && N <= 4, "twelve bits of offset");
  i32x4_t r;
  r[0] = __builtin_amdgcn_readfirstlane(rsrc[0]);
  r[1] = __builtin_amdgcn_readfirstlane(rsrc[1]);
  r[2] = __builtin_amdgcn_readfirstlane(rsrc[2]);
  r[3] = __builtin_amdgcn_readfirstlane(rsrc[3]);
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds_base), u = __builtin_amdgcn_readfirstlane(uniform_off);
  if constexpr (N == 1) {
    buffer_to_lds(r, lane_off[0], u, m0);
  } else if constexpr (N == 2) {
    asm volatile(
        "s_mov_b32 m0, %0\n\t"
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %1, %3, %4 offen lds\n\t"
        "buffer_load_dwordx4 %2, %3, %5 offen offset:1024 lds"
        :
        : "s"(m0), "v"(lane_off[0]), "v"(lane_off[1]), "s"(r), "s"(u), "s"(u - 1024u)
        : "memory", "m0");
  } else if constexpr (N == 3) {
    asm volatile(
        "s_mov_b32 m0, %0\n\t"
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %1, %4, %5 offen lds\n\t"
        "buffer_load_dwordx4 %2, %4, %6 offen offset:1024 lds\n\t"
        "buffer_load_dwordx4 %3, %4, %7 offen offset:2048 lds"
        :
        : "s"(m0), "v"(lane_off[0]), "v"(lane_off[1]), "v"(lane_off[2]), "s"(r), "s"(u), "s"(u - 1024u), "s"(u - 2048u)
        : "memory", "m0");
  } else {
    asm volatile(
        "s_mov_b32 m0, %0\n\t"
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %1, %5, %6 offen lds\n\t"
        "buffer_load_dwordx4 %2, %5, %7 offen offset:1024 lds\n\t"
        "buffer_load_dwordx4 %3, %5, %8 offen offset:2048 lds\n\t"
        "buffer_load_dwordx4 %4, %5, %9 offen offset:3072 lds"
        :
        : "s"(m0), "v"(lane_off[0]), "v"(lane_off[1]), "v"(lane_off[2]), "v"(lane_off[3]), "s"(r), "s"(u), "s"(u - 1024u),
          "s"(u - 2048u), "s"(u - 3072u)
        : "memory", "m0");
  }
}
// At most N vector-memory operations of this wave are outstanding.
template <int N>
__device__ __forceinline__ void wait_but() {
  static_assert(N < 64, "six bits");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
  asm volatile("" ::: "memory");
}

template <bool BF16>
__device__ __forceinline__ f32x16_t mfma(u32x4_t a, u32x4_t b, f32x16_t c) {
  if constexpr (BF16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0,
                                                  0, 0);
  }
}

// One 16-bit part of a pair of non-negative values, cut off towards zero; the values become what is left
// of them (exact: after three bf16 parts nothing is left).
// (OVER: the rest takes the place of the value at once; the compiler copies values that are needed later first.)
template <bool BF16, bool OVER>
__device__ __forceinline__ uint32_t split_part(float& lo, float& hi) {
  if constexpr (BF16) {
    const uint32_t a = __builtin_bit_cast(uint32_t, lo), b = __builtin_bit_cast(uint32_t, hi);
    lo -= __builtin_bit_cast(float, a & 0xffff0000u);
    hi -= __builtin_bit_cast(float, b & 0xffff0000u);
    return __builtin_amdgcn_perm(b, a, 0x07060302u);  // upper halves of both
  } else {
    const auto v = __builtin_amdgcn_cvt_pkrtz(lo, hi);
    const uint32_t h = __builtin_bit_cast(uint32_t, v);
    // value - part, with the part's half read as it is (the compiler converts it first: two instructions more per part)
    if constexpr (OVER) {
      asm("v_fma_mix_f32 %0, %1, -1.0, %0 op_sel_hi:[1,0,0]" : "+v"(lo) : "v"(h));
      asm("v_fma_mix_f32 %0, %1, -1.0, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(hi) : "v"(h));
      return h;
    }
    float a, b;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(a) : "v"(h), "v"(lo));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(b) : "v"(h), "v"(hi));
    lo = a;
    hi = b;
    return h;
  }
}
template <bool BF16>
__device__ __forceinline__ uint16_t from_float(float x) {
  if constexpr (BF16) {
    const __bf16 b = (__bf16)x;
    return __builtin_bit_cast(uint16_t, b);
  } else {
    const _Float16 h = (_Float16)x;
    return __builtin_bit_cast(uint16_t, h);
  }
}

// One 16-bit value as a float (the inverse of a part of split_part).
template <bool BF16>
__device__ __forceinline__ float to_float(uint32_t bits) {
  if constexpr (BF16) {
    return __builtin_bit_cast(float, bits << 16);
  } else {
    return float(__builtin_bit_cast(_Float16, uint16_t(bits)));
  }
}

// x of this lane and of lane ^ 32, in any order.
// (SWAP: without LDS.  The forms that read rows at any alignment have no register left for it.)
template <bool SWAP>
__device__ __forceinline__ void both_halves(float x, float& lo, float& hi) {
  if constexpr (!SWAP) {
    lo = x;
    hi = __shfl_xor(x, 32, 64);
    return;
  }
  typedef __attribute__((ext_vector_type(2))) unsigned u2;
  const unsigned a = __builtin_bit_cast(unsigned, x);
  const u2 r = __builtin_amdgcn_permlane32_swap(a, a, false, false);
  const unsigned r0 = r[0], r1 = r[1];
  lo = __builtin_bit_cast(float, r0);
  hi = __builtin_bit_cast(float, r1);
}

// DT: 32-column tiles of the head dimension; NW: waves.
template <int DT, int NW>
struct GenericTraits {
  static constexpr int kRowBytes = 64 * DT;
  static constexpr int kTileBytes = 32 * kRowBytes;
  // Beyond 128 columns LDS has room for K and V of four waves, one to a SIMD, or for one tile of eight, where V takes
  // the place of K as soon as that is read.  The loads of a wave then run under its softmax and the other wave of the SIMD
  // only, but a list has half the steps per wave and a SIMD two waves to issue from.  (At S=1024 D=208 a lone wave took
  // 29.8 us over eight steps of 1800 cycles of products.)  What eight waves have no registers for is worked out anew in each
  // step (addresses of fragments) or lies in LDS (Q, offsets of rows).  B=1 H=8, bf16, us, four waves -> eight: S=1024 causal 32x32
  // D=136 20.0 -> 15.2, D=208 29.8 -> 19.4, D=256 29.7 -> 21.9; S=64 D=208 10.5 -> 8.5; S=715 rows at any alignment D=165
  // 43.8 -> 23.5, D=250 51.3 -> 30.8; blocks of 40 keys D=256 34.1 -> 23.8.  Twelve waves up to 96 columns: 4 % slower.
  static constexpr bool kShared = DT > 4 && NW == 8;
  static constexpr size_t kWaveBytes = size_t(kShared ? 1 : 2) * kTileBytes;
  static constexpr int kGroup = DT < 4 ? DT : 4;  // output tiles merged per pass
  static constexpr size_t kMergeBytes = size_t(NW) * kGroup * 4096;
  // K and V of every wave; the merge overlaps them
  static constexpr size_t kTiles = NW * kWaveBytes > kMergeBytes ? NW * kWaveBytes : kMergeBytes;
  // From 97 columns on Q lives in LDS, shared by the waves.  (With 129 - 160 in the registers of each of eight waves, rows
  // at any alignment read one chunk after the other: B=1 H=8 S=64 D=131 bf16 12.6 us, 9.7 so, 11.0 with four waves; S=1024 27.3,
  // 24.9, 42.5; rows straight to LDS, D=136 S=64 7.6, 7.4, 8.5.)
  static constexpr bool kQInLds = DT >= 4;
  static constexpr size_t kQBytes = kQInLds ? size_t(kTileBytes) : 0;
  // ... and there the byte offsets of a lane's chunks of 16 rows, K and V, which eight waves have no registers for
  static constexpr bool kOffsetsInLds = kShared && DT >= 7;
  static constexpr size_t kOffsetBytes = kOffsetsInLds ? size_t(2 * DT * 64 * 4) : 0;
  // behind the tiles: Q; per wave, compare key, offset inside the block, tile and row of 32 keys; and
  // the maximum and sum of 32 rows
  static constexpr size_t kLdsBytes = kTiles + kQBytes + NW * (32 * 16 + 32 * 8) + kOffsetBytes;
};

template <bool BF16, int DT, int NW, Rows R>
__device__ __forceinline__ void generic_walk(const GenericParams& p) {
  using Traits = GenericTraits<DT, NW>;
  constexpr int KS = 2 * DT;
  constexpr int C = 4 * DT;     // 16-byte chunks of a tile row
  constexpr int NLD = 2 * DT;   // chunks of a tile per lane
  constexpr int PARTS = 3;
  // The reference point of the exponentials follows the running maximum when that is more than kSlack
  // ahead (log2), so that the sums are rarely rescaled; kShift: log2 of the factor on the weights, which stay
  // below 2^(kSlack + kShift), inside fp16's range.
  constexpr float kSlack = BF16 ? 6.f : 4.f, kShift = BF16 ? 0.f : 11.f;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

  const unsigned wg = blockIdx.x;
  const unsigned rank = omni_attn::divide(wg, p.by_slabs);
  const unsigned bh = wg - rank * p.n_slabs;
  const unsigned tile = unsigned(p.Tq) * unsigned(p.q_tiles) - 1 - rank;  // longest lists of a causal mask first
  const int qb = int(omni_attn::divide(tile, p.by_tiles));
  const int row0 = int(tile - unsigned(qb) * unsigned(p.q_tiles)) * 32;  // first row inside the block
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 5, c = lane & 31;
  const int q_local = row0 + c;
  const int q_idx = qb * p.QB + q_local;
  const bool q_here = q_local < p.QB && q_idx < p.S;  // a row of this tile
  const bool q_live = q_here && q_idx < p.seqlen;

  constexpr bool SHARED = Traits::kShared;
  uint8_t* const sK = lds + size_t(w) * Traits::kWaveBytes;
  uint8_t* const sV = SHARED ? sK : sK + Traits::kTileBytes;
  uint8_t* const sQ = lds + Traits::kTiles;
  int32_t* const sKey = reinterpret_cast<int32_t*>(lds + Traits::kTiles + Traits::kQBytes) + w * 128;
  int32_t* const sOff = sKey + 32;
  int32_t* const sPid = sKey + 64;
  int32_t* const sRow = sKey + 96;  // (rows at any alignment, eight waves) -1: zeros
  constexpr bool ROWS_IN_LDS = SHARED && R == Rows::kWide;
  float* const sStat = reinterpret_cast<float*>(lds + Traits::kTiles + Traits::kQBytes + NW * 512);  // [2][NW][32]

  uint32_t* const sAt = reinterpret_cast<uint32_t*>(sStat + 2 * NW * 32);  // [2][DT][64], K and V

  const int64_t b = omni_attn::divide(bh, p.by_heads), h = bh - unsigned(b) * unsigned(p.H);
  const uint16_t* const q_slab = p.q + b * p.q_at.batch + h * p.q_at.head;
  const uint16_t* const k_slab = p.k + b * p.k_at.batch + h * p.k_at.head;
  const uint16_t* const v_slab = p.v + b * p.v_at.batch + h * p.v_at.head;
  const size_t mrow = size_t(bh) * p.Tq + qb;
  const size_t moff = mrow * p.max_blocks;
  const bool has_partial = p.partial_idx != nullptr && p.partial_masks != nullptr;

  // Block metadata in registers: lane i holds slot 64 chunk + i of the list (block index, and mode in
  // the low two bits with the tile index above).
  int32_t mv_idx = 0, mv_info = kMasked, chunk_at = 0;
  auto info_of = [&](int type, int pid) {
    int mode = (type == kCausal || type == kFull || type == kPartial) ? type : int(kMasked);
    if (mode == kPartial && (pid < 0 || pid >= p.num_partial)) mode = kMasked;  // attn_naive.cu:119-131
    return (mode == kPartial ? pid << 2 : 0) | mode;
  };
  auto load_chunk = [&](int chunk) {
    const int j = chunk * 64 + lane;
    const size_t o = moff + size_t(j < p.max_blocks ? j : 0);
    mv_idx = p.kv_indices[o];
    mv_info = info_of(p.types[o], has_partial ? p.partial_idx[o] : -1);
    chunk_at = chunk;
  };
  load_chunk(0);
  int nb = p.kv_num_blocks[mrow];
  nb = nb < 0 ? 0 : (nb > p.max_blocks ? p.max_blocks : nb);
  if (qb * p.QB + row0 >= p.seqlen) nb = 0;  // only padding rows: zeros (attn_naive.cu:64-72)

  // Chunk (16 bytes) `ch` of row r of a tile.  The XOR keeps 16 consecutive rows of one chunk (K, Q) and
  // four consecutive chunks of four consecutive rows (transposed reads of V) on different banks.
  auto swizzle = [](int r) {
    const int low = (r >> 2) & 3;
    return DT % 2 == 1 ? low : (DT % 4 == 2 ? (low | ((r >> 1) & 1) << 2) : (low | (r & 3) << 2));
  };
  auto tile_at = [&](int r, int ch) { return r * Traits::kRowBytes + (ch ^ swizzle(r)) * 16; };
  // The form with the fewest registers left over takes scores and weights apart in copies, which the compiler orders
  // better there: B=1 H=8 S=1400 causal D=101 28.4 us, 29.3 as the others do it.
  constexpr bool SHORT = R == Rows::kWide && DT == 4;
  constexpr bool WHOLE = R == Rows::kWhole, HALVES = WHOLE || R == Rows::kHalves, DIRECT = HALVES || R == Rows::kKeys;
  // Byte offset of a lane's chunk id of a tile inside its row.
  auto col_at = [&](int id) { return uint32_t(chunk_start(((id % C) ^ swizzle(id / C)) * 8, p.D)) * 2u; };
  if constexpr (Traits::kOffsetsInLds) {  // (read behind the barrier that Q has)
    static_assert(Traits::kQInLds, "a barrier");
    for (int i = w; i < DT; i += NW) {
      const int id = i * 64 + lane;
      sAt[id] = uint32_t(id / C) * uint32_t(p.k_at.row * 2) + col_at(id);
      sAt[DT * 64 + id] = uint32_t(id / C) * uint32_t(p.v_at.row * 2) + col_at(id);
    }
  }
  // Q as B operand: lane holds Q[row][16 s + 8 g .. +7]
  u32x4_t qf[Traits::kQInLds ? 1 : KS];
  {
    const uint16_t* qrow = q_slab + int64_t(q_live ? q_idx : 0) * p.q_at.row;
    if constexpr (DIRECT) {  // (16-byte chunks of D % 8 == 0 columns: none has columns of the one before)
      constexpr int NQ = Traits::kQInLds ? (KS + NW - 1) / NW : KS;  // chunks of this wave
      u32x4_t x[NQ];  // all in flight together, and cleared below: one under a condition is waited for
#pragma unroll
      for (int n = 0; n < NQ; ++n) {
        const int d0 = 16 * (Traits::kQInLds ? n * NW + w : n) + 8 * g;
        x[n] = load8<Rows::kWide>(qrow, d0 < p.D ? d0 : 0, p.D);
      }
      if constexpr (NQ > 1) {
#pragma unroll
        for (int n = 0; n < NQ; ++n) asm volatile("" : "+v"(x[n]));
      }
#pragma unroll
      for (int n = 0; n < NQ; ++n) {
        const int s = Traits::kQInLds ? n * NW + w : n;
        if (!q_live || 16 * s + 8 * g >= p.D) x[n] = u32x4_t{0u, 0u, 0u, 0u};
        if constexpr (Traits::kQInLds) {
          if (s < KS) *reinterpret_cast<u32x4_t*>(sQ + tile_at(c, 2 * s + g)) = x[n];
        } else {
          qf[s] = x[n];
        }
      }
    } else {
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        if (Traits::kQInLds && s % NW != w) continue;
        const int d0 = 16 * s + 8 * g;
        u32x4_t x = load8<R>(qrow, d0, p.D);
        if (!q_live || d0 >= p.D) x = u32x4_t{0u, 0u, 0u, 0u};
        if (R != Rows::kSmall && d0 < p.D) {
          const int repeats = d0 - chunk_start(d0, p.D);  // leading columns that the chunk before has
#pragma unroll
          for (int i = 0; i < 4; ++i)
            x[i] &= (2 * i >= repeats ? 0xffffu : 0u) | (2 * i + 1 >= repeats ? 0xffff0000u : 0u);
        }
        if constexpr (Traits::kQInLds) {
          *reinterpret_cast<u32x4_t*>(sQ + tile_at(c, 2 * s + g)) = x;
        } else {
          qf[s] = x;
        }
      }
    }
    if (Traits::kQInLds) __syncthreads();
  }
  auto q_frag = [&](int s) {
    if constexpr (Traits::kQInLds) {
      return *reinterpret_cast<const u32x4_t*>(sQ + tile_at(c, 2 * s + g));
    } else {
      return qf[s];
    }
  };

  // Position of this lane's key (lanes c and c + 32 follow the same key) in the wave's next step; with steps in halves,
  // of its first key.
  int slot, off;
  using Key32 = std::conditional_t<R == Rows::kSmall, uint32_t, int>;
  auto first_step = [&]() {
    const int pos = 32 * w + (HALVES ? 0 : c);
    slot = pos / p.kb_eff;
    off = pos - slot * p.kb_eff;
  };
  first_step();
  // The key of this lane.  `cmp`: the key is allowed for the query rows >= cmp (all of them for FULL and
  // PARTIAL, none for a key that does not exist, lies beyond the sequence or belongs to a skipped slot).
  struct Key {
    int row, cmp, off, pid;
  };
  auto next_key = [&]() {
    const int first = __builtin_amdgcn_readfirstlane(slot), last = __builtin_amdgcn_readlane(slot, 31);
    if ((first >> 6) != chunk_at) load_chunk(first >> 6);
    int idx = __shfl(mv_idx, slot & 63, 64), info = __shfl(mv_info, slot & 63, 64);
    if ((last >> 6) != (first >> 6) && (slot >> 6) != (first >> 6)) {  // the step runs into the next chunk
      const size_t o = moff + size_t(slot < p.max_blocks ? slot : 0);
      idx = p.kv_indices[o];
      info = info_of(p.types[o], has_partial ? p.partial_idx[o] : -1);
    }
    const int mode = slot < nb ? info & 3 : int(kMasked);
    const int kvb = idx < 0 ? 0 : (idx >= p.Tk ? p.Tk - 1 : idx);
    const long long row = (long long)kvb * p.KB + off;
    const bool live = mode != kMasked && row < p.seqlen;
    Key k;
    k.row = live ? int(row) : -1;
    k.cmp = !live ? 0x7fffffff : (mode == kCausal ? int(row) : -1);
    k.pid = (live && mode == kPartial) ? info >> 2 : -1;
    k.off = off;
    omni_attn::move_on<Key32>(slot, off, p.adv_slot, p.adv_off, p.kb_eff);
    return k;
  };

  // A step of one block (p.whole) is uniform over the wave: its first key, mode, tile and offset.
  struct Block {
    int row0, mode, pid, off;
  };
  auto next_block = [&]() {
    const int first = __builtin_amdgcn_readfirstlane(slot), at = __builtin_amdgcn_readfirstlane(off);
    if ((first >> 6) != chunk_at) load_chunk(first >> 6);
    const int idx = __builtin_amdgcn_readlane(mv_idx, first & 63), info = __builtin_amdgcn_readlane(mv_info, first & 63);
    const int kvb = idx < 0 ? 0 : (idx >= p.Tk ? p.Tk - 1 : idx);
    const long long row0 = (long long)kvb * p.KB + at;  // (beyond the sequence: nothing is allowed)
    Block k;
    k.mode = row0 < p.seqlen ? info & 3 : int(kMasked);
    k.row0 = k.mode != kMasked ? int(row0) : 0;
    k.pid = info >> 2;
    k.off = at;
    omni_attn::move_on<Key32>(slot, off, p.adv_slot, p.adv_off, p.kb_eff);
    return k;
  };

  // A step in halves of 16 keys, each inside one block.
  Block half[2] = {{0, kMasked, 0, 0}, {0, kMasked, 0, 0}};
  auto block_at = [&](int s, int at) {
    if ((s >> 6) != chunk_at) load_chunk(s >> 6);
    const int idx = __builtin_amdgcn_readlane(mv_idx, s & 63), info = __builtin_amdgcn_readlane(mv_info, s & 63);
    const int kvb = idx < 0 ? 0 : (idx >= p.Tk ? p.Tk - 1 : idx);
    const long long row0 = (long long)kvb * p.KB + at;
    Block k;
    k.mode = row0 < p.seqlen && (WHOLE || s < nb) ? info & 3 : int(kMasked);
    // (no rows are read from the end of the sequence on: those of a half that no row attends to would not count, but an
    // infinity in them would send the wave through its list again)
    k.row0 = k.mode != kMasked ? int(row0) : p.seqlen;
    k.pid = info >> 2;
    k.off = at;
    return k;
  };
  auto next_halves = [&]() {
    slot = __builtin_amdgcn_readfirstlane(slot);
    off = __builtin_amdgcn_readfirstlane(off);
    half[0] = block_at(slot, off);
    if constexpr (WHOLE) {  // the second half follows the first (rows beyond the sequence are masked)
      half[1] = {half[0].row0 + 16, half[0].mode, half[0].pid, off + 16};
    } else {
      const bool next = off + 16 >= p.kb_eff;
      half[1] = block_at(slot + int(next), next ? 0 : off + 16);
    }
    omni_attn::move_on<Key32>(slot, off, p.adv_slot, p.adv_off, p.kb_eff);
  };

  // Rows of a step into a tile: lane l takes the chunks l, l + 64, ... of the tile, in the order they
  // lie in LDS.  from[i]: row of the operand that chunk i of this lane comes from, -1 for zeros; of a
  // whole step only the first row matters (base) and from[i] counts from there.  (The chunks of 16 rows are DT per
  // lane, so chunk i + DT is chunk i of the second half: the swizzle repeats after 16 rows.)
  int from[NLD], base = 0;
  auto take_rows = [&](const Key& k) {
#pragma unroll
    for (int i = 0; i < NLD; ++i) from[i] = __shfl(k.row, (i * 64 + lane) / C, 64);
  };
#pragma unroll
  for (int i = 0; i < NLD; ++i) from[i] = (i * 64 + lane) / C;
  // (with steps in halves the buffer begins kBack bytes before the slab; nothing is read there)
  auto resource = [&](const uint16_t* slab, int64_t pitch) {
    constexpr uint32_t back = HALVES ? kBack : 0u;
    const uint64_t a = reinterpret_cast<uint64_t>(slab) - back;
    i32x4_t r;
    r[0] = __builtin_amdgcn_readfirstlane(int32_t(uint32_t(a)));
    r[1] = __builtin_amdgcn_readfirstlane(int32_t(uint32_t(a >> 32) & 0xffffu));
    r[2] = __builtin_amdgcn_readfirstlane(int32_t(uint32_t((int64_t(p.seqlen) - 1) * pitch + p.D) * 2u + back));
    r[3] = 0x00020000;
    return r;
  };
  const i32x4_t rK = resource(k_slab, p.k_at.row), rV = resource(v_slab, p.v_at.row);
  // byte offsets of this lane's chunks inside the rows, and of its rows in a whole step
  uint32_t cols[NLD];
#pragma unroll
  for (int i = 0; i < NLD; ++i) {
    cols[i] = col_at(i * 64 + lane);
  }
  // ... and of its chunks in half a step, K and V
  constexpr int NAT = HALVES && !Traits::kOffsetsInLds ? DT : 1;
  uint32_t k_at[NAT], v_at[NAT];
#pragma unroll
  for (int i = 0; i < NAT; ++i) {
    k_at[i] = uint32_t(from[i]) * uint32_t(p.k_at.row * 2) + cols[i];
    v_at[i] = uint32_t(from[i]) * uint32_t(p.v_at.row * 2) + cols[i];
  }
  auto load_tile = [&](auto again, bool is_k, const uint16_t* slab, const i32x4_t& rsrc, int64_t pitch, uint8_t* dst) {
    if constexpr (DIRECT) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the tile has been read
      const uint32_t to = uint32_t(size_t((__attribute__((address_space(3))) void*)dst));
      const uint32_t pitch2 = uint32_t(pitch * 2);
      if constexpr (HALVES) {
        uint32_t at[DT];
#pragma unroll
        for (int i = 0; i < DT; ++i) {
          if constexpr (Traits::kOffsetsInLds) {
            at[i] = sAt[((is_k ? 0 : DT) + i) * 64 + lane];
          } else {
            at[i] = is_k ? k_at[i] : v_at[i];
          }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          // (of a half that begins at the end of the sequence or behind it every lane is outside the buffer)
          const uint32_t row0_at =
              kBack + (WHOLE ? uint32_t(half[0].row0) * pitch2 + (h == 0 ? 0u : 16u * pitch2) : uint32_t(half[h].row0) * pitch2);
          buffer_to_lds_in_a_row<(DT < 4 ? DT : 4)>(rsrc, at, row0_at, to + uint32_t(h * DT) * 1024u);
          if constexpr (DT > 4) buffer_to_lds_in_a_row<DT - 4>(rsrc, at + 4, row0_at, to + uint32_t(h * DT + 4) * 1024u);
        }
      } else {
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
          const uint32_t at = uint32_t(from[i]) * pitch2 + cols[i];
          buffer_to_lds(rsrc, from[i] < 0 ? 0xffffffffu : at, 0u, to + uint32_t(i) * 1024u);
        }
      }
    } else if constexpr (SHARED) {
      int l = lane;  // (addresses are worked out anew: eight waves have no registers to keep them in)
      asm volatile("" : "+v"(l));
#pragma unroll
      for (int h = 0; h < 2; ++h) {  // 16 rows in flight together
        u32x4_t x[DT];
#pragma unroll
        for (int i = 0; i < DT; ++i) {
          const int id = i * 64 + l, row = sRow[16 * h + id / C];
          x[i] = load8<R>(slab + int64_t(row < 0 ? 0 : row) * pitch, ((id % C) ^ swizzle(id / C)) * 8, p.D);
          if (row < 0) x[i] = u32x4_t{0u, 0u, 0u, 0u};
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < DT; ++i) *reinterpret_cast<u32x4_t*>(dst + size_t((h * DT + i) * 64 + l) * 16) = x[i];
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      int l = lane;
      // (addresses worked out anew: kept over the walk they cost it registers)
      if constexpr (decltype(again)::value) asm volatile("" : "+v"(l));
#pragma unroll
      for (int i = 0; i < NLD; ++i) {
        if constexpr (decltype(again)::value) __builtin_amdgcn_sched_barrier(0);
        const int id = i * 64 + l;
        const int row = from[i] + base;  // (base is 0 unless the step is whole)
        const bool none = from[i] < 0 || row >= p.seqlen;
        u32x4_t x = load8<R>(slab + int64_t(none ? 0 : row) * pitch, ((id % C) ^ swizzle(id / C)) * 8, p.D);
        if (none) x = u32x4_t{0u, 0u, 0u, 0u};
        *reinterpret_cast<u32x4_t*>(dst + size_t(id) * 16) = x;
      }
    }
  };

  const f32x16_t zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  f32x16_t ot[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) ot[dt] = zero16;
  float m_run = -INFINITY, l_run = 0.f;  // log2 domain; l_run is this lane's share of the row

  // A wave is done when the first position of its step is beyond the list.
  auto more = [&]() { return __builtin_amdgcn_readfirstlane(slot) < nb; };
  bool go = more() && p.seqlen > 0;
  Key cur = {-1, 0x7fffffff, 0, -1};
  Block blk = {0, kMasked, 0, 0};
  auto advance = [&]() {
    if constexpr (HALVES) {
      next_halves();
    } else if (!DIRECT && p.whole) {
      blk = next_block();
      base = blk.row0;
      if constexpr (ROWS_IN_LDS) {
        if (g == 0) sRow[c] = base + c < p.seqlen ? base + c : -1;
      }
    } else {
      cur = next_key();
      if constexpr (ROWS_IN_LDS) {
        if (g == 0) sRow[c] = cur.row;
      } else {
        take_rows(cur);
      }
    }
  };
  auto first_rows = [&](auto again) {
    advance();
    load_tile(again, true, k_slab, rK, p.k_at.row, sK);
    if constexpr (!SHARED) load_tile(again, false, v_slab, rV, p.v_at.row, sV);
  };
  const int q_first = qb * p.QB + row0;  // first row of the workgroup
  // `again`: the second walk of a wave whose first met an infinity or a NaN in V (or overflowed); rare, so
  // that it may be slow.  (Code of its own: a branch in one loop doubles the registers of the sums.)
  auto walk = [&](auto again) {
    while (go) {
      // Allowed keys of this step as bits: register r (key 8 (r / 4) + 4 g + r % 4) is bit r.
      uint32_t keep = 0xffffu;
      bool masked;  // (uniform) some of them are not allowed
      uint32_t word[2][2];
      if constexpr (HALVES) {
        constexpr int BLOCKS = WHOLE ? 1 : 2, KEYS = 32 / BLOCKS;
        masked = false;
#pragma unroll
        for (int h = 0; h < BLOCKS; ++h) {
          const Block& k = half[h];
          masked |= !(k.row0 + KEYS <= p.seqlen && (k.mode == kFull || (k.mode == kCausal && k.row0 + KEYS - 1 <= q_first)));
          // PARTIAL (attn_naive.cu:143-154): the tile's bytes are asked for here and looked at behind the products
          if (k.mode == kPartial) {
            const uint8_t* t = p.partial_masks + (size_t(k.pid) * p.QB + (q_here ? q_local : 0)) * p.KB + k.off + 4 * g;
#pragma unroll
            for (int i = 0; i < KEYS / 8; ++i) word[h + i / 2][i % 2] = *reinterpret_cast<const uint32_t*>(t + 8 * i);
          }
        }
      } else if (!DIRECT && p.whole) {
        masked = !(p.seqlen - blk.row0 >= 32 && (blk.mode == kFull || (blk.mode == kCausal && blk.row0 + 31 <= q_first)));
        if (masked) {
          if (blk.mode == kPartial) {  // attn_naive.cu:143-154: any non-zero byte of the tile = attend
            const uint8_t* t = p.partial_masks + (size_t(blk.pid) * p.QB + (q_here ? q_local : 0)) * p.KB + blk.off + 4 * g;
            uint32_t word[4];
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) word[r4] = *reinterpret_cast<const uint32_t*>(t + 8 * r4);
            keep = 0;
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
              uint32_t x = word[r4];
              x |= x >> 4;
              x |= x >> 2;
              x |= x >> 1;
              keep |= (((x & 0x01010101u) * 0x01020408u) >> 24) << (4 * r4);
            }
          }
          int limit = p.seqlen - 1;
          if (blk.mode == kCausal) limit = limit < q_idx ? limit : q_idx;
          if (blk.mode == kMasked) limit = -1;
          const int n = limit - blk.row0 - 4 * g + 1;  // leading keys of this half-wave's pattern that are allowed
#pragma unroll
          for (int r4 = 0; r4 < 4; ++r4) {
            const int m = n - 8 * r4;
            const uint32_t four = m >= 4 ? 15u : (m <= 0 ? 0u : (1u << m) - 1u);
            keep &= ~((15u & ~four) << (4 * r4));
          }
        }
      } else {
        // what is known about the 32 keys, by key
        if (g == 0) {
          sKey[c] = cur.cmp;
          sOff[c] = cur.off;
          sPid[c] = cur.pid;
        }
        const bool any_partial = __builtin_amdgcn_ballot_w64(cur.pid >= 0) != 0;
        masked = any_partial || __builtin_amdgcn_ballot_w64(cur.cmp > q_first) != 0;
        if (masked) {
          keep = 0;
#pragma unroll
          for (int r4 = 0; r4 < 4; ++r4) {
            const i32x4_t cmp = *reinterpret_cast<const i32x4_t*>(sKey + 8 * r4 + 4 * g);
            uint32_t bytes = 0x01010101u;
            if (any_partial) {
              const i32x4_t pid = *reinterpret_cast<const i32x4_t*>(sPid + 8 * r4 + 4 * g);
              const i32x4_t po = *reinterpret_cast<const i32x4_t*>(sOff + 8 * r4 + 4 * g);
              const int ql = q_here ? q_local : 0;
              if (p.mask_words) {  // the four keys are neighbours in one block
                const int p0 = pid[0], o0 = po[0];
                if (p0 >= 0)
                  bytes = *reinterpret_cast<const uint32_t*>(p.partial_masks + (size_t(p0) * p.QB + ql) * p.KB + o0);
              } else {
                bytes = 0;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                  const int pi = pid[i], oi = po[i];
                  const uint32_t byte = pi >= 0 ? p.partial_masks[(size_t(pi) * p.QB + ql) * p.KB + oi] : 1u;
                  bytes |= byte << (8 * i);
                }
              }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int ci = cmp[i];
              keep |= uint32_t(ci <= q_idx && ((bytes >> (8 * i)) & 0xffu) != 0) << (4 * r4 + i);
            }
          }
        }
      }
      if constexpr (SHARED && DIRECT) {
        wait_but<0>();  // K is there
      } else if constexpr (DIRECT) {
        wait_but<NLD>();  // ... (V was requested after it)
      }
      f32x16_t st = zero16;
      // (SHARED: the addresses of the fragments are worked out anew in every step, from one register that the compiler
      // knows nothing about: kept over the walk they are what the eight waves have no registers for)
      uint32_t k_turn = uint32_t(g ^ swizzle(c)) * 16u;
      if constexpr (SHARED) asm volatile("" : "+v"(k_turn));
      auto k_frag = [&](int s) {
        if constexpr (SHARED) {
          return *reinterpret_cast<const u32x4_t*>(sK + c * Traits::kRowBytes + ((32u * s) ^ k_turn));
        } else {
          return *reinterpret_cast<const u32x4_t*>(sK + tile_at(c, 2 * s + g));
        }
      };
      auto q_operand = [&](int s) {
        if constexpr (SHARED && Traits::kQInLds) {
          return *reinterpret_cast<const u32x4_t*>(sQ + c * Traits::kRowBytes + ((32u * s) ^ k_turn));
        } else {
          return q_frag(s);
        }
      };
      // (fragments are fetched in groups, so that a group waits for LDS once)
      constexpr int AHEAD = SHARED ? 4 : (DIRECT ? (KS < 8 ? KS : 8) : 1);
#pragma unroll
      for (int s0 = 0; s0 < KS; s0 += AHEAD) {
        u32x4_t kf[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
          if (s0 + i < KS) kf[i] = k_frag(s0 + i);
        if constexpr (AHEAD > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
          if (s0 + i < KS) st = mfma<BF16>(kf[i], q_operand(s0 + i), st);
      }
      if constexpr (HALVES) {
        if (masked) {
          keep = 0;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const Block& k = half[h];
            int limit = p.seqlen - 1;
            if (k.mode == kCausal) limit = limit < q_idx ? limit : q_idx;
            if (k.mode == kMasked) limit = -1;
            const int n = limit - k.row0 - 4 * g + 1;  // leading keys of this half-wave's pattern that are allowed
#pragma unroll
            for (int i = 0; i < 2; ++i) {
              const int m = n - 8 * i;
              uint32_t four = m >= 4 ? 15u : (m <= 0 ? 0u : (1u << m) - 1u);
              if (k.mode == kPartial) {  // any non-zero byte of the tile = attend
                uint32_t x = word[h][i];
                x |= x >> 4;
                x |= x >> 2;
                x |= x >> 1;
                four &= ((x & 0x01010101u) * 0x01020408u) >> 24;
              }
              keep |= four << (4 * (2 * h + i));
            }
          }
        }
      }
      asm volatile("" : "+v"(keep));  // (the mask's own loads are waited for here, not behind the next request)
      // K has been read: the rows of the wave's next step, or V into its place
      if constexpr (SHARED) {
        load_tile(again, false, v_slab, rV, p.v_at.row, sV);
      } else {
        go = more();
        if (go) {
          advance();
          load_tile(again, true, k_slab, rK, p.k_at.row, sK);
        }
      }
      if (p.softcap > 0.f) {
#pragma unroll
        for (int r = 0; r < 16; ++r) st[r] = tanhf(st[r] * p.scale / p.softcap) * p.softcap;
      }
      // the lowest score of this lane (fp16, for the rests of the weights; allowed or not: a step that looks for rests in
      // vain costs less than a selection per score)
      float mn = INFINITY;
      if constexpr (!BF16 && !SHORT) {
#pragma unroll
        for (int r = 0; r < 16; ++r) mn = fminf(mn, st[r]);
        asm volatile("" : "+v"(mn));  // (here, before the scores change)
      }
      if (masked) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const bool kept = (keep >> r) & 1u;
          if constexpr (!BF16 && SHORT) mn = fminf(mn, kept ? st[r] : INFINITY);
          st[r] = kept ? st[r] : -INFINITY;
        }
      } else if constexpr (!BF16 && SHORT) {
#pragma unroll
        for (int r = 0; r < 16; ++r) mn = fminf(mn, st[r]);
      }
      float mx = -INFINITY;
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, st[r]);
      mx *= p.sl2;
      {
        float lower, upper;
        both_halves<DIRECT>(mx, lower, upper);
        mx = fmaxf(lower, upper);
      }
      if (__builtin_amdgcn_ballot_w64(mx > m_run + kSlack) != 0) {
        const float m_new = fmaxf(m_run, mx);
        const float m_ref = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_ref);
        l_run *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) ot[dt][r] *= alpha;
        m_run = m_new;
      }
      const float m_ref = m_run == -INFINITY ? 0.f : m_run;
      if constexpr (SHARED && DIRECT) {  // V is there
        wait_but<0>();
      } else if constexpr (DIRECT) {  // ... (the next K was requested after it)
        if (go) {
          wait_but<NLD>();
        } else {
          wait_but<0>();
        }
      }
      // O^T += V^T.P^T: k-slot e of lane group g in 16-key half ts is key 16 ts + 8 (e / 4) + 4 g + e % 4
      const int i16 = c & 15, j16 = c >> 4;
      // (row r0 + 8 has the swizzle of r0 with bit 1 flipped)
      uint32_t v_turn = uint32_t((2 * j16 + ((i16 & 3) >> 1)) ^ swizzle(4 * g + (i16 >> 2))) * 16u;
      if constexpr (SHARED) asm volatile("" : "+v"(v_turn));
      auto v_frag = [&](const uint8_t* tile, int ts, int dt) {
        if constexpr (SHARED) {
          const uint8_t* row = tile + (16 * ts + 4 * g + (i16 >> 2)) * Traits::kRowBytes + (i16 & 1) * 8;
          const uint8_t* a0 = row + ((64u * dt) ^ v_turn);
          const uint8_t* a1 = row + 8 * Traits::kRowBytes + ((64u * dt) ^ v_turn ^ 32u);
          const u32x2_t lo = __builtin_bit_cast(
              u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(a0)));
          const u32x2_t hi = __builtin_bit_cast(
              u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(a1)));
          return u32x4_t{lo[0], lo[1], hi[0], hi[1]};
        }
        const int chunk = 2 * (2 * dt + j16) + ((i16 & 3) >> 1);
        const int r0 = 16 * ts + 4 * g + (i16 >> 2), r1 = r0 + 8;
        const uint8_t* a0 = tile + tile_at(r0, chunk) + (i16 & 1) * 8;
        const uint8_t* a1 = tile + tile_at(r1, chunk) + (i16 & 1) * 8;
        const u32x2_t lo = __builtin_bit_cast(
            u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(a0)));
        const u32x2_t hi = __builtin_bit_cast(
            u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(a1)));
        return u32x4_t{lo[0], lo[1], hi[0], hi[1]};
      };
      // (the fragments of the first half are fetched under the weights)
      constexpr bool FETCHED = DIRECT && DT <= 4 && !decltype(again)::value;
      u32x4_t vf[DT];
      if constexpr (FETCHED) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) vf[dt] = v_frag(sV, 0, dt);
        __builtin_amdgcn_sched_barrier(0);
      }
      // The weights, in place of the scores, and their parts.
      u32x4_t pb[PARTS][2];
      auto split = [&](int r) {
        float p0 = st[r], p1 = st[r + 1];
#pragma unroll
        for (int n = 0; n < PARTS; ++n) pb[n][r >> 3][(r & 7) >> 1] = split_part<BF16, SHORT>(p0, p1);
      };
      float sum = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float x = __builtin_amdgcn_exp2f(__builtin_fmaf(st[r], p.sl2, kShift - m_ref));
        sum += x;
        st[r] = x;
        if (!decltype(again)::value && (r & 1)) split(r - 1);
      }
      l_run += sum;
      if constexpr (decltype(again)::value) {
        // one key after the other, without those of weight zero
#pragma unroll 1
        for (int key = 0; key < 32; ++key) {
          const int r = (key >> 3) * 4 + (key & 3);  // its register in half-wave (key / 4) % 2
          float weight = 0.f;
#pragma unroll
          for (int i = 0; i < 16; ++i) weight = i == r ? st[i] : weight;
          weight = __shfl(weight, c + 32 * ((key >> 2) & 1), 64);
          // (the fences keep this path from costing the first walk registers)
          int turn = swizzle(key) * 16;
          const uint8_t* row = sV + key * Traits::kRowBytes;
          asm volatile("" : "+v"(turn));
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
              __builtin_amdgcn_sched_barrier(0);
              const u32x2_t four = *reinterpret_cast<const u32x2_t*>(row + ((4 * dt + r4) * 16 ^ turn) + 8 * g);
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const uint32_t pair = four[i >> 1];
                const float x = to_float<BF16>((i & 1 ? pair >> 16 : pair) & 0xffffu), y = ot[dt][4 * r4 + i];
                ot[dt][4 * r4 + i] = weight != 0.f ? __builtin_fmaf(weight, x, y) : y;
              }
            }
          }
        }
      }
      if constexpr (!decltype(again)::value && SHARED) {
        constexpr int FAR = 3;  // fragments in flight
        u32x4_t a[FAR];
#pragma unroll
        for (int j = 0; j < FAR; ++j) a[j] = v_frag(sV, j / DT, j % DT);
#pragma unroll
        for (int j = 0; j < 2 * DT; ++j) {
#pragma unroll
          for (int n = 0; n < PARTS; ++n) ot[j % DT] = mfma<BF16>(a[j % FAR], pb[n][j / DT], ot[j % DT]);
          if (j + FAR < 2 * DT) a[j % FAR] = v_frag(sV, (j + FAR) / DT, (j + FAR) % DT);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if constexpr (!decltype(again)::value) {
#pragma unroll
        for (int ts = 0; ts < (SHARED ? 0 : 2); ++ts) {
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            const u32x4_t a = FETCHED ? vf[dt] : v_frag(sV, ts, dt);
#pragma unroll
            for (int n = 0; n < PARTS; ++n) ot[dt] = mfma<BF16>(a, pb[n][ts], ot[dt]);
            if constexpr (FETCHED) if (ts == 0) vf[dt] = v_frag(sV, 1, dt);
          }
        }
        // Weights below 1/2 (2^-(1 + kShift) of the reference) may have bits below 2^-24, where fp16 ends: that rest,
        // times 2^39, in two rounded parts.  (Nothing above 2^-74 of the reference is dropped; beside a maximum that
        // a V row of zeros belongs to, small weights are the result.)
        if (!BF16 && __builtin_amdgcn_ballot_w64(__builtin_fmaf(mn, p.sl2, kShift - m_ref) < -1.f) != 0) {
          u32x4_t part[2][2];
#pragma unroll
          for (int r = 0; r < 16; r += 2) {
            float p0 = st[r], p1 = st[r + 1];
            asm volatile("" : "+v"(p0), "+v"(p1));  // (nothing of this path is worked out before it)
            p0 = __builtin_amdgcn_fractf(p0 * 0x1p24f) * 0x1p15f;
            p1 = __builtin_amdgcn_fractf(p1 * 0x1p24f) * 0x1p15f;
#pragma unroll
            for (int n = 0; n < 2; ++n) {
              const f16x2_t h = {(_Float16)p0, (_Float16)p1};
              part[n][r >> 3][(r & 7) >> 1] = __builtin_bit_cast(uint32_t, h);
              p0 -= float(h[0]);
              p1 -= float(h[1]);
            }
          }
          int fresh = 0;  // (an offset that the compiler knows nothing about: it would otherwise keep the
          asm volatile("" : "+v"(fresh));  // fragments of this path in registers for the products below)
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            __builtin_amdgcn_sched_barrier(0);
            f32x16_t add = zero16;
#pragma unroll
            for (int ts = 0; ts < 2; ++ts) {
              const u32x4_t a = v_frag(sV + fresh, ts, dt);
#pragma unroll
              for (int n = 0; n < 2; ++n) add = mfma<BF16>(a, part[n][ts], add);
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) ot[dt][r] = __builtin_fmaf(add[r], 0x1p-39f, ot[dt][r]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if constexpr (SHARED) {
        go = more();
        if (go) {
          advance();
          load_tile(again, true, k_slab, rK, p.k_at.row, sK);
        }
      } else {
        if (go) load_tile(again, false, v_slab, rV, p.v_at.row, sV);
      }
    }
  };
  if (go) {
    first_rows(std::false_type{});
    walk(std::false_type{});
    float probe = 0.f;  // becomes NaN with any sum that is not finite
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) probe = __builtin_fmaf(ot[dt][r], 0.f, probe);
    if (__builtin_amdgcn_ballot_w64(probe != probe) != 0) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) ot[dt] = zero16;
      l_run = 0.f;
      m_run += kSlack;  // no score is beyond this: weights stay below 2^kShift, nothing is rescaled
      first_step();
      go = true;
      first_rows(std::true_type{});
      walk(std::true_type{});
    }
  }

  // Merge: row maxima and sums of the waves, then the O^T tiles, kGroup at a time: every wave
  // writes its tiles, wave i adds up and stores tile i of the group.
  {
    float lower, upper;
    both_halves<DIRECT>(l_run, lower, upper);
    l_run = lower + upper;
  }
  if (g == 0) {
    sStat[w * 32 + c] = m_run;
    sStat[(NW + w) * 32 + c] = l_run;
  }
  __syncthreads();
  float m_all = -INFINITY;
#pragma unroll
  for (int i = 0; i < NW; ++i) m_all = fmaxf(m_all, sStat[i * 32 + c]);
  const float m_fin = m_all == -INFINITY ? 0.f : m_all;
  float l_all = 0.f;
#pragma unroll
  for (int i = 0; i < NW; ++i)
    l_all += sStat[(NW + i) * 32 + c] * __builtin_amdgcn_exp2f(sStat[i * 32 + c] - m_fin);
  const bool some = q_live && l_all > 0.f;
  const bool empty = !q_live || m_all == -INFINITY;  // no score above minus infinity (:177-183)
  const float inv = some ? 1.f / l_all : 0.f;  // :283-288; rows without a key: zeros (:177-183)
  const float mine = __builtin_amdgcn_exp2f(m_run - m_fin) * inv;
  if (w == 0 && g == 0 && q_here && p.lse)
    p.lse[size_t(bh) * p.S + q_idx] = some ? (m_fin + __builtin_amdgcn_logf(l_all) - kShift) * 0.6931471805599453f : -INFINITY;
  float* const stage = reinterpret_cast<float*>(lds);
  constexpr int G = Traits::kGroup;
  // A list of no more steps than half of the waves leaves the others nothing to add.  (Rows at any alignment beyond 128
  // columns, where eight waves took longer over such lists than four: B=1 H=8 S=128 bf16, four waves -> eight -> so, D=131 11.4
  // -> 10.2 -> 9.6 us, D=165 13.5 -> 11.6 -> 10.9, D=225 14.7 -> 15.1 -> 14.2; B=8 H=32 D=225 63.5 -> 65.1 -> 62.7.
  // Elsewhere eight waves take no longer, and the question costs long lists 0.1 us.)
  const bool half_full = ROWS_IN_LDS && (long long)nb * p.kb_eff <= 32 * (NW / 2);
#pragma unroll
  for (int d0 = 0; d0 < DT; d0 += G) {
    if (d0 > 0) __syncthreads();  // the previous group has been read
    if (!half_full || w < NW / 2) {
#pragma unroll
      for (int i = 0; i < G; ++i) {
        if (d0 + i >= DT) continue;
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
          f32x4_t x;
#pragma unroll
          for (int j = 0; j < 4; ++j) x[j] = ot[d0 + i][4 * r4 + j] * mine;
          *reinterpret_cast<f32x4_t*>(stage + ((size_t(w) * G + i) * 4 + r4) * 256 + lane * 4) = x;
        }
      }
    }
    __syncthreads();
    // pieces (tile, four registers) of the group, dealt to the waves
    for (int u = w; u < 4 * G; u += NW) {
      const int i = u >> 2, r4 = u & 3;
      if (d0 + i >= DT) break;
      f32x4_t x = {0.f, 0.f, 0.f, 0.f};
      auto add = [&](int j) { x += *reinterpret_cast<const f32x4_t*>(stage + ((size_t(j) * G + i) * 4 + r4) * 256 + lane * 4); };
      if (half_full) {
#pragma unroll
        for (int j = 0; j < NW / 2; ++j) add(j);
      } else {
#pragma unroll
        for (int j = 0; j < NW; ++j) add(j);
      }
      if (empty) x = f32x4_t{0.f, 0.f, 0.f, 0.f};
      const int d = 32 * (d0 + i) + 8 * r4 + 4 * g;
      uint16_t* orow = p.o + (size_t(bh) * p.S + q_idx) * p.D;
      uint16_t hv[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) hv[j] = from_float<BF16>(x[j]);
      if (q_here) {
        if (p.o_vec) {  // D is a multiple of 8: four columns are inside together
          if (d < p.D) {
            const u32x2_t two = {uint32_t(hv[0]) | uint32_t(hv[1]) << 16, uint32_t(hv[2]) | uint32_t(hv[3]) << 16};
            *reinterpret_cast<u32x2_t*>(orow + d) = two;
          }
        } else {
          const int chunk = d & ~7;
          const int col = R == Rows::kSmall ? d : chunk_start(chunk, p.D) + (d & 7);
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (chunk < p.D && col + j < p.D && col + j >= chunk) orow[col + j] = hv[j];
        }
      }
    }
  }
}

template <bool BF16, int DT, int NW, Rows R>
__global__ void __launch_bounds__(64 * NW, DT == 1 && NW == 8 ? 4 : 2) fwd_generic_kernel(const GenericParams p) {
  generic_walk<BF16, DT, NW, R>(p);
}
// Steps that may cross a block.
template <bool BF16, int DT, int NW, Rows R>
__global__ void __launch_bounds__(64 * NW, DT == 1 && NW == 8 ? 4 : 2) fwd_generic_steps_kernel(const GenericParams p) {
  generic_walk<BF16, DT, NW, R>(p);
}

constexpr int kMaxDevices = 64;

template <bool BF16, int DT, int NW, Rows R>
int launch(const GenericParams& p, unsigned grid, hipStream_t stream) {
  const void* fn;
  if constexpr (R == Rows::kHalves || R == Rows::kKeys) {
    fn = reinterpret_cast<const void*>(fwd_generic_steps_kernel<BF16, DT, NW, R>);
  } else {
    fn = reinterpret_cast<const void*>(fwd_generic_kernel<BF16, DT, NW, R>);
  }
  constexpr int lds = int(GenericTraits<DT, NW>::kLdsBytes);
  static_assert(lds <= 160 * 1024, "LDS of a compute unit");
  if (lds > 48 * 1024) {  // the dynamic-LDS limit of an instance is raised once per device
    static std::atomic<bool> raised[kMaxDevices];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return int(e);
    const bool cached = dev >= 0 && dev < kMaxDevices;
    if (!cached || !raised[dev].load(std::memory_order_acquire)) {
      e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      if (e != hipSuccess) return int(e);
      if (cached) raised[dev].store(true, std::memory_order_release);
    }
  }
  GenericParams params = p;
  params.adv_slot = 32 * NW / p.kb_eff;
  params.adv_off = 32 * NW % p.kb_eff;
  params.by_slabs = omni_attn::fast_div(p.n_slabs);
  params.by_tiles = omni_attn::fast_div(uint32_t(p.q_tiles));
  params.by_heads = omni_attn::fast_div(uint32_t(p.H));
  void* args[] = {&params};
  return int(hipLaunchKernel(fn, dim3(grid), dim3(64 * NW), args, lds, stream));
}

template <bool BF16, int DT>
int launch_rows(const GenericParams& p, Rows rows, unsigned grid, hipStream_t s) {
  return rows == Rows::kWhole    ? launch<BF16, DT, 8, Rows::kWhole>(p, grid, s)
         : rows == Rows::kHalves ? launch<BF16, DT, 8, Rows::kHalves>(p, grid, s)
         : rows == Rows::kKeys   ? launch<BF16, DT, 8, Rows::kKeys>(p, grid, s)
                                 : launch<BF16, DT, 8, Rows::kWide>(p, grid, s);
}

template <bool BF16, int... I>
int launch_tiles(const GenericParams& p, Rows rows, unsigned grid, hipStream_t s, std::integer_sequence<int, I...>) {
  if (rows == Rows::kSmall) return launch<BF16, 1, 4, Rows::kSmall>(p, grid, s);
  int rc = int(hipErrorInvalidValue);
  ((((p.D + 31) / 32 == I + 1) ? (void)(rc = launch_rows<BF16, I + 1>(p, rows, grid, s)) : (void)0), ...);
  return rc;
}

}  // namespace

namespace omni_attn {
int forward_generic(const void* q, const void* k, const void* v, const omni_attn_strides& q_at,
                    const omni_attn_strides& k_at, const omni_attn_strides& v_at, int S_out, void* o,
                    float* lse_or_null, const int32_t* kv_num_blocks, const int32_t* kv_indices,
                    const int32_t* block_mask_types, const int32_t* partial_idx_or_null,
                    const uint8_t* partial_masks_or_null, int B, int H, int S_pad, int D, int Tq, int max_blocks,
                    int QB, int KB, int num_partial, int seqlen_orig, int dtype, float softcap, void* stream) {
  if (!q || !k || !v || !o || !kv_num_blocks || !kv_indices || !block_mask_types)
    return OMNI_ATTN_ERR_NULL_POINTER;
  const auto misaligned = [](const void* ptr, uintptr_t a) { return (reinterpret_cast<uintptr_t>(ptr) & (a - 1)) != 0; };
  if (misaligned(q, 2) || misaligned(k, 2) || misaligned(v, 2) || misaligned(o, 2) || misaligned(lse_or_null, 4) ||
      misaligned(kv_num_blocks, 4) || misaligned(kv_indices, 4) || misaligned(block_mask_types, 4) ||
      misaligned(partial_idx_or_null, 4))
    return OMNI_ATTN_ERR_MISALIGNED;
  if (dtype != OMNI_ATTN_DTYPE_F16 && dtype != OMNI_ATTN_DTYPE_BF16) return OMNI_ATTN_ERR_UNSUPPORTED_DTYPE;
  if (D <= 0 || D > kMaxD) return OMNI_ATTN_ERR_UNSUPPORTED_HEAD_DIM;  // the reference's bound, attn_naive.cu:189-190
  if (QB <= 0 || KB <= 0) return OMNI_ATTN_ERR_UNSUPPORTED_BLOCK;
  if (B <= 0 || H <= 0 || S_pad <= 0 || Tq <= 0 || max_blocks <= 0 || seqlen_orig < 0 || num_partial < 0 ||
      !(softcap >= 0.f) || std::isinf(softcap))
    return OMNI_ATTN_ERR_BAD_SHAPE;
  // (rows of the last query block are ints, also those behind the sequence)
  if ((long long)S_pad + QB - 1 > 0x7fffffffLL || Tq != omni_attn::blocks_of(S_pad, QB)) return OMNI_ATTN_ERR_BAD_SHAPE;
  const long long rows = (long long)B * H * S_pad;
  if ((long long)S_pad * D > 0x7fffffffLL || rows > (1LL << 33) || (long long)B * H * Tq * max_blocks > (1LL << 40))
    return OMNI_ATTN_ERR_TOO_LARGE;
  GenericParams p;
  p.q = static_cast<const uint16_t*>(q);
  p.k = static_cast<const uint16_t*>(k);
  p.v = static_cast<const uint16_t*>(v);
  p.o = static_cast<uint16_t*>(o);
  p.q_at = q_at;
  p.k_at = k_at;
  p.v_at = v_at;
  p.lse = lse_or_null;
  p.kv_num_blocks = kv_num_blocks;
  p.kv_indices = kv_indices;
  p.types = block_mask_types;
  const bool has_partial = partial_idx_or_null && partial_masks_or_null && num_partial > 0;
  p.partial_idx = has_partial ? partial_idx_or_null : nullptr;
  p.partial_masks = has_partial ? partial_masks_or_null : nullptr;
  p.num_partial = has_partial ? num_partial : 0;
  p.S = S_out;
  p.D = D;
  p.H = H;
  p.Tq = Tq;
  p.Tk = omni_attn::blocks_of(S_pad, KB);
  p.max_blocks = max_blocks;
  p.QB = QB;
  p.KB = KB;
  p.seqlen = seqlen_orig < S_pad ? seqlen_orig : S_pad;
  p.kb_eff = omni_attn::walked_keys(KB, S_pad, 1);
  p.q_tiles = omni_attn::blocks_of(QB < S_pad ? QB : S_pad, 32);
  p.mask_words = KB % 4 == 0 && p.kb_eff % 4 == 0 && !misaligned(partial_masks_or_null, 4);
  p.whole = KB % 32 == 0 && !misaligned(partial_masks_or_null, 4);
  p.n_slabs = unsigned(B) * unsigned(H);
  p.scale = float(1.0 / std::sqrt(double(D)));
  p.softcap = softcap;
  // the factor of the scores in the log2 domain (a soft-capped score is scaled before the cap)
  p.sl2 = softcap > 0.f ? 1.4426950408889634f : float(1.4426950408889634 / std::sqrt(double(D)));
  p.o_vec = D % 8 == 0 && !misaligned(o, 8);
  const long long grid = (long long)B * H * Tq * p.q_tiles;
  if (grid > 0x7fffffffLL) return OMNI_ATTN_ERR_TOO_LARGE;
  const auto direct = [&](const void* ptr, const omni_attn_strides& at) {  // 32-bit offsets inside a slab
    return !misaligned(ptr, 16) && at.batch % 8 == 0 && at.head % 8 == 0 && at.row % 8 == 0 && at.row >= D &&
           ((long long)p.seqlen + 32) * at.row * 2 < 0xffffff00LL - kBack;  // (a step that is not read begins behind the sequence)
  };
  const bool halves = KB % 16 == 0 && !misaligned(partial_masks_or_null, 4);  // half a step never crosses a block
  const Rows reads = D < 8                                                         ? Rows::kSmall
                     : !(D % 8 == 0 && direct(k, k_at) && direct(v, v_at))         ? Rows::kWide
                     : p.whole                                                     ? Rows::kWhole
                     : halves                                                      ? Rows::kHalves
                                                                                   : Rows::kKeys;
  // (the keys of such a block behind the sequence are masked like any others, up to the end of a step)
  if (p.whole || reads == Rows::kHalves) p.kb_eff = omni_attn::walked_keys(KB, S_pad, p.whole ? 32 : 16);
  const auto tiles = std::make_integer_sequence<int, kMaxD / 32>{};
  const int e = dtype == OMNI_ATTN_DTYPE_BF16
                    ? launch_tiles<true>(p, reads, unsigned(grid), static_cast<hipStream_t>(stream), tiles)
                    : launch_tiles<false>(p, reads, unsigned(grid), static_cast<hipStream_t>(stream), tiles);
  if (e != 0) {
    omni_attn::record_hip_error(e);
    return OMNI_ATTN_ERR_LAUNCH;
  }
  return OMNI_ATTN_OK;
}
}  // namespace omni_attn

extern "C" int omni_attn_fwd_generic_gfx950(const void* q, const void* k, const void* v, void* o,
                                            float* lse_or_null, const int32_t* kv_num_blocks,
                                            const int32_t* kv_indices, const int32_t* block_mask_types,
                                            const int32_t* partial_idx_or_null,
                                            const uint8_t* partial_masks_or_null, int B, int H, int S_pad,
                                            int D, int Tq, int max_blocks, int QB, int KB, int num_partial,
                                            int seqlen_orig, int dtype, float softcap, void* stream) {
  const omni_attn_strides at = {int64_t(H) * S_pad * D, int64_t(S_pad) * D, D};
  return omni_attn::forward_generic(q, k, v, at, at, at, S_pad, o, lse_or_null, kv_num_blocks, kv_indices,
                                    block_mask_types, partial_idx_or_null, partial_masks_or_null, B, H, S_pad, D, Tq,
                                    max_blocks, QB, KB, num_partial, seqlen_orig, dtype, softcap, stream);
}
