// Block-sparse FlashAttention-2 forward for gfx950 (MI355X, CDNA4).
//
// One workgroup owns one query block (QB rows) of one (batch, head) and walks only
// the KV blocks listed for it, like the reference's per-Q-block CTA
// (omni-attn-mma/mma/omni_attn_shared_kv.cu:33-647); the mask semantics are those of
// the reference's scalar kernel (omni-attn-mma/mma/attn_naive.cu:21-302).
//
// Everything is computed transposed so that one lane owns one query row:
//   S^T[kv, q] = K[kv, :] . Q[q, :]      A = K tile (LDS), B = Q (registers)
//   O^T[d,  q] = V^T[d, kv] . P^T[kv, q]  A = V^T (LDS transpose read), B = P^T
// With v_mfma_f32_32x32x16 the accumulator of S^T puts query row (lane % 32) in a
// lane and 16 kv positions in its registers, which is exactly the B-operand layout
// the second product needs: P never leaves registers, row sums (and maxima, in the few steps
// that look at them) are in-lane reductions plus one exchange with lane ^ 32, and the
// online-softmax rescale is a per-lane scalar.
//
// A wave owns 32 query rows; a workgroup has QB/32 waves.  KV blocks are consumed in
// steps of 64 keys (a 128-key block is two steps; 32 keys for 64-row query blocks).  K and
// V tiles are double-buffered in LDS and filled by direct buffer->LDS loads (no register
// staging, out-of-range rows read as zeros).
//
// The walk is software-pipelined so that the matrix cores and the vector ALU work on
// different steps inside ONE instruction stream: iteration i of a wave issues the 2*D/16
// MFMAs of S^T(i+1) and the D/8 MFMAs of O^T += V^T.P^T(i-1) while its vector
// instructions do the online softmax of step i.  None of the three depends on another
// inside the iteration, and the source spells the interleaving out: the iteration is a
// sequence of slots, each with one MFMA, the LDS fetch of the operand three slots ahead, a
// share of the softmax and -- in the early slots -- one tile load, with a scheduling fence
// after every slot.  (A wave that issues MFMAs back to back leaves other waves of its
// SIMD almost no vector issue slots; vector instructions placed between the MFMAs of the
// same wave are nearly free.)  Two iterations are unrolled so that the accumulators of
// S^T and the packed P alternate between two register sets without copies.
// One workgroup barrier per step.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <utility>

#include "omni_attn_deal.hpp"
#include "omni_attn_split_rules.hpp"

namespace omni_attn {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2_t;
typedef __attribute__((ext_vector_type(4))) short s16x4_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;

enum : int { kMasked = 0, kCausal = 1, kFull = 2, kPartial = 3 };

// The hipError_t of the last HIP call of this thread that made an entry point return
// OMNI_ATTN_ERR_LAUNCH (read back through omni_attn_last_hip_error()); defined beside that function.
void record_hip_error(int hip_error);

// Where the rows of a [B, H, rows, D] operand lie, in elements (multiples of 8; the last dimension is
// contiguous): a projection's [B, rows, H, D] result is read as it is.
struct RowStrides {
  int64_t b, h;
  uint32_t row;
};

struct FwdParams {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  RowStrides q_at, k_at, v_at;  // (o is contiguous; K and V have one row stride)
  uint16_t* o;
  float* lse;                    // may be null
  const int32_t* kv_num_blocks;  // [B,H,Tq]
  const int32_t* kv_indices;     // [B,H,Tq,max_blocks]
  const int32_t* types;          // [B,H,Tq,max_blocks]
  const int32_t* partial_idx;    // [B,H,Tq,max_blocks] (any such array where num_partial is 0)
  const uint8_t* partial_masks;  // [P,QB,KB] bytes or null
  const uint32_t* partial_bits;  // [P,QB,KB/32] words (bit j of word c = key 32c + j) or null;
                                 // at most one of partial_masks / partial_bits is set
  int num_partial; // P: tiles stored in partial_masks
  int S;           // padded sequence length (rows per (b,h) slab)
  int Tq;          // query blocks per slab
  int Tk;          // ceil(S / KB)
  int max_blocks;  // slots per query block
  int seqlen;      // min(seqlen_orig, S): rows/keys at or beyond it are padding
  int H;
  FwdSplit split;  // how the walks are split over waves
  int QB, KB;      // block sizes
  int tiles;       // workgroups per slab (query blocks, or parts of them)
  int parts;       // parts a slab is dealt to the XCDs in
  int n_slabs;     // B*H
  DealPlan deal;
  int n_xcd;       // XCDs (L2 domains) of the device; workgroup ids go round-robin over them
  int slab_group;  // slabs of one XCD that are walked together (>= 1)
  int flat_first;  // (at most 64 slabs per XCD) slabs without short lists go first
  float sl2;       // log2(e) / sqrt(D); log2(e) when scores are soft-capped (they are scaled there)
  float softcap;   // > 0: scores s / sqrt(D) are replaced by softcap * tanh(s / sqrt(D) / softcap)
  float cap_c2;    // 2 * log2(e) / (sqrt(D) * softcap)
};

template <bool BF16>
__device__ __forceinline__ f32x16_t mfma_32x32x16(u32x4_t a, u32x4_t b, f32x16_t c) {
  if constexpr (BF16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  }
}

// Two fp32 values -> two 16-bit values (round to nearest even), low half first.
template <bool BF16>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  if constexpr (BF16) {
    bf16x2_t v = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, v);
  } else {
    f16x2_t v = {(_Float16)lo, (_Float16)hi};
    return __builtin_bit_cast(uint32_t, v);
  }
}

// 32 mask bytes -> 32 bits, byte i -> bit i; any non-zero byte means attend (attn_naive.cu:151).  Bit 7 of a
// byte is brought to that, and the dot products of eight such bytes with 1, 2, 4 .. 128 are 128 times their bits:
// 41 vector instructions (folding each byte onto its lowest bit and multiplying the nibbles out: 80).
__device__ __forceinline__ uint32_t pack_mask_bytes(u32x4_t m0, u32x4_t m1) {
  uint32_t part[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t sum = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t x = i < 2 ? m0[2 * i + h] : m1[2 * i + h - 4];
      const uint32_t set = (((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) & 0x80808080u;
      sum = __builtin_amdgcn_udot4(set, h == 0 ? 0x08040201u : 0x80402010u, sum, false);
    }
    part[i] = sum;
  }
  return (part[0] >> 7) | (part[1] << 1) | (part[2] << 9) | (part[3] << 17);
}

// LDS tiles are [64 rows][D] 16-bit elements with no padding; 16-byte chunks are
// XOR-swizzled inside a row so that the operand reads are bank-conflict free.
// K is read with ds_read_b128 by 32 consecutive rows at one chunk column: the chunk
// index is XORed with the row so 16 consecutive rows cover all 64 banks.
template <int D>
__device__ __forceinline__ int k_swizzle(int row) {
  constexpr int C = D / 8;  // 16-byte chunks per row
  return (row / (16 / C)) % C;
}
// V is read with ds_read_b64_tr_b16: within 16 lanes, 4 lanes read 32 contiguous bytes
// of one row and the next 4 lanes the next row; lanes 16-31 read the neighbouring 32-byte
// unit of the same 4 rows.  Bit 0 of the unit index (which half-wave group) is left
// alone and the higher bits are XORed with the row, so the 32 lanes that are served
// together touch 8 different 32-byte bank groups.
template <int D>
__device__ __forceinline__ int v_swizzle(int row) {
  constexpr int U = D / 16;  // 32-byte units per row
  if constexpr (U <= 2) return 0;
  return 2 * ((row / (8 / U)) % (U / 2));
}

__device__ __forceinline__ s16x4_t lds_read_tr16(const uint16_t* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4_t*)(p));
}

// Exchange between the lane pair (l, l ^ 32) without touching LDS: v_permlane32_swap
// swaps the upper 32 lanes of its first operand with the lower 32 lanes of its second,
// so with x in both operands one result holds {lo, lo} and the other {hi, hi}.
// (The elements are copied to scalars before the bit cast: a bit cast applied directly
// to a vector element expression reads element 0 for both.)
__device__ __forceinline__ void pair_split(float x, float& lo, float& hi) {
  typedef __attribute__((ext_vector_type(2))) unsigned u2;
  const unsigned a = __builtin_bit_cast(unsigned, x);
  const u2 r = __builtin_amdgcn_permlane32_swap(a, a, false, false);
  const unsigned r0 = r[0], r1 = r[1];
  lo = __builtin_bit_cast(float, r0);
  hi = __builtin_bit_cast(float, r1);
}
// Maximum of values that are never NaN, as exactly one v_max_f32 / v_max3_f32 (the library
// function also quiets signalling NaNs: one more instruction for every operand the compiler
// knows nothing about).
__device__ __forceinline__ float vmax(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float vmax3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ float pair_max(float x) {
  float lo, hi;
  pair_split(x, lo, hi);
  return vmax(lo, hi);
}
__device__ __forceinline__ float pair_sum(float x) {
  float lo, hi;
  pair_split(x, lo, hi);
  return lo + hi;
}

// How a workgroup walks: QT query rows of one query block (QT / 32 waves), KG groups of such waves that
// share the steps of the list (group i takes the steps i, i + KG, ...) and merge their results at the
// end, STEP keys per step.  QB, KB: the block sizes, 0 where they are not known at compile time.
template <bool BF16_, int D_, int QB_, int KB_, int QT_, int KG_, int STEP_>
struct FwdShape {
  static constexpr bool BF16 = BF16_;
  static constexpr int D = D_, QB = QB_, KB = KB_, QT = QT_, KG = KG_, kStep = STEP_;
  static constexpr int kGroupThreads = QT * 2;  // QT/32 waves of 64 lanes
  static constexpr int kThreads = kGroupThreads * KG;
  static constexpr int kTileElems = kStep * D;
  static constexpr bool kLone = QT == 32;  // a group is one wave: its steps need no barriers
  static constexpr int kSets = kLone ? 1 : 2;  // tiles of K, and of V
  // per group: K tiles, V tiles, one mask byte per row and key in transit
  static constexpr size_t kTileBytes = size_t(kSets) * 2 * kTileElems * sizeof(uint16_t);
  static constexpr size_t kGroupBytes = kTileBytes + size_t(QT) * kStep;
  static constexpr size_t kLdsBytes = kGroupBytes * KG;
};

// A lone wave is bound by its own instructions (about one in five cycles) and by what a step costs beside
// its slots, so its steps are long: 64 keys at head_dim <= 64.  What leaves LDS room for that (and for two
// workgroups per compute unit) is one tile of K and one of V: a step fetches all its operands first, and
// the loads of the next tiles go out once they are in registers.  Two tiles each, steps of 32 keys, one
// tile load per instruction group, us -> now: B H=8 D=64 S=512 7.3 -> 6.6, S=2048 16.0 -> 13.5, B H=4 S=4096 26.4 -> 21.5;
// D=32 B H=8 S=2048 13.4 -> 9.7; D=128 (32 keys) B H=4 S=2048 18.6 -> 16.2.  Eight groups of 32 rows: 6.6 -> 8.1
// at S=512, 8.5 -> 9.0 at S=1024 (the merge, and a workgroup of eight waves).

// One workgroup per query block, all steps in one group.
// Keys per step.  A 64-row query block has half the waves; at D = 128 its 64-key tiles would
// leave LDS room for only two workgroups per CU (one wave per SIMD): it steps by 32 keys, four
// workgroups fit and every SIMD has two waves again.  At D <= 64 four workgroups fit with 64-key
// tiles, and a step has twice the matrix work per barrier.
template <bool BF16, int D, int QB, int KB>
using FwdBlockShape = FwdShape<BF16, D, QB, KB, QB, 1, (QB == 64 && D == 128) ? 32 : 64>;

// One step of the walk: kStep keys starting at row0, with the effective block mode.
struct StepInfo {
  int row0;
  int mode;
  int pid;
};

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((ext_vector_type(4))) int32_t i32x4_t;

// Buffer resource for a slab of `bytes` bytes: raw (unstructured) addressing, so a lane
// whose byte offset is at or beyond `bytes` reads zeros instead of faulting.
__device__ __forceinline__ i32x4_t make_buffer_resource(const void* base, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  i32x4_t r;
  r[0] = __builtin_amdgcn_readfirstlane(int32_t(uint32_t(a)));
  r[1] = __builtin_amdgcn_readfirstlane(int32_t(uint32_t(a >> 32) & 0xffffu));
  r[2] = __builtin_amdgcn_readfirstlane(int32_t(bytes));
  r[3] = 0x00020000;
  return r;
}
// First row of slab bh of an operand, and a buffer resource that ends with its last live row (so rows
// at or beyond the sequence read as zeros).
// `heads`: DealPlan's division by H.
__device__ __forceinline__ const uint16_t* row_base(const uint16_t* base, const RowStrides& at, int bh, int H,
                                                    const FastDiv& heads) {
  const int b = int(divide(bh, heads));
  return base + int64_t(b) * at.b + int64_t(bh - b * H) * at.h;
}
template <int D>
__device__ __forceinline__ i32x4_t row_resource(const uint16_t* base, const RowStrides& at, int bh, int H,
                                                const FastDiv& heads, int live) {
  const uint32_t bytes = live > 0 ? uint32_t(live - 1) * at.row * 2u + uint32_t(D * 2) : 0u;
  return make_buffer_resource(row_base(base, at, bh, H, heads), bytes);
}
// 16 bytes per lane from a buffer of rows into registers, at a lane offset and a constant inside the row.  A lane at
// kNoRow gets zeros: no buffer of rows that 32-bit offsets reach ends behind it, and no constant leads past 2^32.  (The
// constant goes with the lane's offset, where the check of the range sees the sum.)
template <int D>
constexpr uint32_t kNoRow = 0u - 2u * uint32_t(D);
__device__ __forceinline__ u32x4_t buffer_load_b128(const i32x4_t& r, uint32_t lane_off, int constant) {
  const uint64_t base = uint64_t(uint32_t(r[0])) | uint64_t(uint32_t(r[1])) << 32;
  auto rsrc = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(base), 0, r[2], r[3]);
  return __builtin_amdgcn_raw_buffer_load_b128(rsrc, int(lane_off) + constant, 0, 0);
}
// 16 bytes per lane from a buffer straight into LDS: the wave's 64 chunks land at
// lds_base + 16 * lane.  The source offset is a wave-uniform part plus a per-lane part.
// Written as inline asm so that the compiler does not order later LDS reads of *other*
// buffers behind it with a vmcnt(0) wait; completion is waited for explicitly (vmcnt(0) +
// workgroup barrier) before the filled buffer is read.
__device__ __forceinline__ void buffer_to_lds_b128(i32x4_t rsrc, uint32_t lane_off,
                                                   uint32_t uniform_off, uint32_t lds_base) {
  // (Every scalar operand goes through readfirstlane: that is free for a value that is
  // already in scalar registers and keeps the operand legal if the compiler has chosen
  // to compute a uniform value with vector instructions.)
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
// Four such loads, 1 KiB of LDS apart.
__device__ __forceinline__ void buffer_to_lds_4xb128(i32x4_t rsrc, const uint32_t (&lane_off)[4],
                                                     const uint32_t (&uniform_off)[4], uint32_t lds_base) {
  i32x4_t r;
  r[0] = __builtin_amdgcn_readfirstlane(rsrc[0]);
  r[1] = __builtin_amdgcn_readfirstlane(rsrc[1]);
  r[2] = __builtin_amdgcn_readfirstlane(rsrc[2]);
  r[3] = __builtin_amdgcn_readfirstlane(rsrc[3]);
  // (the instruction offset counts for both addresses)
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %1, %5, %6 offen lds\n\t"
      "buffer_load_dwordx4 %2, %5, %7 offen offset:1024 lds\n\t"
      "buffer_load_dwordx4 %3, %5, %8 offen offset:2048 lds\n\t"
      "buffer_load_dwordx4 %4, %5, %9 offen offset:3072 lds"
      :
      : "s"(__builtin_amdgcn_readfirstlane(lds_base)), "v"(lane_off[0]), "v"(lane_off[1]), "v"(lane_off[2]),
        "v"(lane_off[3]), "s"(r), "s"(__builtin_amdgcn_readfirstlane(uniform_off[0])),
        "s"(__builtin_amdgcn_readfirstlane(uniform_off[1] - 1024u)),
        "s"(__builtin_amdgcn_readfirstlane(uniform_off[2] - 2048u)),
        "s"(__builtin_amdgcn_readfirstlane(uniform_off[3] - 3072u))
      : "memory", "m0");
}
// 4 bytes per lane: the dword of lane l lands at lds_base + 4 * l (lanes switched off by the
// execution mask neither load nor store).
__device__ __forceinline__ void buffer_to_lds_b32(i32x4_t rsrc, uint32_t lane_off,
                                                  uint32_t uniform_off, uint32_t lds_base) {
  i32x4_t r;
  r[0] = __builtin_amdgcn_readfirstlane(rsrc[0]);
  r[1] = __builtin_amdgcn_readfirstlane(rsrc[1]);
  r[2] = __builtin_amdgcn_readfirstlane(rsrc[2]);
  r[3] = __builtin_amdgcn_readfirstlane(rsrc[3]);
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "buffer_load_dword %1, %2, %3 offen lds"
      :
      : "s"(__builtin_amdgcn_readfirstlane(lds_base)), "v"(lane_off), "s"(r),
        "s"(__builtin_amdgcn_readfirstlane(uniform_off))
      : "memory", "m0");
}
// Waits until this wave's vector-memory operations are complete.  (The builtin, not inline asm: the
// compiler then knows that its own loads have landed too, and does not wait for them again behind
// tile loads that have been issued since.)
__device__ __forceinline__ void wait_loads() {
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  asm volatile("" ::: "memory");
}
// ... all but the N that were issued last.
template <int N>
__device__ __forceinline__ void wait_loads_but() {
  static_assert(N < 64, "six bits");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
  asm volatile("" ::: "memory");
}
// Block-mask metadata is read-only for the whole launch and every read of it is
// wave-uniform: reading it through the constant address space makes these scalar loads
// (SGPR results, no vector-memory latency in the instruction stream).
__device__ __forceinline__ int32_t load_uniform(const int32_t* p) {
  return *reinterpret_cast<const __attribute__((address_space(4))) int32_t*>(
      reinterpret_cast<size_t>(p));
}
__device__ __forceinline__ uint32_t lds_offset_of(const void* p) {
  return uint32_t(size_t((lds_void_t*)p));
}

// An empty asm that "modifies" its operands: the values have to be computed before
// this point of the instruction stream (the optimizer would otherwise sink work whose
// results are only needed much later out of the place it was written in).
__device__ __forceinline__ void pin(float& a) { asm volatile("" : "+v"(a)); }
__device__ __forceinline__ void pin(uint32_t& a) { asm volatile("" : "+v"(a)); }
__device__ __forceinline__ void pin(float& a, float& b) { asm volatile("" : "+v"(a), "+v"(b)); }

template <int V>
struct IntC {
  static constexpr int value = V;
};
// f(IntC<0>{}), f(IntC<1>{}), ... f(IntC<N-1>{}): a loop whose index is a compile-time
// constant inside the body (register arrays indexed with it never go to scratch memory).
template <class F, int... Is>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, Is...>) {
  (f(IntC<Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// Which slab (or part of one) a workgroup has, and which of its tiles, longest first; slab -1: none.
// `group` slabs are walked together (the kernels say why); Params: of the forward or the backward.
struct Dealt {
  int slab, rank;
};
template <class Params>
__device__ __forceinline__ Dealt deal_slab(const Params& p, int group, bool flat_first) {
  const int wg = blockIdx.x;
  const int slot = int(divide(wg, p.deal.xcd));
  const int xcd = wg - slot * p.n_xcd;
  const bool one_more = xcd < p.deal.one_more;
  const int slabs_here = p.deal.slabs + int(one_more);
  const int part_tiles = p.deal.part_tiles;
  if (slot >= slabs_here * part_tiles) return {-1, 0};
  // Batch elements may have different masks.  Slabs whose first query block lists more than half of the
  // KV blocks (nothing is masked, say: all their lists are long) go first, so that the launch ends with
  // short lists: a load at the start of a workgroup, and a sequence of groups for either kind.  Where all
  // slabs are one group: a third of the batch unmasked, D=128 B H=64 S=1536, 67.1 us in groups, 75.6 as one,
  // 63.2 as one with this.  With many groups the load costs 1-2 % and the end of the launch is small.
  uint64_t kind = 0;  // bit i: slab i of this XCD is of the kind that is dealt here (0: all are)
  int at = slot, slabs_kind = slabs_here;
  if (flat_first) {
    const int i = threadIdx.x & 63;
    bool flat = false;
    if (i < slabs_here)
      flat = 2 * p.kv_num_blocks[size_t((xcd + p.n_xcd * i) >> p.deal.part_shift) * size_t(p.Tq)] > p.Tk;
    const uint64_t flats = __builtin_amdgcn_ballot_w64(flat);
    const int n = __builtin_popcountll(flats);
    if (n != 0 && n != slabs_here) {
      const bool early = slot < n * part_tiles;
      kind = __builtin_amdgcn_ballot_w64(i < slabs_here && flat == early);
      at = early ? slot : slot - n * part_tiles;
      slabs_kind = early ? n : slabs_here - n;
    }
  }
  const int per_group = group * part_tiles;
  const int gi = int(divide(at, p.deal.per_group));
  const int in_group = at - gi * per_group;
  const int g_left = slabs_kind - gi * group;
  const int g_eff = g_left < group ? g_left : group;
  int qrank;
  if (g_left >= group) {
    qrank = int(divide(in_group, p.deal.group));
  } else if (kind == 0) {
    qrank = int(divide(in_group, one_more ? p.deal.last[1] : p.deal.last[0]));
  } else {
    qrank = in_group / g_eff;
  }
  int pick = gi * group + (in_group - qrank * g_eff);  // which slab of its kind
  if (kind != 0) {
    const int i = threadIdx.x & 63;
    const int rank = __builtin_amdgcn_mbcnt_hi(uint32_t(kind >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(kind), 0u));
    pick = __builtin_ctzll(__builtin_amdgcn_ballot_w64(((kind >> i) & 1) != 0 && rank == pick));
  }
  return {xcd + p.n_xcd * pick, qrank};
}

template <class Shape>
__device__ __forceinline__ void fwd_walk(const FwdParams& p) {
  constexpr bool BF16 = Shape::BF16;
  constexpr int D = Shape::D;
  constexpr int QT = Shape::QT;
  constexpr int KG = Shape::KG;
  constexpr bool LONE = Shape::kLone;
  constexpr int NT = Shape::kGroupThreads;
  constexpr int STEP = Shape::kStep;
  const int QB = Shape::QB != 0 ? Shape::QB : p.QB;
  const int KB = Shape::KB != 0 ? Shape::KB : p.KB;
  const int SPB = KB / STEP;            // steps per KV block (a power of two)
  constexpr int NTL = STEP / 32;        // 32-key accumulator tiles of S^T per step
  constexpr int CPR = D / 8;            // 16-byte chunks per row
  constexpr int NCH = STEP * CPR / NT;  // 16-byte chunks per thread per tile
  constexpr int KS = D / 16;            // MFMA k-steps of Q.K
  constexpr int DT = D / 32;            // 32-row tiles of O^T
  constexpr int TILE = Shape::kTileElems;
  constexpr int WQ = QT / 32;           // waves of a group
  static_assert(STEP * CPR % NT == 0, "tile must divide over the workgroup");

  const int w_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = KG == 1 ? 0 : w_all / WQ;  // group of the wave (wave-uniform)
  const int w = KG == 1 ? w_all : w_all % WQ;  // wave of the group
  extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
  constexpr int SETS = Shape::kSets;
  uint16_t* sK = reinterpret_cast<uint16_t*>(lds_raw + size_t(kg) * Shape::kGroupBytes);  // [SETS][TILE]
  uint16_t* sV = sK + SETS * TILE;                                  // [SETS][TILE]
  uint8_t* sMaskBytes = reinterpret_cast<uint8_t*>(sV + SETS * TILE);  // [QT][STEP]

  // Workgroup -> (slab, query block).  Consecutive workgroup ids go round-robin over
  // the XCDs.  XCD x takes the slabs bh with bh % n_xcd == x (every batch element's heads
  // are spread over all XCDs, which balances batches with different masks) and works
  // through them in groups of p.slab_group slabs, sized so that one group's query
  // blocks just fill the XCD's workgroup slots: the workgroups that run together then
  // belong to one or two slabs and walk the same K/V rows at about the same time, so
  // each K/V tile is fetched from HBM once and served from the XCD's L2 to the other
  // query blocks.  Inside a group the order is longest-first: query block Tq-1 of each
  // slab of the group, then Tq-2, ...
  // (Launches of few rounds walk all slabs of an XCD as one group.)
  // Where there are too few slabs to go round, a slab is dealt in p.parts parts (part i has the
  // query tiles i, i + parts, ... from the end): "slab" in the lines below is a part then.
  const Dealt deal = deal_slab(p, p.slab_group, p.flat_first != 0);
  if (deal.slab < 0) return;
  const int bh = deal.slab >> p.deal.part_shift;
  const int qt = p.tiles - 1 - ((deal.rank << p.deal.part_shift) + deal.slab - (bh << p.deal.part_shift));  // query tile
  const int q0 = qt * QT;  // first row of this workgroup
  if (qt < 0 || (KG > 1 && q0 >= p.S)) return;
  const int qb = KG == 1 ? qt : q0 >> (QB == 128 ? 7 : 6);
  const int rb0 = KG == 1 ? 0 : q0 - qb * QB;  // ... inside its query block

  static_assert((NT & (NT - 1)) == 0, "threads of a group");
  const int tid = threadIdx.x & (NT - 1);  // thread of the group
  const int lane = tid & 63;
  const int g = lane >> 5;
  const int c = lane & 31;

  const size_t slab = size_t(bh) * size_t(p.S) * D;  // of o
  const int q_row = q0 + 32 * w + c;  // this lane's query row inside the slab
  const int q_wave_min = q0 + 32 * w;

  const size_t meta_row = size_t(bh) * p.Tq + qb;
  const size_t meta_off = meta_row * p.max_blocks;

  // Block metadata lives in registers: lane i of every wave holds the (validated) words of
  // block 64 * chunk + i of this query block's list -- first key row, effective mode,
  // partial-mask index -- and a step's words are picked out with v_readlane: no memory
  // instruction per step.  A new chunk is fetched when the walk reaches it (every 64
  // blocks).  The loads of a chunk do not depend on the block count, so the first chunk,
  // the count and Q are all in flight together at the start of the kernel.
  const bool packed_tiles = p.partial_bits != nullptr;
  int32_t mv_row0 = 0, mv_mode = kMasked, mv_pid = -1;
  struct Raw {
    int32_t kvb, ty, pid;
  };
  auto request_chunk = [&](int chunk) {
    const int j = chunk * 64 + lane;
    const size_t o = meta_off + size_t(j < p.max_blocks ? j : 0);
    return Raw{p.kv_indices[o], p.types[o], p.partial_idx[o]};
  };
  auto take_chunk = [&](const Raw& raw) {
    const int32_t kvb = raw.kvb < 0 ? 0 : (raw.kvb >= p.Tk ? p.Tk - 1 : raw.kvb);
    int32_t mode = (raw.ty == kCausal || raw.ty == kFull || raw.ty == kPartial) ? raw.ty : int32_t(kMasked);
    if (raw.ty == kPartial && (raw.pid < 0 || raw.pid >= p.num_partial)) mode = kMasked;
    mv_row0 = kvb * KB;
    mv_mode = mode;
    mv_pid = raw.pid;
  };
  auto load_chunk = [&](int chunk) { take_chunk(request_chunk(chunk)); };
  // The list and its length are requested as soon as their addresses are known; what else depends on the slab is
  // worked out meanwhile.  (The length was requested behind the list's arrival, and Q with a branch per load:
  // B=2 H=16 S=1237 D=128 unaligned spans 29.3 -> 28.75 us without.)
  int nb = load_uniform(p.kv_num_blocks + meta_row);
  const Raw first_chunk = request_chunk(0);
  __builtin_amdgcn_sched_barrier(0);
  // Rows at or beyond the sequence are never used: the resources of K and V end there (those
  // rows arrive as zeros) and the query rows beyond it are replaced by zeros, whatever the caller
  // left in the padding.
  const uint32_t pitch = p.k_at.row * 2u;  // bytes from row to row of K, and of V
  const i32x4_t rK = row_resource<D>(p.k, p.k_at, bh, p.H, p.deal.heads, p.seqlen);
  const i32x4_t rV = row_resource<D>(p.v, p.v_at, bh, p.H, p.deal.heads, p.seqlen);
  const i32x4_t rQ = row_resource<D>(p.q, p.q_at, bh, p.H, p.deal.heads, p.seqlen);
  // Q as the B operand of S^T = K.Q^T: lane holds Q[q_row][16s + 8g .. +7].  Lone waves ask for it while
  // the list is on its way (D=64 B H=8 S=512 6.33 -> 6.08 us, 64-row blocks S=2048 12.17 -> 12.28), others when it is
  // there (no difference at B H=32 S=1237 D=128).
  u32x4_t qf[KS];
  auto request_q = [&]() {
    const uint32_t at = q_row < p.seqlen ? uint32_t(q_row) * (p.q_at.row * 2u) + 16u * uint32_t(g) : kNoRow<D>;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = buffer_load_b128(rQ, at, 32 * s);
  };
  if constexpr (LONE) request_q();
  take_chunk(first_chunk);
  nb = nb < 0 ? 0 : (nb > p.max_blocks ? p.max_blocks : nb);
  int all_steps = nb * SPB;
  // Groups share the steps of the live slots only (those that allow something), so a list and the same
  // list with MASKED slots in between give the same result bit for bit: the live slots of a chunk are
  // moved to the lanes 0, 1, ...
  const int sub_bits = KG == 1 ? 0 : 31 - __builtin_clz(SPB);
  int chunk_at = 0, live_before = 0, live_here = 0;  // chunk in registers; live slots before it and of it
  auto take_live = [&](int chunk) {
    const bool live = (chunk * 64 + lane < nb) & (mv_mode != kMasked) & (mv_row0 < p.seqlen);
    const uint64_t m = __builtin_amdgcn_ballot_w64(live);
    const int rank = __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u));
    const int rest = __builtin_popcountll(m) + lane - rank;  // (slots that are not live go behind)
    const int to = (live ? rank : rest) * 4;
    mv_row0 = __builtin_amdgcn_ds_permute(to, mv_row0);
    mv_mode = __builtin_amdgcn_ds_permute(to, mv_mode);
    mv_pid = __builtin_amdgcn_ds_permute(to, mv_pid);
    live_here = __builtin_popcountll(m);
  };
  if constexpr (KG > 1) {
    if (q0 >= p.seqlen) nb = 0;
    int live = 0, last_row0 = 0, last_mode = kMasked;
    for (int chunk = 0; chunk * 64 < nb; ++chunk) {
      if (chunk > 0) load_chunk(chunk);
      take_live(chunk);
      if (live_here != 0) {
        live += live_here;
        last_row0 = __builtin_amdgcn_readlane(mv_row0, live_here - 1);
        last_mode = __builtin_amdgcn_readlane(mv_mode, live_here - 1);
      }
    }
    if (nb > 64) {
      load_chunk(0);
      take_live(0);
    }
    all_steps = live << sub_bits;
    if (live > 0) {
      // The last block of a list usually holds the diagonal or the end of the sequence: its steps
      // behind both allow nothing.
      int last_key = p.seqlen - 1;
      if (last_mode == kCausal && q0 + QT - 1 < last_key) last_key = q0 + QT - 1;
      const int useful = last_key < last_row0 ? 0 : (last_key - last_row0) / STEP + 1;
      all_steps -= SPB - (useful < SPB ? useful : SPB);
    }
  }
  const int nsteps = KG == 1 ? all_steps : (all_steps + KG - 1) / KG;  // iterations of every group

  if constexpr (!LONE) request_q();
  // Step `it` (clamped to the last step of the walk; steps past the end are only ever
  // used as the address of a tile load whose data nobody reads).
  auto step_info = [&](int i) {
    const int it = KG == 1 ? i : i * KG + kg;
    StepInfo si;
    int ln;
    if constexpr (KG == 1) {
      const int itc = it < nsteps ? it : nsteps - 1;
      const int j = unsigned(itc) / unsigned(SPB), sub = unsigned(itc) % unsigned(SPB);
      if (itc == it && sub == 0 && (j & 63) == 0 && j > 0) load_chunk(j >> 6);
      ln = j & 63;
      si.row0 = sub * STEP;
    } else {
      if (it >= all_steps) return StepInfo{0, kMasked, -1};  // a step that this group does not have (see the drain)
      const int block = it >> sub_bits;
      while (block >= live_before + live_here) {
        live_before += live_here;
        load_chunk(++chunk_at);
        take_live(chunk_at);
      }
      ln = block - live_before;
      si.row0 = (it & (SPB - 1)) * STEP;
    }
    si.row0 += __builtin_amdgcn_readlane(mv_row0, ln);
    si.mode = __builtin_amdgcn_readlane(mv_mode, ln);
    si.pid = __builtin_amdgcn_readlane(mv_pid, ln);
    return si;
  };

  // Direct buffer->LDS tile load: every lane fetches 16 bytes, the wave's 64 chunks land
  // at consecutive LDS addresses: one wave-wide load fills 64 / CPR rows of the tile.
  // The swizzle is applied on the source side: the lane that fills physical chunk
  // (row, pch) fetches the logical chunk that belongs there.  The swizzle depends on the
  // row modulo 16 at most and a thread's loads are ROW_STRIDE rows apart, so one or two
  // per-lane byte offsets serve all loads of a thread; the rest of the address is
  // wave-uniform and goes through the scalar offset of the load.
  constexpr int ROWS_PER_CALL = 64 / CPR;                // rows filled by one wave-wide load
  constexpr int ROW_STRIDE = ROWS_PER_CALL * (NT / 64);  // rows between a thread's loads
  constexpr int KPER = ROW_STRIDE % 16 == 0 ? 1 : 16 / ROW_STRIDE;  // distinct K lane offsets
  static_assert((KPER * ROW_STRIDE) % 16 == 0, "K swizzle must repeat over a thread's loads");
  static_assert(ROW_STRIDE % 4 == 0, "V swizzle must be the same for all loads of a thread");
  const int ld_row = tid / CPR;  // row of this thread's first load
  const int ld_pch = tid % CPR;
  auto k_off = [&](int row) { return uint32_t(row) * pitch + uint32_t(ld_pch ^ k_swizzle<D>(row)) * 16u; };
  auto v_off = [&](int row) {
    return uint32_t(row) * pitch + uint32_t((((ld_pch >> 1) ^ v_swizzle<D>(row)) << 1) | (ld_pch & 1)) * 16u;
  };
  uint32_t koff[KPER];
#pragma unroll
  for (int i = 0; i < KPER; ++i)
    koff[i] = k_off(ld_row + i * ROW_STRIDE) - uint32_t(i * ROW_STRIDE) * pitch;
  const uint32_t voff = v_off(ld_row);
  const uint32_t lds_k0 = lds_offset_of(sK) + uint32_t(w) * 1024u;
  const uint32_t lds_v0 = lds_offset_of(sV) + uint32_t(w) * 1024u;
  // Load number n of a tile pair: n < NCH is part n of the V tile, the rest the K tile.
  auto issue_load = [&](int n, int buf, int k_row0, int v_row0) {
    const bool is_v = n < NCH;
    const int i = is_v ? n : n - NCH;
    const uint32_t dst = (is_v ? lds_v0 : lds_k0) + uint32_t(buf) * (TILE * 2u) + uint32_t(i) * (NT * 16u);
    const uint32_t row = uint32_t(is_v ? v_row0 : k_row0) + uint32_t(i * ROW_STRIDE);
    buffer_to_lds_b128(is_v ? rV : rK, is_v ? voff : koff[i % KPER], row * pitch, dst);
  };
  // Four of a lone wave's loads (rows ROW_STRIDE apart, which are 1 KiB of its tile).
  auto issue_four = [&](bool is_v, int part, int row0, uint32_t lds_tile) {
    uint32_t lane_off[4], uniform_off[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      lane_off[i] = is_v ? voff : koff[i % KPER];
      uniform_off[i] = uint32_t(row0 + (4 * part + i) * ROW_STRIDE) * pitch;
    }
    buffer_to_lds_4xb128(is_v ? rV : rK, lane_off, uniform_off, lds_tile + uint32_t(part) * 4096u);
  };
  static_assert(!LONE || (NCH % 4 == 0 && 4 % KPER == 0), "loads of a lone wave come in fours");

  // PARTIAL blocks.  The mask of a step is one word per row and 32 keys; lane (g, c) of a wave has word g of row c
  // (of its only word, with steps of 32 keys).  Packed tiles: the word is requested an iteration ahead.  Byte tiles:
  // one iteration ahead each wave fetches the STEP mask bytes of its 32 rows for that step straight into LDS
  // (buffer->LDS loads, no registers; the resource covers exactly the tile); at the end of that iteration a
  // lane looks at the 32 bytes of its word, and packs them unless the tile leaves nothing out.  Writer and readers are
  // the same wave, so no workgroup barrier is needed.
  uint32_t mask_word = 0;
  constexpr int MCPR = STEP / 16;  // 16-byte chunks per row of mask bytes
  auto prefetch_mask_bytes = [&](int it, const StepInfo& si) {
    int l = lane;  // (addresses are worked out here, not kept in registers over the walk)
    asm volatile("" : "+v"(l));
    const int half = (KG == 1 ? it : it * KG + kg) & (SPB - 1);
    const i32x4_t rM = make_buffer_resource(p.partial_masks + size_t(si.pid) * size_t(QB * KB), uint32_t(QB * KB));
    const uint32_t dst = lds_offset_of(sMaskBytes) + uint32_t(w) * uint32_t(32 * STEP);
#pragma unroll
    for (int i = 0; i < MCPR / 2; ++i) {  // 64 / MCPR rows per load
      const uint32_t row = uint32_t(rb0 + 32 * w + i * (64 / MCPR)) + uint32_t(l / MCPR);
      buffer_to_lds_b128(rM, row * uint32_t(KB) + uint32_t(l % MCPR) * 16u, uint32_t(half * STEP),
                         dst + uint32_t(i) * 1024u);
    }
  };
  auto prefetch_mask_word = [&](int it, const StepInfo& si) {
    int l = lane;
    asm volatile("" : "+v"(l));
    const int half = (KG == 1 ? it : it * KG + kg) & (SPB - 1);
    const uint32_t words = uint32_t(QB) * uint32_t(KB / 32);
    auto rM = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(p.partial_bits) + size_t(si.pid) * words, 0,
                                                words * 4u, 0x00020000);
    mask_word = __builtin_amdgcn_raw_buffer_load_b32(
        rM, (uint32_t(32 * w + l % 32) * uint32_t(KB / 32) + uint32_t(NTL == 2 ? l / 32 : 0)) * 4u,
        (uint32_t(rb0) * uint32_t(KB / 32) + uint32_t(half * NTL)) * 4u, 0);
  };
  // A tile that leaves nothing out for the rows of this wave that lie inside the sequence: with a length that is no
  // multiple of the block, every block that the last query block lists is PARTIAL, because rows beyond the sequence
  // attend nothing.
  auto leaves_nothing_out = [&]() { return __builtin_amdgcn_ballot_w64(mask_word != 0xffffffffu && q_row < p.seqlen) == 0; };
  auto pack_own_bytes = [&](int l) {
    const uint8_t* mp = sMaskBytes + size_t(32 * w) * STEP + (l % 32) * STEP + (NTL == 2 ? l & 32 : 0);
    mask_word = pack_mask_bytes(*reinterpret_cast<const u32x4_t*>(mp), *reinterpret_cast<const u32x4_t*>(mp + 16));
  };
  // Returns whether the tile leaves nothing out: whether the lowest bit of every byte is set, as it is in a tensor of
  // booleans (bytes of other values are packed, and looked at again).  (The bytes have landed.)
  auto take_mask_bytes = [&]() {
    int l = lane;
    asm volatile("" : "+v"(l));
    const uint8_t* wave_bytes = sMaskBytes + size_t(32 * w) * STEP;
    bool whole = true;
#pragma unroll
    for (int i = 0; i < NTL; ++i) {  // 16 neighbouring bytes per lane: reads without bank conflicts
      const u32x4_t m = *reinterpret_cast<const u32x4_t*>(wave_bytes + (64 * i + l) * 16);
      whole &= ((m[0] & m[1] & m[2] & m[3] & 0x01010101u) == 0x01010101u) |
               (q_wave_min + (64 * i + l) / MCPR >= p.seqlen);
    }
    if (__builtin_amdgcn_ballot_w64(!whole) == 0) return true;
    pack_own_bytes(l);
    return false;
  };

  // Does this wave's 32 x STEP tile of the step need no mask at all?  (wave-uniform)
  auto unmasked = [&](const StepInfo& si) {
    const bool inside = si.row0 + STEP <= p.seqlen;  // (written without branches: scalar selects)
    const bool full = si.mode == kFull;
    const bool below = (si.mode == kCausal) & (si.row0 + STEP - 1 <= q_wave_min);
    return inside & (full | below);
  };

  // LDS operand fetches.  K: rows 32t + c of the tile at k-step s.
  auto k_frag = [&](const uint16_t* tK, int s, int t) {
    const int row = 32 * t + c;
    const int ch = (2 * s + g) ^ k_swizzle<D>(row);
    return *reinterpret_cast<const u32x4_t*>(tK + row * D + ch * 8);
  };
  // V^T: operand j = (ts, dt) is rows 32 dt .. +31 of V^T (d) at keys 16 ts .. +15; k-slot e
  // of lane group g in k-step ts = (t, s2) is key 32t + 16 s2 + 8(e/4) + 4g + e%4 -- the
  // accumulator order of S^T.
  const int i16 = c & 15;
  const int j16 = c >> 4;
  auto v_frag = [&](const uint16_t* tV, int j) {
    const int ts = j / DT, dt = j % DT;
    const int vrow = 16 * ts + 4 * g + (i16 >> 2);
    const int unit = 2 * dt + j16;
    const int u0 = unit ^ v_swizzle<D>(vrow);
    const int u1 = unit ^ v_swizzle<D>(vrow + 8);
    const s16x4_t lo = lds_read_tr16(tV + vrow * D + u0 * 16 + (i16 & 3) * 4);
    const s16x4_t hi = lds_read_tr16(tV + (vrow + 8) * D + u1 * 16 + (i16 & 3) * 4);
    const u32x2_t lo2 = __builtin_bit_cast(u32x2_t, lo);
    const u32x2_t hi2 = __builtin_bit_cast(u32x2_t, hi);
    const u32x4_t a = {lo2[0], lo2[1], hi2[0], hi2[1]};
    return a;
  };

  const f32x16_t zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  f32x16_t ot[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) ot[dt] = zero16;
  f32x16_t st[2][NTL];   // [set][32-key tile]: S^T of the current / next step, alternating
  u32x4_t pb[2][NTL][2];  // [set][tile][16-key half]: P^T packed to 16 bits, B-operand order
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int t = 0; t < NTL; ++t) {
      st[a][t] = zero16;
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) pb[a][t][s2] = u32x4_t{0u, 0u, 0u, 0u};
    }
  // reference point of the exponentials, log2 domain (score * sl2); -inf: the row has seen no key so far
  float m_run = q_row < p.seqlen ? -INFINITY : 0.f;  // (a row of zeros beyond the sequence needs none)
  float m_ref = 0.f;        // what exponents are taken against: m_run, or 0 where that is -inf
  float l_run = 0.f;        // this lane's share of the running row sum
  // When the reference point moves, the rescale of O waits until the top of the next
  // iteration: the PV product that is in flight still belongs to the old reference.
  float alpha_pending = 1.f;
  // What is owed before the next step (wave-uniform): that rescale; a look at the row maxima, because
  // some row has no reference yet or has outgrown the one it has.
  constexpr uint32_t kOwesRescale = 1, kOwesLook = 2;
  uint32_t owed = kOwesLook;

  // ---- one iteration of the pipeline ----------------------------------------------------
  // SET = it % 2.  Reads K(it+1) from sK[SET^1] into st[SET^1], V(it-1) from sV[SET^1] with
  // pb[SET^1]; softmax of st[SET] into pb[SET]; loads K(it+2) into sK[SET] and V(it) into
  // sV[SET] (both last read one iteration ago).
  constexpr int NQK = NTL * KS;            // MFMAs of S^T
  constexpr int NPV_ALL = (STEP / 16) * DT; // MFMAs of O^T
  constexpr int NL = 2 * NCH;     // tile loads per thread
  constexpr int PF_ALL = LONE ? NQK + NPV_ALL : 3;  // operand fetch distance in slots
  // The reference point of a row's exponentials only has to stay near the running maximum -- the
  // result is the same sum with a different common factor -- so the slots do not look at the maximum
  // at all: a step takes the reference as it is, and its row sums (a lane's 32 weights) tell whether a
  // row has outgrown it.  Beyond kGrown the maxima are looked at before the next step, and the reference of
  // rows that are more than 2^kSlack ahead moves; beyond kRedo the step itself is done again from its
  // scores, which are still in registers (16-bit weights end at 65504; sums and O^T are far from fp32's end).
  // Looked at in every step, on the vector pipe, the maxima cost 27 of a step's 157 vector
  // instructions: B=2 H=32 S=4096 D=128 interleaved 316 -> 301 us, B=4 H=16 S=2048 D=64 causal 54.6 -> 51.2,
  // B=2 H=16 S=8192 D=32 interleaved 259 -> 233.
  constexpr float kSlack = 6.f, kGrown = 0x1p10f, kRedo = 0x1p13f;

  // Mask of a step whose 32x64 tile is not entirely allowed, applied to S^T before the
  // iteration that does its softmax: disallowed scores become -inf.  Register r of tile t
  // holds key  row0 + 32t + 8(r/4) + 4g + r%4.
  auto apply_mask = [&](auto set_c, const StepInfo& si) {
    constexpr int SET = decltype(set_c)::value;
    int limit = p.seqlen - 1;
    if (si.mode == kCausal) limit = limit < q_row ? limit : q_row;
    if (si.mode == kMasked) limit = -1;
    const int lim_l = limit - si.row0 - 4 * g;
    uint32_t kw[NTL];
#pragma unroll
    for (int t = 0; t < NTL; ++t) kw[t] = 0xffffffffu;
    if (si.mode == kPartial) {
      if constexpr (NTL == 2) {
        float w0, w1;
        pair_split(__builtin_bit_cast(float, mask_word), w0, w1);
        kw[0] = __builtin_bit_cast(uint32_t, w0);
        kw[1] = __builtin_bit_cast(uint32_t, w1);
      } else {
        kw[0] = mask_word;
      }
    }
    // the limit becomes part of the bit words: positions 0 .. lim_l - 32t of word t stay
    static_for<NTL>([&](auto tc) {
      constexpr int t = decltype(tc)::value;
      kw[t] >>= 4 * g;
      const int n = lim_l - 32 * t + 1;  // allowed low positions of word t
      const uint32_t low = n >= 32 ? 0xffffffffu : (n <= 0 ? 0u : ((1u << (n & 31)) - 1u));
      kw[t] &= low;
    });
    // two instructions per score: the bit, sign-extended to a full word, selects between the
    // score and -inf
    static_for<16 * NTL>([&](auto ec) {
      constexpr int e = decltype(ec)::value;
      constexpr int t = e / 16, r = e % 16;
      constexpr int kl = 8 * (r >> 2) + (r & 3);
      const uint32_t keep = uint32_t(__builtin_amdgcn_sbfe(int(kw[t]), kl, 1));  // 0 or ~0
      const uint32_t bits = __builtin_bit_cast(uint32_t, float(st[SET][t][r]));
      st[SET][t][r] = __builtin_bit_cast(float, (bits & keep) | (0xff800000u & ~keep));
    });
  };

  // Soft-capped scores (the score_mod of transfusion_pytorch/transfusion.py:358-364, applied to the
  // scaled score as at :958-959 and :968): cap * tanh(x / cap) = cap * (1 - 2 / (exp(2 x / cap) + 1)),
  // written into S^T before the mask and the softmax of the step; the softmax then runs on
  // scores that are already scaled (sl2 = log2 e).
  auto apply_softcap = [&](auto set_c) {
    constexpr int SET = decltype(set_c)::value;
    const float cap = p.softcap, c2 = p.cap_c2;
    static_for<16 * NTL>([&](auto ec) {
      constexpr int e = decltype(ec)::value;
      constexpr int t = e / 16, r = e % 16;
      const float ex = __builtin_amdgcn_exp2f(st[SET][t][r] * c2);
      const float rc = __builtin_amdgcn_rcpf(ex + 1.f);
      st[SET][t][r] = __builtin_fmaf(rc, -2.f * cap, cap);
    });
  };

  // Row maximum of a step's scores, in the log2 domain (the row lives in lanes c and c + 32).
  auto step_max = [&](auto set_c) {
    constexpr int SET = decltype(set_c)::value;
    float a = vmax(st[SET][0][0], st[SET][0][1]), b = vmax(st[SET][0][2], st[SET][0][3]);
    static_for<8 * NTL - 2>([&](auto ic) {
      constexpr int e = 2 * decltype(ic)::value + 4;
      float& m = e & 2 ? b : a;
      m = vmax3(m, st[SET][e / 16][e % 16], st[SET][e / 16][e % 16 + 1]);
    });
    return pair_max(vmax(a, b)) * p.sl2;
  };
  // Pair i of a step's weights, packed for the second product and added to the sums.
  auto weights = [&](auto set_c, auto ic, float& s0, float& s1) {
    constexpr int SET = decltype(set_c)::value, i = decltype(ic)::value;
    constexpr int t = i / 8, r = 2 * (i % 8);
    const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[SET][t][r], p.sl2, -m_ref));
    const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[SET][t][r + 1], p.sl2, -m_ref));
    if constexpr (i == 0) {
      s0 = p0;
      s1 = p1;
    } else {
      s0 += p0;
      s1 += p1;
    }
    uint32_t packed = pack2<BF16>(p0, p1);
    pin(packed);
    pb[SET][t][r >> 3][(r & 7) >> 1] = packed;
    pin(s0, s1);
  };
  // The reference becomes m_new (at least the old one); returns the factor for what was summed against
  // the old one (exactly 0 for a row that has not seen a key yet: its sums are still 0).
  auto set_reference = [&](float m_new) {
    m_ref = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_ref);
    l_run *= alpha;
    m_run = m_new;
    return alpha;
  };
  auto look_again = [&]() { return __builtin_amdgcn_ballot_w64(m_run == -INFINITY) != 0 ? kOwesLook : 0u; };
  auto look = [&](auto set_c) {
    const float m_cand = step_max(set_c);
    // (a step that allows nothing, a MASKED slot say, leaves the look to the next one and changes no bits; groups that
    // share a list have no such slots)
    if (KG == 1 && __builtin_amdgcn_ballot_w64(m_cand != -INFINITY) == 0) return;
    owed = 0;
    if (__builtin_amdgcn_ballot_w64(m_cand > m_run + kSlack) != 0) {
      alpha_pending = set_reference(vmax(m_run, m_cand));
      owed = kOwesRescale;
    }
    owed |= look_again();
  };
  auto redo = [&](auto set_c, float& sum) {
    const float alpha = set_reference(vmax(m_run, step_max(set_c)));
    alpha_pending = owed & kOwesRescale ? alpha_pending * alpha : alpha;
    float s0, s1;
    static_for<8 * NTL>([&](auto ic) { weights(set_c, ic, s0, s1); });
    sum = s0 + s1;
    owed = kOwesRescale | look_again();
  };

  // The operands that were requested from a lone wave's tiles are in registers: the tiles may be overwritten.
  auto tile_read = [&]() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };

  // The first operands of an iteration are fetched right after the barrier, ahead of everything
  // else that happens between two bodies: their LDS latency runs under that bookkeeping.
  auto body_prefetch = [&](auto set_c, auto first_c, u32x4_t* opq) {
    constexpr int SET = decltype(set_c)::value;
    constexpr int NPV = decltype(first_c)::value != 0 ? 0 : NPV_ALL;
    constexpr int NS = NQK + NPV;
    constexpr int PF = PF_ALL < NS ? PF_ALL : NS;
    const uint16_t* tK = LONE ? (NPV == 0 ? sV : sK) : sK + (SET ^ 1) * TILE;  // (K(1) of a lone wave waits in V's tile)
    const uint16_t* tV = LONE ? sV : sV + (SET ^ 1) * TILE;
    static_for<PF>([&](auto nc) {
      constexpr int n = decltype(nc)::value;
      if constexpr (n < NPV) {
        opq[n] = v_frag(tV, n);
      } else {
        opq[n] = k_frag(tK, (n - NPV) / NTL, (n - NPV) % NTL);
      }
    });
  };
  auto body = [&](auto set_c, auto first_c, int k_row0, int v_row0, u32x4_t* opq) {
    constexpr int SET = decltype(set_c)::value;
    // The first iteration of a walk has no previous step: no PV slots.
    constexpr int NPV = decltype(first_c)::value != 0 ? 0 : NPV_ALL;
    constexpr int NS = NQK + NPV;  // slots
    constexpr int LSP = (NS / 2) / NL > 0 ? (NS / 2) / NL : 1;  // slots between tile loads
    constexpr int LPS = (NL * LSP + NS - 1) / NS;               // loads per slot that has some
    constexpr int PF = PF_ALL < NS ? PF_ALL : NS;
    constexpr int NPR = 8 * NTL;          // pairs of exponentials
    const uint16_t* tK = sK + (SET ^ 1) * TILE;
    const uint16_t* tV = sV + (SET ^ 1) * TILE;
    auto operand = [&](int n) { return n < NPV ? v_frag(tV, n) : k_frag(tK, (n - NPV) / NTL, (n - NPV) % NTL); };

    float rs0, rs1;
    // The slots run at a raised wave priority and everything between two bodies (barrier, rescale,
    // mask, metadata of the next steps) at the default one: the other wave of the SIMD, from the
    // other workgroup of the compute unit, is then not held up by this wave's bookkeeping while
    // it has matrix instructions to issue.
    __builtin_amdgcn_s_setprio(1);
    static_for<NS>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      if constexpr (j < NPV) {
        constexpr int ts = j / DT, dt = j % DT;
        ot[dt] = mfma_32x32x16<BF16>(opq[j % PF], pb[SET ^ 1][ts >> 1][ts & 1], ot[dt]);
      } else {
        constexpr int s = (j - NPV) / NTL, t = (j - NPV) % NTL;
        st[SET ^ 1][t] = mfma_32x32x16<BF16>(opq[j % PF], qf[s], s == 0 ? zero16 : st[SET ^ 1][t]);
      }
      if constexpr (j + PF < NS) opq[j % PF] = operand(j + PF);
      static_for<LPS>([&](auto lc) {
        constexpr int n = (j / LSP) * LPS + decltype(lc)::value;
        if constexpr (!LONE && j % LSP == 0 && n < NL) issue_load(n, SET, k_row0, v_row0);
      });
      if constexpr (LONE) {  // K(it + 2) and V(it), once the operands have left the tiles
        constexpr int J0 = NS / 4, FOURS = NL / 4, PER = (FOURS + NS - J0 - 1) / (NS - J0);
        if constexpr (j == J0) tile_read();
        static_for<PER>([&](auto lc) {
          constexpr int n = (j - J0) * PER + decltype(lc)::value;
          if constexpr (n >= 0 && n < FOURS) {
            constexpr bool is_v = n < FOURS / 2;
            issue_four(is_v, n % (FOURS / 2), is_v ? v_row0 : k_row0, is_v ? lds_v0 : lds_k0);
          }
        });
      }
      constexpr int i_lo = j * NPR / NS, i_hi = (j + 1) * NPR / NS;
      static_for<i_hi - i_lo>([&](auto dc) { weights(set_c, IntC<i_lo + decltype(dc)::value>{}, rs0, rs1); });
      __builtin_amdgcn_sched_barrier(0);
    });
    __builtin_amdgcn_s_setprio(0);
    return rs0 + rs1;
  };

  // The tiles (and packed mask words) that were requested an iteration ago have landed, for
  // every wave that reads them.
  auto step_barrier = [&]() {
    wait_loads();
    if constexpr (!LONE) __syncthreads();
  };
  // ---- the walk -------------------------------------------------------------------------
  StepInfo cur = {0, kMasked, -1}, nxt = cur, nn = cur;
  if (nsteps > 0) {
    cur = step_info(0);
    nxt = step_info(1);
    nn = step_info(2);
    // Prologue: K(0) and K(1).
    if constexpr (LONE) {
#pragma unroll
      for (int i = 0; i < NCH / 4; ++i) issue_four(false, i, cur.row0, lds_k0);
#pragma unroll
      for (int i = 0; i < NCH / 4; ++i) issue_four(false, i, nxt.row0, lds_v0);
    } else {
#pragma unroll
      for (int i = 0; i < NCH; ++i) issue_load(NCH + i, 0, cur.row0, 0);
#pragma unroll
      for (int i = 0; i < NCH; ++i) issue_load(NCH + i, 1, nxt.row0, 0);
    }
    if (cur.mode == kPartial) {
      if (packed_tiles) {
        prefetch_mask_word(0, cur);
      } else {
        prefetch_mask_bytes(0, cur);
        wait_loads();
      }
    }
    wait_loads_but<NCH>();  // K(1) may be under way
    if constexpr (!LONE) __syncthreads();
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int t = 0; t < NTL; ++t)
        st[0][t] = mfma_32x32x16<BF16>(k_frag(sK, s, t), qf[s], s == 0 ? zero16 : st[0][t]);
    // (packed whether it leaves something out or not: its first use looks at the word.  Looked at first, one block's list of bytes
    // took a pass over LDS more: D=64 B=2 H=8 S=384 5.8 -> 5.6 us, S=1152 7.0 -> 6.7)
    if (cur.mode == kPartial && !packed_tiles) pack_own_bytes(lane);
  }

  auto iteration = [&](auto set_c, auto first_c, int it) {
    constexpr int SET = decltype(set_c)::value;
    step_barrier();
    u32x4_t opq[PF_ALL];
    body_prefetch(IntC<SET>{}, first_c, opq);
    // The common step -- every score allowed, no rescale owed, no PARTIAL tile ahead, no soft cap
    // -- goes from the barrier into the slots over one scalar condition and one branch.
    const bool next_partial = it + 1 < nsteps && nxt.mode == kPartial;
    const bool plain = (owed == 0) & !(p.softcap > 0.f) & unmasked(cur) & !next_partial;
    if (!plain) {
      if (cur.mode == kPartial && leaves_nothing_out()) cur.mode = kFull;
      if ((owed != 0) | (p.softcap > 0.f) | !unmasked(cur)) {
        if (owed & kOwesRescale) {
#pragma unroll
          for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r = 0; r < 16; ++r) ot[dt][r] *= alpha_pending;
          owed &= ~kOwesRescale;
        }
        if (p.softcap > 0.f) apply_softcap(IntC<SET>{});
        if (!unmasked(cur)) apply_mask(IntC<SET>{}, cur);
        if (owed & kOwesLook) look(set_c);
      }
      if (next_partial) {
        if (packed_tiles) {
          prefetch_mask_word(it + 1, nxt);
        } else {
          prefetch_mask_bytes(it + 1, nxt);
        }
      }
    }
    float sum = body(set_c, first_c, nn.row0, cur.row0, opq);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(sum <= kGrown)) != 0, 0)) {
      owed |= kOwesLook;
      if (__builtin_amdgcn_ballot_w64(!(sum <= kRedo)) != 0) redo(set_c, sum);
    }
    l_run += sum;
    if (__builtin_expect(next_partial && !packed_tiles, 0)) {
      wait_loads_but<NL>();  // (the tile loads of the iteration were requested behind the bytes)
      if (take_mask_bytes()) nxt.mode = kFull;
    }
    const StepInfo n3 = step_info(it + 3);
    cur = nxt;
    nxt = nn;
    nn = n3;
  };
  if (nsteps > 0) {
    iteration(IntC<0>{}, IntC<1>{}, 0);
    if (1 < nsteps) iteration(IntC<1>{}, IntC<0>{}, 1);
  }
  for (int it = 2; it < nsteps; it += 2) {
    iteration(IntC<0>{}, IntC<0>{}, it);
    if (it + 1 < nsteps) iteration(IntC<1>{}, IntC<0>{}, it + 1);
  }

  // Drain: O^T += V^T . P^T of the last step.
  if (nsteps > 0) {
    step_barrier();
    if (owed & kOwesRescale) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) ot[dt][r] *= alpha_pending;
    }
    auto drain = [&](auto set_c) {
      constexpr int SET = decltype(set_c)::value;
#pragma unroll
      for (int j = 0; j < NPV_ALL; ++j) {
        const int ts = j / DT, dt = j % DT;
        ot[dt] = mfma_32x32x16<BF16>(v_frag(LONE ? sV : sV + SET * TILE, j), pb[SET][ts >> 1][ts & 1], ot[dt]);
      }
    };
    // (A group without a step in the last round has weights of zero and whatever tile its loads were
    // pointed at: rows that the list may not hold, and zero times an infinity would reach the result.)
    if (KG == 1 || (nsteps - 1) * KG + kg < all_steps) {
      if ((nsteps - 1) & 1) {
        drain(IntC<1>{});
      } else {
        drain(IntC<0>{});
      }
    }
  }

  // Epilogue: O = O^T / l, zeros for rows without any allowed key or beyond seqlen.
  // A lane holds 4 consecutive d of its row per accumulator group; stored directly, one
  // store instruction would touch 32 rows with 16 bytes each.  So the wave transposes its
  // 32 x D output through LDS -- its own 32 rows of the K buffers, which nobody reads after
  // the barrier of the drain, 16-byte chunks swizzled like a K tile -- and stores whole
  // rows: 64 lanes x 16 bytes = 64 / CPR complete rows per instruction.
  float l_tot = pair_sum(l_run);
  if constexpr (KG > 1) {
    // Merge of the groups.  Row maxima and sums go where the mask bytes were (a wave
    // writes and has read its own rows only), the scaled O^T into the tiles once every group is
    // done with them; then each group adds up and stores its share of the columns.
    constexpr int UNITS = DT * 4;           // 4-register pieces of a lane's O^T
    constexpr int MINE = (UNITS + KG - 1) / KG;  // ... that a group stores
    static_assert(QT * D * 4 <= Shape::kTileBytes && QT * STEP >= QT * 8, "merge layout");
    auto group_at = [&](int i) { return lds_raw + size_t(i) * Shape::kGroupBytes; };
    constexpr size_t kStatM = Shape::kTileBytes, kStatL = kStatM + size_t(QT) * 4;
    const int row = 32 * w + c;
    if (g == 0) {
      reinterpret_cast<float*>(group_at(kg) + kStatM)[row] = m_run;
      reinterpret_cast<float*>(group_at(kg) + kStatL)[row] = l_tot;
    }
    __syncthreads();
    float m_all = -INFINITY;
#pragma unroll
    for (int i = 0; i < KG; ++i) m_all = fmaxf(m_all, reinterpret_cast<const float*>(group_at(i) + kStatM)[row]);
    const float m_fin = m_all == -INFINITY ? 0.f : m_all;
    l_tot = 0.f;
#pragma unroll
    for (int i = 0; i < KG; ++i)
      l_tot += reinterpret_cast<const float*>(group_at(i) + kStatL)[row] *
               __builtin_amdgcn_exp2f(reinterpret_cast<const float*>(group_at(i) + kStatM)[row] - m_fin);
    const bool live = (q_row < p.seqlen) && (l_tot > 0.f);
    const float mine = live ? __builtin_amdgcn_exp2f(m_run - m_fin) / l_tot : 0.f;
    typedef __attribute__((ext_vector_type(4))) float f32x4_t;
    auto piece_at = [&](int i, int u) {
      return reinterpret_cast<f32x4_t*>(group_at(i)) + (w * UNITS + u) * 64 + lane;
    };
    static_for<UNITS>([&](auto uc) {
      constexpr int u = decltype(uc)::value, dt = u / 4, r4 = u % 4;
      f32x4_t x;
      x[0] = ot[dt][4 * r4 + 0] * mine;
      x[1] = ot[dt][4 * r4 + 1] * mine;
      x[2] = ot[dt][4 * r4 + 2] * mine;
      x[3] = ot[dt][4 * r4 + 3] * mine;
      *piece_at(kg, u) = x;
    });
    __syncthreads();
#pragma unroll
    for (int n = 0; n < MINE; ++n) {
      const int u = kg * MINE + n;
      if (UNITS % KG != 0 && u >= UNITS) break;
      f32x4_t x = *piece_at(0, u);
#pragma unroll
      for (int i = 1; i < KG; ++i) x += *piece_at(i, u);
      const u32x2_t ov = {pack2<BF16>(x[0], x[1]), pack2<BF16>(x[2], x[3])};
      if (q_row < p.S) *reinterpret_cast<u32x2_t*>(p.o + slab + size_t(q_row) * D + 8 * u + 4 * g) = ov;
    }
    if (kg == 0 && g == 0 && q_row < p.S && p.lse != nullptr)
      p.lse[size_t(bh) * p.S + q_row] = live ? (m_fin + __builtin_amdgcn_logf(l_tot)) * 0.6931471805599453f : -INFINITY;
    return;
  }
  const bool live = (q_row < p.seqlen) && (l_tot > 0.f);
  const float inv = live ? 1.f / l_tot : 0.f;
  {
    uint16_t* stage = sK + size_t(w) * 32 * D;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        u32x2_t ov;
        ov[0] = pack2<BF16>(ot[dt][4 * r4 + 0] * inv, ot[dt][4 * r4 + 1] * inv);
        ov[1] = pack2<BF16>(ot[dt][4 * r4 + 2] * inv, ot[dt][4 * r4 + 3] * inv);
        const int ch = (4 * dt + r4) ^ k_swizzle<D>(c);
        *reinterpret_cast<u32x2_t*>(stage + c * D + ch * 8 + 4 * g) = ov;
      }
    }
    constexpr int ROWS_PER_STORE = 64 / CPR;
    const int srow = lane / CPR, pch = lane % CPR;
#pragma unroll
    for (int i = 0; i < 32 / ROWS_PER_STORE; ++i) {
      const int row = i * ROWS_PER_STORE + srow;  // row of the wave
      const u32x4_t val = *reinterpret_cast<const u32x4_t*>(stage + row * D + pch * 8);
      const int grow = q_wave_min + row;
      if (grow < p.S)
        *reinterpret_cast<u32x4_t*>(p.o + slab + size_t(grow) * D + (pch ^ k_swizzle<D>(row)) * 8) = val;
    }
  }
  if (q_row < p.S && p.lse != nullptr && g == 0) {
    const float lse = live ? (m_run + __builtin_amdgcn_logf(l_tot)) * 0.6931471805599453f : -INFINITY;
    p.lse[size_t(bh) * p.S + q_row] = lse;
  }
}

template <bool BF16, int D, int QB, int KB>
__global__ void __launch_bounds__(QB * 2, 2) fwd_kernel(const FwdParams p) {
  fwd_walk<FwdBlockShape<BF16, D, QB, KB>>(p);
}

// The steps of a list shared by the groups of a workgroup (fwd_choose_split says when).
template <bool BF16, int D, int QT, int KG, int STEP>
__global__ void __launch_bounds__(QT * 2 * KG, 2) fwd_ksplit(const FwdParams p) {
  fwd_walk<FwdShape<BF16, D, 0, 0, QT, KG, STEP>>(p);
}

// Host-side launch of one instance; returns the hipError_t of the launch itself (the
// thread's sticky "last error" of earlier, unrelated HIP calls is neither read nor cleared).
// The dynamic-LDS limit of an instance is raised once per device, not on every launch.
constexpr int kMaxDevices = 64;
template <class Shape, auto Kernel>
int launch_fwd_shape(const FwdParams& p, hipStream_t stream) {
  static std::atomic<bool> lds_limit_set[kMaxDevices];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return int(e);
  const bool cached = dev >= 0 && dev < kMaxDevices;
  if (!cached || !lds_limit_set[dev].load(std::memory_order_acquire)) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(Kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, int(Shape::kLdsBytes));
    if (e != hipSuccess) return int(e);
    if (cached) lds_limit_set[dev].store(true, std::memory_order_release);
  }
  const unsigned slabs_per_xcd = unsigned(p.n_slabs * p.parts + p.n_xcd - 1) / unsigned(p.n_xcd);
  const dim3 grid(unsigned(p.n_xcd) * slabs_per_xcd * (unsigned(p.tiles + p.parts - 1) / unsigned(p.parts)));
  FwdParams params = p;
  params.deal = plan_deal(p.n_slabs, p.parts, p.n_xcd, p.slab_group, p.tiles, p.H);
  void* args[] = {&params};
  return int(hipLaunchKernel(reinterpret_cast<const void*>(Kernel), grid, dim3(Shape::kThreads), args,
                             Shape::kLdsBytes, stream));
}

template <bool BF16, int D, int QB, int KB>
int launch_fwd(const FwdParams& p, hipStream_t stream) {
  return launch_fwd_shape<FwdBlockShape<BF16, D, QB, KB>, fwd_kernel<BF16, D, QB, KB>>(p, stream);
}
template <bool BF16, int D, int QT, int KG, int STEP>
int launch_fwd_ksplit(const FwdParams& p, hipStream_t stream) {
  return launch_fwd_shape<FwdShape<BF16, D, 0, 0, QT, KG, STEP>, fwd_ksplit<BF16, D, QT, KG, STEP>>(p, stream);
}

}  // namespace omni_attn
