// Backward of the block-sparse attention forward for gfx950 (MI355X, CDNA4).
//
// The reference has no backward (its operator is forward-only, omni-attn-mma/pybind/omni_attn.cc:70-77);
// what is differentiated here is exactly the function the forward kernel computes -- per
// query block the listed KV blocks with their FULL / CAUSAL / PARTIAL / MASKED semantics
// (omni-attn-mma/mma/attn_naive.cu:21-302), softmax scale 1/sqrt(D):
//
//   P_ij  = exp(q_i.k_j / sqrt(D) - LSE_i)   for allowed (i, j) of a listed block, else 0
//   delta_i = sum_d dO_id O_id
//   dV_j  = sum_i P_ij dO_i
//   dS_ij = P_ij (dO_i.v_j - delta_i)
//   dQ_i  = sum_j dS_ij k_j / sqrt(D)         dK_j = sum_i dS_ij q_i / sqrt(D)
//
// Two kernels, no atomics, bitwise reproducible:
//   bwd_dq_kernel    one workgroup per query block; walks that block's list like the forward;
//                    also writes -delta and the rows' score offsets (workspace, read by the
//                    second kernel).
//   bwd_dkdv_kernel  one workgroup per KV block; finds the (query block, slot) pairs that list
//                    it by scanning the slab's metadata (a bitmap of the matches is built in
//                    LDS -- in windows, where the metadata has more words than LDS holds --
//                    and visited in ascending order).  Each 32 keys have two waves
//                    with different work (weights and dV / dP, dS and dK), so two waves share
//                    a SIMD.
// Both use the forward's building blocks with the operands exchanged: every product is a
// v_mfma_f32_32x32x16 whose A operand comes from an LDS tile (row-wise or transposed read of
// the same tile) and whose B operand is in registers, and the accumulator of the first product
// of a step is the B operand of the second one, so P and dS never leave registers (the dK/dV
// kernel hands P from one wave to its partner through LDS).
// Tiles are loaded one step ahead (one barrier per step).  A step of 64 rows (or keys) is two
// 32-wide halves and runs as one sequence of slots like an iteration of the forward: one MFMA,
// the LDS fetch of an operand two or three slots ahead and a share of the vector work of the
// half whose first products have just finished, with a scheduling fence after every slot -- the
// exponentials of one half run under the products of the other inside one wave.  Offsets
// (-LSE sqrt(D), -delta) and masks (-inf) go into the accumulators the products start from, so a
// weight is one multiplication and one exp2 and an unmasked step carries no mask instruction.
// Masks of PARTIAL steps come with the step's tiles, straight into LDS, and a step whose tile leaves nothing out
// for the rows inside the sequence runs as an unmasked one: where the length is no multiple of the block, every block of
// the last list is PARTIAL.  (Requested by the step that uses them, a memory latency each, and always applied:
// forward and backward, us, before -> now, B=1 H=8 S=3000 D=128 images 230 -> 196, B=4 H=8 S=1157 D=64 85 -> 72,
// soft-capped 95 -> 86.)
// Workgroups are dealt to the XCDs by slab, so the workgroups that run together on an XCD share
// their operands through its L2.
#pragma once

#include "omni_attn_bwd_plan.hpp"
#include "omni_attn_fwd_kernel.hpp"
#include "omni_attn_softcap.hpp"

namespace omni_attn {

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

struct BwdParams {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const uint16_t* o;
  const uint16_t* dout;
  RowStrides q_at, k_at, v_at, dout_at;  // (o, dq, dk, dv are contiguous)
  const float* lse;  // [B,H,S] natural-log logsumexp written by the forward
  uint16_t* dq;
  uint16_t* dk;
  uint16_t* dv;
  // workspace [2][B,H,S], written by the dQ kernel and read by the dK/dV kernel: plane 0 is
  // -delta = -rowsum(dO . O); plane 1 the offset of the row's scores, -LSE * sqrt(D), -inf for a
  // row without any allowed key or beyond the sequence (every weight of such a row becomes 0) --
  // or, in the soft-capped instances, the exponent offset -LSE * log2(e), -inf for such a row
  float* ws;
  const int32_t* kv_num_blocks;
  const int32_t* kv_indices;
  const int32_t* types;
  const int32_t* partial_idx;  // null where no tiles are stored
  const uint8_t* partial_masks;
  const uint32_t* partial_bits;
  int num_partial;
  int S, Tq, Tk, max_blocks, seqlen, H, n_slabs;
  int QB, KB;     // block sizes
  int parts;      // parts a slab is dealt to the XCDs in
  FwdSplit dq_split;       // how the walks of the dQ kernel are split over waves
  int dq_step;             // keys per step of dQ where they are not (bwd_dq_step)
  DkdvSplit dkdv_split;    // ... and of the dK/dV kernel
  int win_words, table_steps;  // metadata words and steps that the dK/dV kernel holds in LDS (dkdv_plan)
  int slab_group;  // slabs of one XCD that are walked together (>= 1)
  int flat_first;  // (at most 64 slabs per XCD) slabs without short lists go first
  int n_xcd;      // XCDs (L2 domains) of the device; workgroup ids go round-robin over them
  DealPlan deal;
  float sl2;      // log2(e) / sqrt(D)
  float scale;    // 1 / sqrt(D)
  float softcap;  // > 0: the forward replaced x = s / sqrt(D) by softcap * tanh(x / softcap)
  float cap_c2;   // 2 * log2(e) / (sqrt(D) * softcap)
  float cap_l2;   // softcap * log2(e)
};

// sqrt(D) for the head dimensions of the instances.
template <int D>
struct SqrtOf {
  static constexpr float value = D == 128 ? 11.313708498984761f : (D == 64 ? 8.f : 5.656854249492381f);
};

// The kernel's arguments, read again where they are used: what only a rare path needs is not kept in scalar
// registers over the walk (there are none left: they would be spilled to vector lanes and read back in every step).
__device__ __forceinline__ const __attribute__((address_space(4))) BwdParams& params_again() {
  auto* at = (const __attribute__((address_space(4))) BwdParams*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(at));
  return *at;
}

// Pair of 16-bit values of registers r, r + 1, zero where the mask word (shifted by 4 g) forbids them.
template <int R>
__device__ __forceinline__ uint32_t keep_pair(uint32_t pair, uint32_t kw) {
  constexpr int bit = 8 * (R >> 2) + (R & 3);
  const uint32_t lo = uint32_t(__builtin_amdgcn_sbfe(int(kw), bit, 1)), hi = uint32_t(__builtin_amdgcn_sbfe(int(kw), bit + 1, 1));
  return pair & ((lo & 0xffffu) | (hi & 0xffff0000u));
}

// LDS reads at a byte address.  A fragment's address is (tile + lane part) ^ (k-step bits) + a
// constant: the swizzles of both tile layouts only touch the chunk bits inside a row, and they
// repeat every 16 rows, so rows and tiles are immediate offsets and a fragment costs one XOR.
__device__ __forceinline__ u32x4_t lds_b128_at(uint32_t addr) {
  return *(const __attribute__((address_space(3))) u32x4_t*)(addr);
}
__device__ __forceinline__ uint32_t lds_u32_at(uint32_t addr) {
  return *(const __attribute__((address_space(3))) uint32_t*)(addr);
}
__device__ __forceinline__ f32x4_t lds_f32x4_at(uint32_t addr) {
  return *(const __attribute__((address_space(3))) f32x4_t*)(addr);
}
__device__ __forceinline__ u32x4_t lds_tr_pair_at(uint32_t lo_addr, uint32_t hi_addr) {
  const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(lo_addr));
  const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(hi_addr));
  const u32x2_t lo2 = __builtin_bit_cast(u32x2_t, lo);
  const u32x2_t hi2 = __builtin_bit_cast(u32x2_t, hi);
  const u32x4_t a = {lo2[0], lo2[1], hi2[0], hi2[1]};
  return a;
}
// A transposed A fragment at (tile + lane part of its first half) ^ (column bits) + a constant:
// the second half lies 8 tile rows further, where every swizzle differs by chunk bit 1 (32 bytes).
template <int D>
__device__ __forceinline__ u32x4_t lds_tr_frag(uint32_t lo_lane, uint32_t col_bits, uint32_t off) {
  return lds_tr_pair_at((lo_lane ^ col_bits) + off, (lo_lane ^ (col_bits ^ 32u)) + off + 8u * D * 2u);
}

// One LDS layout serves both kinds of operand reads of a backward tile ([rows][D] 16-bit, the
// 16-byte chunk index of a row XORed with a function of the row, period 16 rows):
//   row-wise (ds_read_b128): 16 lanes read the same chunk of 16 consecutive rows -- the 16 XOR
//   values of 16 consecutive rows put them on 16 different 16-byte bank groups;
//   transposed (ds_read_b64_tr_b16): 32 lanes read 4 consecutive chunks of 4 consecutive rows
//   (starting at a multiple of 4) -- those 16 chunks land on 16 different bank groups too.
// So a tile is loaded once however it is read.
template <int D>
__device__ __forceinline__ int bwd_swizzle(int row) {
  if constexpr (D == 128) return ((row & 3) << 2) | ((row >> 2) & 3);
  if constexpr (D == 64) return (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
  return (row >> 2) & 3;
}
// Lane part (bytes) of a row-wise A fragment: row 32 t + c of the tile, k-step s at
// ((tile + lane part) ^ 32 s) + 32 t rows.
template <int D>
__device__ __forceinline__ uint32_t bwd_row_lane(int g, int c) {
  return uint32_t(c * D + (g ^ bwd_swizzle<D>(c)) * 8) * 2u;
}
// Lane part (bytes) of a transposed A fragment: rows 32 dt .. +31 of tile^T at tile rows
// 16 ts .. +15 (taken in the accumulator order of the first product) at
// ((tile + lane part) ^ 64 dt) + 16 ts rows; `upper` selects the second half, 8 rows further.
template <int D>
__device__ __forceinline__ uint32_t bwd_tr_lane(int g, int c, int upper) {
  const int i16 = c & 15, j16 = c >> 4, r = 4 * g + (i16 >> 2) + 8 * upper;
  const int chunk = 2 * j16 + ((i16 & 3) >> 1);
  return uint32_t(r * D * 2 + (chunk ^ bwd_swizzle<D>(r)) * 16 + (i16 & 1) * 8);
}

// [ROWS][D] tile from a slab into LDS in that layout.  Rows at or beyond the end of the slab
// read as zeros.
template <int D, int NT, int ROWS>
__device__ __forceinline__ void bwd_load_tile(i32x4_t rsrc, uint32_t pitch, int row0, uint32_t lds_tile, int tid,
                                              int w) {
  constexpr int CPR = D / 8;
  constexpr int TOTAL = ROWS * CPR;  // 16-byte chunks of the tile
  constexpr int NCH = TOTAL >= NT ? TOTAL / NT : 1;
  static_assert(TOTAL >= NT ? TOTAL % NT == 0 : TOTAL % 64 == 0, "tile must divide over the threads (or whole waves)");
  constexpr int ROW_STRIDE = NT / CPR;
  if (TOTAL < NT && tid >= TOTAL) return;  // a small tile is loaded by the first waves only
  const int ld_row = tid / CPR, ld_pch = tid % CPR;
  // The swizzle repeats every 16 rows and a thread's loads are ROW_STRIDE rows apart: one or two
  // per-lane offsets (four where a single wave loads) serve all of them, the rest of the address is wave-uniform.
  constexpr int PER = (NCH == 1 || ROW_STRIDE % 16 == 0) ? 1 : 16 / ROW_STRIDE;
  static_assert(NCH == 1 || (PER * ROW_STRIDE) % 16 == 0, "swizzle must repeat over a thread's loads");
  uint32_t lane_off[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int row = ld_row + i * ROW_STRIDE;
    lane_off[i] = uint32_t(ld_row) * pitch + uint32_t(ld_pch ^ bwd_swizzle<D>(row)) * 16u;
  }
#pragma unroll
  for (int i = 0; i < NCH; ++i)
    buffer_to_lds_b128(rsrc, lane_off[i % PER], uint32_t(row0 + i * ROW_STRIDE) * pitch,
                       lds_tile + uint32_t(w) * 1024u + uint32_t(i) * (NT * 16u));
}

// Effective mode of a slot, as the forward decides it.
__device__ __forceinline__ int32_t bwd_slot_mode(int32_t ty, int32_t pid, bool has_partial, int num_partial) {
  int32_t mode = (ty == kCausal || ty == kFull || ty == kPartial) ? ty : int32_t(kMasked);
  if (ty == kPartial && (!has_partial || pid < 0 || pid >= num_partial)) mode = kMasked;
  return mode;
}

// Transposed accumulators [D rows][32 columns] x factor -> 16-bit rows of the output, staged
// through LDS so that whole rows are stored (the forward's epilogue).
template <bool BF16, int D>
__device__ __forceinline__ void bwd_store_rows(const f32x16_t (&acc)[D / 32], float factor, uint16_t* stage,
                                               uint16_t* out_slab, int first_row, int n_rows_slab, int lane) {
  constexpr int CPR = D / 8, DT = D / 32;
  const int g = lane >> 5, c = lane & 31;
  static_for<DT * 4>([&](auto ic) {
    constexpr int dt = decltype(ic)::value / 4, r4 = decltype(ic)::value % 4;
    u32x2_t ov;
    ov[0] = pack2<BF16>(acc[dt][4 * r4 + 0] * factor, acc[dt][4 * r4 + 1] * factor);
    ov[1] = pack2<BF16>(acc[dt][4 * r4 + 2] * factor, acc[dt][4 * r4 + 3] * factor);
    const int ch = (4 * dt + r4) ^ k_swizzle<D>(c);
    *reinterpret_cast<u32x2_t*>(stage + c * D + ch * 8 + 4 * g) = ov;
  });
  constexpr int ROWS_PER_STORE = 64 / CPR;
  const int srow = lane / CPR, pch = lane % CPR;
#pragma unroll
  for (int i = 0; i < 32 / ROWS_PER_STORE; ++i) {
    const int row = i * ROWS_PER_STORE + srow;
    const u32x4_t val = *reinterpret_cast<const u32x4_t*>(stage + row * D + pch * 8);
    const int grow = first_row + row;
    if (grow < n_rows_slab)
      *reinterpret_cast<u32x4_t*>(out_slab + size_t(grow) * D + (pch ^ k_swizzle<D>(row)) * 8) = val;
  }
}


// Sum of the transposed accumulators of KG groups (W waves each, 32 columns = output rows per wave)
// x factor -> 16-bit rows.  Each group gets a share of the 4-register pieces from the others through LDS,
// adds up and stores it; `row`: this lane's output row, `stores`: it has one.  LDS: G (G - 1) W
// (pieces / G) KiB, nobody else may use it any more.
template <bool BF16, int D, int G, int W>
__device__ __forceinline__ void bwd_merge_store(const f32x16_t (&acc)[D / 32], float factor, uint8_t* lds, int group,
                                                int w, int lane, uint16_t* row, bool stores) {
  constexpr int UNITS = D / 8;                  // 4-register pieces of a lane's accumulators
  constexpr int SHARE = (UNITS + G - 1) / G;    // ... of a group
  const int g = lane >> 5;
  auto piece_at = [&](int to, int from, int n) {
    const int src = from < to ? from : from - 1;
    return reinterpret_cast<f32x4_t*>(lds) + (((to * (G - 1) + src) * W + w) * SHARE + n) * 64 + lane;
  };
  static_for<UNITS>([&](auto uc) {
    constexpr int u = decltype(uc)::value, dt = u / 4, r4 = u % 4, to = u / SHARE;
    if (to != group) {
      const f32x4_t x = {acc[dt][4 * r4 + 0], acc[dt][4 * r4 + 1], acc[dt][4 * r4 + 2], acc[dt][4 * r4 + 3]};
      *piece_at(to, group, u % SHARE) = x;
    }
  });
  __syncthreads();
  static_for<UNITS>([&](auto uc) {
    constexpr int u = decltype(uc)::value, dt = u / 4, r4 = u % 4, to = u / SHARE;
    if (to == group) {
      f32x4_t x = {acc[dt][4 * r4 + 0], acc[dt][4 * r4 + 1], acc[dt][4 * r4 + 2], acc[dt][4 * r4 + 3]};
      // in the order of the groups, whoever adds: group 0's piece first
      f32x4_t sum = group == 0 ? x : *piece_at(to, 0, u % SHARE);
#pragma unroll
      for (int i = 1; i < G; ++i) sum += i == to ? x : *piece_at(to, i, u % SHARE);
      const u32x2_t ov = {pack2<BF16>(sum[0] * factor, sum[1] * factor), pack2<BF16>(sum[2] * factor, sum[3] * factor)};
      if (stores) *reinterpret_cast<u32x2_t*>(row + 8 * u + 4 * g) = ov;
    }
  });
}

// One step of a backward walk.
struct BwdStepInfo {
  int row0;   // first key row (dQ kernel) / first query row (dK/dV kernel) of the step
  int mode;   // effective block mode
  int pid;    // partial tile
  int blk;    // dK/dV kernel: query block of the step
  int sub;    // index of the step inside its block
  bool valid;
};

// How a workgroup of the dQ kernel walks: QT query rows (QT / 32 waves), KG groups of such waves that
// share the steps of the list (step n is group n % KG's) and add up at the end, STEP keys per step: 64
// are two 32-key halves whose products and vector work overlap inside a wave.  QB, KB: the block
// sizes, 0 where they are not known at compile time.
template <bool BF16_, bool CAP_, int D_, int QB_, int KB_, int QT_, int KG_, int STEP_>
struct BwdDqShape {
  static constexpr bool BF16 = BF16_, CAP = CAP_;
  static constexpr int D = D_, QB = QB_, KB = KB_, QT = QT_, KG = KG_, kStep = STEP_;
  static constexpr int kGroupThreads = QT * 2;
  static constexpr int kThreads = kGroupThreads * KG;
  static constexpr int kTileElems = kStep * D;
  // two sets of two tiles (K, V), or the output staging; then one byte per row and key of a PARTIAL step
  static constexpr size_t kTileBytes = (4 * kTileElems > QT * D ? 4 * kTileElems : QT * D) * sizeof(uint16_t);
  static constexpr size_t kGroupBytes = kTileBytes + size_t(QT) * kStep;
  static constexpr size_t kMergeBytes = size_t(KG) * (KG - 1) * (QT / 32) * ((D / 8 + KG - 1) / KG) * 1024;
  static constexpr size_t kLdsBytes = kGroupBytes * KG > kMergeBytes ? kGroupBytes * KG : kMergeBytes;
};

template <class Shape>
__device__ __forceinline__ void bwd_dq_walk(const BwdParams& p) {
  constexpr bool BF16 = Shape::BF16, CAP = Shape::CAP;
  constexpr int D = Shape::D;
  constexpr int QT = Shape::QT;
  constexpr int KG = Shape::KG;
  constexpr bool LONE = QT == 32;  // a group is one wave: its steps need no barriers
  constexpr int NT = Shape::kGroupThreads;
  constexpr int STEP = Shape::kStep;
  const int QB = Shape::QB != 0 ? Shape::QB : p.QB;
  const int KB = Shape::KB != 0 ? Shape::KB : p.KB;
  const int SPB = KB / STEP;
  constexpr int NTL = STEP / 32;
  constexpr int KS = D / 16;
  constexpr int DT = D / 32;
  constexpr int TILE = Shape::kTileElems;
  constexpr int WQ = QT / 32;

  const int w_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = KG == 1 ? 0 : w_all / WQ;     // group of the wave (wave-uniform)
  const int w = KG == 1 ? w_all : w_all % WQ;  // wave of the group
  extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
  uint16_t* const lds16 = reinterpret_cast<uint16_t*>(lds_raw + size_t(kg) * Shape::kGroupBytes);  // [2 sets][K, V][TILE]

  // Workgroup -> (slab, query block): XCD x takes the slabs bh with bh % n_xcd == x in groups,
  // longest query blocks of a group first, so the workgroups that run together on an XCD walk the
  // K/V rows of a few slabs and share them through that XCD's L2.
  // (A slab may be dealt in parts, see the forward.)
  const int tiles = KG == 1 ? p.Tq : p.Tq * (QB / QT);
  const Dealt deal = deal_slab(p, p.slab_group, p.flat_first != 0);
  if (deal.slab < 0) return;
  const int bh = deal.slab >> p.deal.part_shift;
  const int qt = tiles - 1 - ((deal.rank << p.deal.part_shift) + deal.slab - (bh << p.deal.part_shift));
  const int q0 = qt * QT;  // first row of this workgroup
  if (qt < 0 || (KG > 1 && q0 >= p.S)) return;
  const int qb = KG == 1 ? qt : q0 >> (QB == 128 ? 7 : 6);
  static_assert((NT & (NT - 1)) == 0, "threads of a group");
  const int tid = threadIdx.x & (NT - 1);  // thread of the group
  const int lane = tid & 63;
  const int g = lane >> 5, c = lane & 31;

  const int q_row = q0 + 32 * w + c;
  const int q_wave_min = q0 + 32 * w;
  const int qr = q_row < p.S ? q_row : p.S - 1;
  const size_t meta_row = size_t(bh) * p.Tq + qb;
  const size_t meta_off = meta_row * p.max_blocks;
  const bool has_partial = p.partial_idx != nullptr;

  // Block metadata in registers, as in the forward: lane i holds block 64 * chunk + i of the list.
  int32_t mv_kvb = 0, mv_info = kMasked;  // info: effective mode in the low two bits, tile index above
  struct Raw {
    int32_t kvb, ty, pid;
  };
  auto request_chunk = [&](int chunk) {
    const int j = chunk * 64 + lane;
    const size_t o = meta_off + size_t(j < p.max_blocks ? j : 0);
    return Raw{p.kv_indices[o], p.types[o], has_partial ? p.partial_idx[o] : -1};
  };
  auto take_chunk = [&](const Raw& raw) {
    mv_kvb = raw.kvb < 0 ? 0 : (raw.kvb >= p.Tk ? p.Tk - 1 : raw.kvb);
    const int32_t mode = bwd_slot_mode(raw.ty, raw.pid, has_partial, p.num_partial);
    mv_info = (mode == kPartial ? raw.pid << 2 : 0) | mode;
  };
  auto load_chunk = [&](int chunk) { take_chunk(request_chunk(chunk)); };
  // The list is requested as soon as its address is known, and looked at when the rows are under way.  (With that,
  // and rows read through buffers instead of under a condition each: forward and backward, B=4 H=8 S=1157 D=64
  // soft-capped, 85.35 -> 84.55 us.)
  int nb = load_uniform(p.kv_num_blocks + meta_row);
  const Raw first_chunk = request_chunk(0);
  __builtin_amdgcn_sched_barrier(0);
  // Rows at or beyond the sequence are never used: the resources of K and V end there (those
  // rows arrive as zeros) and the query rows beyond it are replaced by zeros below, whatever the
  // caller left in the padding.
  const size_t slab = size_t(bh) * size_t(p.S) * D;  // of the contiguous ones
  const uint32_t k_pitch = p.k_at.row * 2u, v_pitch = p.v_at.row * 2u;  // bytes from row to row
  const i32x4_t rK = row_resource<D>(p.k, p.k_at, bh, p.H, p.deal.heads, p.seqlen);
  const i32x4_t rV = row_resource<D>(p.v, p.v_at, bh, p.H, p.deal.heads, p.seqlen);
  // Q and dO as B operands; delta = rowsum(dO . O) on the way.
  u32x4_t qf[KS], dof[KS];
  float dsum = 0.f;
  {
    const i32x4_t rQ = row_resource<D>(p.q, p.q_at, bh, p.H, p.deal.heads, p.seqlen);
    const i32x4_t rDo = row_resource<D>(p.dout, p.dout_at, bh, p.H, p.deal.heads, p.seqlen);
    const i32x4_t rO = make_buffer_resource(p.o + slab, uint32_t(p.seqlen) * (D * 2u));
    // (rows beyond the sequence: an offset beyond any buffer, so zeros)
    const bool row_in = q_row < p.seqlen;
    const uint32_t q_lane = row_in ? uint32_t(q_row) * (p.q_at.row * 2u) + 16u * uint32_t(g) : kNoRow<D>;
    const uint32_t do_lane = row_in ? uint32_t(q_row) * (p.dout_at.row * 2u) + 16u * uint32_t(g) : kNoRow<D>;
    const uint32_t o_lane = row_in ? uint32_t(q_row) * (D * 2u) + 16u * uint32_t(g) : kNoRow<D>;
    u32x4_t of[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      of[s] = buffer_load_b128(rO, o_lane, 32 * s);
      dof[s] = buffer_load_b128(rDo, do_lane, 32 * s);
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = buffer_load_b128(rQ, q_lane, 32 * s);
    take_chunk(first_chunk);
    nb = nb < 0 ? 0 : (nb > p.max_blocks ? p.max_blocks : nb);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        // (elements are copied to scalars first: a bit cast applied directly to a vector element
        // expression reads element 0)
        const uint32_t da = dof[s][e], ob = of[s][e];
        float a0, a1, b0, b1;
        if constexpr (BF16) {
          const uint32_t da_lo = da << 16, da_hi = da & 0xffff0000u, ob_lo = ob << 16, ob_hi = ob & 0xffff0000u;
          a0 = __builtin_bit_cast(float, da_lo);
          a1 = __builtin_bit_cast(float, da_hi);
          b0 = __builtin_bit_cast(float, ob_lo);
          b1 = __builtin_bit_cast(float, ob_hi);
        } else {
          const f16x2_t a = __builtin_bit_cast(f16x2_t, da);
          const f16x2_t b = __builtin_bit_cast(f16x2_t, ob);
          a0 = float(a[0]); a1 = float(a[1]); b0 = float(b[0]); b1 = float(b[1]);
        }
        dsum = __builtin_fmaf(a0, b0, dsum);
        dsum = __builtin_fmaf(a1, b1, dsum);
      }
    }
  }
  const float delta = pair_sum(dsum);  // the row lives in lanes c and c + 32
  const float lse = p.lse[size_t(bh) * p.S + qr];
  const bool row_live = q_row < p.seqlen && lse != -INFINITY;
  // What a row's exponents start from; -inf for rows without any allowed key so that every weight becomes 0.
  // The dK/dV kernel, too, starts the accumulator of a row's scores at -LSE * sqrt(D), so that the
  // exponent of a weight is the score times log2(e) / sqrt(D) and nothing else.  A soft-capped score is not
  // linear in the product: there it is the offset of the exponent itself.
  const float row_start = !row_live ? -INFINITY : (CAP ? lse * -1.4426950408889634f : -lse * SqrtOf<D>::value);
  if (q_row < p.S && g == 0 && kg == 0) {
    p.ws[size_t(bh) * p.S + q_row] = -delta;
    p.ws[size_t(p.n_slabs) * p.S + size_t(bh) * p.S + q_row] = row_start;
  }

  const f32x16_t zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  f32x16_t dq[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) dq[dt] = zero16;

  // The steps of the walk in order, skipping what contributes nothing: MASKED slots, keys at or
  // beyond the sequence, CAUSAL steps entirely above the diagonal of this query block.
  // Inside a KV block the next step is the previous one moved on by STEP keys (both reasons to
  // skip a step only get truer with the key index, so a block's steps are a prefix of it): that
  // path is a handful of scalar instructions; the slots of the list are only read at the first
  // step of a block.
  int gj = 0;  // next slot of the list to look at
  BwdStepInfo g_last = {0, kMasked, -1, 0, 0, false};
  const int q_last = q0 + QT - 1;
  auto next_step = [&]() {
    if (g_last.valid) {
      const int r = g_last.row0 + STEP, sb = g_last.sub + 1;
      const bool inside = bool(int(sb < SPB) & int(r < p.seqlen) & int(!(g_last.mode == kCausal && r > q_last)));
      if (inside) {
        g_last.row0 = r;
        g_last.sub = sb;
        return g_last;
      }
    }
    g_last.valid = false;
    while (gj < nb) {
      if ((gj & 63) == 0 && gj > 0) load_chunk(gj >> 6);
      const int ln = gj & 63;
      const int kvb = __builtin_amdgcn_readlane(mv_kvb, ln);
      const int info = __builtin_amdgcn_readlane(mv_info, ln);
      const int mode = info & 3, pid = info >> 2;
      ++gj;
      const int row0 = kvb * KB;
      if (mode == kMasked || row0 >= p.seqlen || (mode == kCausal && row0 > q_last)) continue;
      g_last.row0 = row0;
      g_last.mode = mode;
      g_last.pid = pid;
      g_last.sub = 0;
      g_last.valid = true;
      break;
    }
    return g_last;
  };
  const uint32_t lds_tiles = lds_offset_of(lds_raw) + uint32_t(kg) * uint32_t(Shape::kGroupBytes);
  auto issue_loads = [&](const BwdStepInfo& st, int set) {
    const uint32_t base = lds_tiles + uint32_t(set) * (2u * TILE * 2u);
    bwd_load_tile<D, NT, STEP>(rK, k_pitch, st.row0, base, tid, w);
    bwd_load_tile<D, NT, STEP>(rV, v_pitch, st.row0, base + TILE * 2u, tid, w);
  };
  const uint32_t row_lane = bwd_row_lane<D>(g, c);
  const uint32_t tr_lo = bwd_tr_lane<D>(g, c, 0);
  // One step, as one sequence of slots -- first the products S^T = K.Q^T and dP^T = V.dO^T of the
  // 32-key halves (lane = query row, registers = keys; the two products of a k-step alternate),
  // then the products dQ^T += K^T.dS^T of the halves -- each slot one MFMA, the LDS fetch of the
  // operand three slots ahead and a share of the vector work of the half whose first products
  // have just finished: dS^T = P^T (dP^T - delta), packed to 16 bits in the order the last
  // product reads it, is computed for half u under the first products of half u + 1 (or under the
  // last products of half 0).  The accumulator of S^T starts at the row's offset -LSE * sqrt(D) --
  // at -inf where the step's mask forbids the pair (`masked`, wave-uniform) -- so that a weight is
  // exp2(score * sl2); that of dP^T starts at -delta.  A soft-capped score is not linear in the
  // product: there S^T starts at zero, the offset goes into the exponents and the mask onto dS.
  constexpr int NSUB = NTL;
  static_assert(NSUB == 1 || NSUB == 2, "halves of a step");
  constexpr int NTR = 2 * DT;                    // last products of a half
  constexpr int NS = NSUB * (2 * KS + NTR);      // slots of a step
  constexpr int PF = D == 128 ? 2 : 3;           // operand fetch distance in slots (registers are tight at 128)
  const float neg_delta = -delta;
  auto compute = [&](int set, const uint32_t (&kw)[NTL], bool masked) {
    const uint32_t base = lds_tiles + uint32_t(set) * (2u * TILE * 2u);
    const uint32_t aK = base + row_lane, aV = aK + TILE * 2u, tK0 = base + tr_lo;
    f32x16_t st[NSUB], dp[NSUB];
    u32x4_t dsb[NSUB][2];
    auto operand = [&](auto nc) {
      constexpr int n = decltype(nc)::value;
      if constexpr (n < NSUB * 2 * KS) {
        constexpr int u = n / (2 * KS), s = (n % (2 * KS)) / 2, which = n % 2;
        return lds_b128_at(((which ? aV : aK) ^ uint32_t(32 * s)) + uint32_t(u) * (32u * D * 2u));
      } else {
        constexpr int m = n - NSUB * 2 * KS, u = m / NTR, ts = (m % NTR) / DT, dt = m % DT;
        constexpr uint32_t off = uint32_t(2 * u + ts) * (16u * D * 2u);
        return lds_tr_frag<D>(tK0, uint32_t(64 * dt), off);
      }
    };
    auto keep_bits = [&](auto uc, auto rc) {  // 0 or ~0 for register r of half u
      constexpr int u = decltype(uc)::value, r = decltype(rc)::value;
      return uint32_t(__builtin_amdgcn_sbfe(int(kw[u]), 8 * (r >> 2) + (r & 3), 1));
    };
    // the score gradients of registers r, r + 1 of half u
    auto grads = [&](auto uc, auto rc) {
      constexpr int u = decltype(uc)::value, r = decltype(rc)::value;
      float w0, w1;
      if constexpr (CAP) {
        const float d0 = capped_d(st[u][r], p.cap_c2), d1 = capped_d(st[u][r + 1], p.cap_c2), t0 = 1.f - d0, t1 = 1.f - d1;
        w0 = __builtin_amdgcn_exp2f(capped_exponent(t0, p.cap_l2, row_start)) * capped_slope(d0, t0);
        w1 = __builtin_amdgcn_exp2f(capped_exponent(t1, p.cap_l2, row_start)) * capped_slope(d1, t1);
      } else {
        w0 = __builtin_amdgcn_exp2f(st[u][r] * p.sl2);
        w1 = __builtin_amdgcn_exp2f(st[u][r + 1] * p.sl2);
      }
      dsb[u][r >> 3][(r & 7) >> 1] = pack2<BF16>(w0 * dp[u][r], w1 * dp[u][r + 1]);
    };
    u32x4_t opq[PF];
    static_for<PF>([&](auto nc) { opq[decltype(nc)::value] = operand(nc); });
    __builtin_amdgcn_s_setprio(1);  // products first: the other wave of the SIMD fills the gaps
    static_for<NS>([&](auto nc) {
      constexpr int n = decltype(nc)::value;
      constexpr bool first = n < NSUB * 2 * KS;
      constexpr int ch = first ? n / (2 * KS) : NSUB + (n - NSUB * 2 * KS) / NTR;  // chain of the slot
      constexpr int sl = first ? n % (2 * KS) : (n - NSUB * 2 * KS) % NTR;          // slot inside it
      constexpr int len = first ? 2 * KS : NTR;
      if constexpr (first) {
        constexpr int s = sl / 2;
        if constexpr (sl == 0) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            st[ch][r] = CAP ? 0.f : row_start;
            dp[ch][r] = neg_delta;
          }
          if constexpr (!CAP) {
            if (masked) {
              static_for<16>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                const uint32_t keep = keep_bits(IntC<ch>{}, rc);
                const uint32_t bits = __builtin_bit_cast(uint32_t, float(st[ch][r]));
                st[ch][r] = __builtin_bit_cast(float, (bits & keep) | (0xff800000u & ~keep));
              });
            }
          }
        }
        if constexpr (sl % 2 == 0) {
          st[ch] = mfma_32x32x16<BF16>(opq[n % PF], qf[s], st[ch]);
        } else {
          dp[ch] = mfma_32x32x16<BF16>(opq[n % PF], dof[s], dp[ch]);
        }
      } else {
        constexpr int u = ch - NSUB, ts = sl / DT, dt = sl % DT;
        if constexpr (CAP && sl == 0) {
          if (masked)
            static_for<8>([&](auto ic) {
              constexpr int i = decltype(ic)::value;
              const uint32_t pair = dsb[u][i >> 2][i & 3];
              dsb[u][i >> 2][i & 3] = keep_pair<2 * i>(pair, kw[u]);
            });
        }
        dq[dt] = mfma_32x32x16<BF16>(opq[n % PF], dsb[u][ts], dq[dt]);
      }
      if constexpr (n + PF < NS) opq[n % PF] = operand(IntC<n + PF>{});
      // the score gradients of half ch - 1 go beside the products of chain ch: 8 register pairs
      // spread over the chain's slots
      if constexpr (NSUB == 2 && ch >= 1 && ch <= NSUB) {
        constexpr int lo = sl * 8 / len, hi = (sl + 1) * 8 / len;
        static_for<hi - lo>([&](auto ic) { grads(IntC<ch - 1>{}, IntC<2 * (lo + decltype(ic)::value)>{}); });
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (NSUB == 1 && n == 2 * KS - 1) {  // a one-half step: nothing to put them under
        static_for<8>([&](auto ic) { grads(IntC<0>{}, IntC<2 * decltype(ic)::value>{}); });
        __builtin_amdgcn_sched_barrier(0);
      }
    });
    __builtin_amdgcn_s_setprio(0);
  };

  // Tiles of step i + 1 are loaded while step i is computed: one barrier per step.
  // A round is KG steps, one of each group (the last round of a walk may have fewer).
  bool more = false;  // the round that next_round() returned this group's step of has steps
  auto next_round = [&]() {
    BwdStepInfo mine = next_step();
    more = mine.valid;
    if constexpr (KG > 1) {
#pragma unroll
      for (int i = 1; i < KG; ++i) {
        const BwdStepInfo st = next_step();
        if (i == kg) mine = st;
      }
    }
    return mine;
  };
  // PARTIAL steps: the mask bytes of the wave's 32 rows, or the packed words, are requested with the tiles,
  // straight into LDS; a lane packs the 32 bytes of its row and of key half g and gets the other half's word
  // from the lane that has it.  (Writer and reader are the same wave.)
  const uint32_t lds_mask = lds_tiles + uint32_t(Shape::kTileBytes) + uint32_t(w) * (32u * STEP);
  const int row_in_block = q0 + 32 * w - qb * QB;  // first row of the wave in its query block
  auto request_mask = [&](const BwdStepInfo& st) {
    const auto& pp = params_again();
    int l = lane;  // (addresses are worked out here, not kept in registers over the walk)
    asm volatile("" : "+v"(l));
    if (pp.partial_bits != nullptr) {
      const uint32_t words = uint32_t(QB) * uint32_t(KB / 32);
      const i32x4_t rM = make_buffer_resource(pp.partial_bits + size_t(st.pid) * words, words * 4u);
      if (l < 32 * NTL)
        buffer_to_lds_b32(rM, (uint32_t(row_in_block + l % 32) * uint32_t(KB / 32) + uint32_t(l / 32)) * 4u,
                          uint32_t(st.sub * NTL) * 4u, lds_mask);
    } else {
      constexpr int MCPR = STEP / 16;  // 16-byte chunks per row
      const i32x4_t rM = make_buffer_resource(pp.partial_masks + size_t(st.pid) * size_t(QB * KB), uint32_t(QB * KB));
#pragma unroll
      for (int i = 0; i < MCPR / 2; ++i)
        buffer_to_lds_b128(rM, uint32_t(row_in_block + i * (64 / MCPR) + l / MCPR) * uint32_t(KB) + uint32_t(l % MCPR) * 16u,
                           uint32_t(st.sub * STEP), lds_mask + uint32_t(i) * 1024u);
    }
  };
  auto take_mask = [&](uint32_t (&kw)[NTL]) {
    const auto& pp = params_again();
    int l = lane;
    asm volatile("" : "+v"(l));
    uint32_t mine;  // word g (of two; the only one otherwise) of row c
    if (pp.partial_bits != nullptr) {
      mine = lds_u32_at(lds_mask + 4u * uint32_t(NTL == 2 ? l : l % 32));
    } else {
      const uint32_t at = lds_mask + uint32_t((l % 32) * STEP + (NTL == 2 ? (l & 32) : 0));
      mine = pack_mask_bytes(lds_b128_at(at), lds_b128_at(at + 16u));
    }
    if constexpr (NTL == 2) {
      float w0, w1;
      pair_split(__builtin_bit_cast(float, mine), w0, w1);
      kw[0] = __builtin_bit_cast(uint32_t, w0);
      kw[1] = __builtin_bit_cast(uint32_t, w1);
    } else {
      kw[0] = mine;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (read before the next request overwrites it)
  };
  BwdStepInfo cur = next_round();
  int set = 0;
  if (cur.valid) {
    issue_loads(cur, 0);
    if (cur.mode == kPartial) request_mask(cur);
  }
  while (more) {
    const BwdStepInfo nxt = next_round();
    wait_loads();  // the tiles (and mask) that this wave loaded have landed
    // Mask words of this lane's row: bit j of word t = key row0 + 32 t + j allowed.  `masked`: something is left
    // out for the rows of this wave (that a length which is no multiple of the block makes every block of the last
    // list PARTIAL, because of the rows beyond it, costs a look at the words).
    uint32_t kw[NTL];
    bool masked = false;
    if (__builtin_expect(!(cur.mode == kFull && cur.row0 + STEP <= p.seqlen), 0)) {
      if (cur.mode == kPartial) {
        take_mask(kw);
      } else {
#pragma unroll
        for (int t = 0; t < NTL; ++t) kw[t] = 0xffffffffu;
      }
      int limit = p.seqlen - 1;
      if (cur.mode == kCausal) limit = limit < q_row ? limit : q_row;
      uint32_t all = 0xffffffffu;
      static_for<NTL>([&](auto tc) {
        constexpr int t = decltype(tc)::value;
        const int n = limit - cur.row0 - 32 * t + 1;
        kw[t] &= n >= 32 ? 0xffffffffu : (n <= 0 ? 0u : ((1u << (n & 31)) - 1u));
        all &= kw[t];
        kw[t] >>= 4 * g;
      });
      masked = __builtin_amdgcn_ballot_w64(all != 0xffffffffu && q_row < p.seqlen) != 0;
    }
    if constexpr (!LONE) __syncthreads();  // ... for every wave; and the other set is no longer read
    if (nxt.valid) {
      issue_loads(nxt, set ^ 1);
      if (__builtin_expect(nxt.mode == kPartial, 0)) request_mask(nxt);
    }
    if (KG == 1 || cur.valid) compute(set, kw, masked);
    set ^= 1;
    cur = nxt;
  }
  __syncthreads();  // tiles are dead: the staging area overlaps them
  if constexpr (KG > 1) {
    bwd_merge_store<BF16, D, KG, WQ>(dq, p.scale, lds_raw, kg, w, lane,
                                     p.dq + slab + size_t(q_row < p.S ? q_row : 0) * D, q_row < p.S);
    return;
  }
  uint16_t* stage = lds16 + size_t(w) * 32 * D;
  // (the lane number goes through an empty asm: the addresses of the epilogue are then computed
  // here and not kept in registers across the walk, where every register counts)
  int lane_out = lane;
  asm volatile("" : "+v"(lane_out));
  bwd_store_rows<BF16, D>(dq, p.scale, stage, p.dq + slab, q_wave_min, p.S, lane_out);
}

// One workgroup per query block, all steps in one group.
template <bool BF16, bool CAP, int D, int QB, int KB>
__global__ void __launch_bounds__(QB * 2, 2) bwd_dq_kernel(const BwdParams p) {
  bwd_dq_walk<BwdDqShape<BF16, CAP, D, QB, KB, QB, 1, 64>>(p);
}
// With 32 keys per step: 64-row blocks at head_dim 128 in large launches (bwd_dq_step says why and where the line lies).  Both
// backward kernels, us, 64 -> 32 keys, causal B H=128 S=4096 bf16 2273 -> 2016, spans 2744 -> 2456, images 2613 -> 2325.  (The
// sums are formed in the same order: the same bits.)
template <bool BF16, bool CAP, int D, int QB, int KB>
__global__ void __launch_bounds__(QB * 2, 2) bwd_dq_short(const BwdParams p) {
  bwd_dq_walk<BwdDqShape<BF16, CAP, D, QB, KB, QB, 1, 32>>(p);
}
// The steps of a list shared by the groups of a workgroup (fwd_choose_split says when).
template <bool BF16, bool CAP, int D, int QT, int KG, int STEP>
__global__ void __launch_bounds__(QT * 2 * KG, 2) bwd_dq_ksplit(const BwdParams p) {
  bwd_dq_walk<BwdDqShape<BF16, CAP, D, 0, 0, QT, KG, STEP>>(p);
}

// First step of STEP query rows of a query block that can contribute to the keys from first_key on: a CAUSAL
// step whose rows all lie above the block's first key contributes nothing (the dK/dV kernel starts
// a block's walk there, and never stores score gradients for the steps before it).
template <int STEP>
__device__ __forceinline__ int bwd_first_step(int mode, int first_key, int first_row) {
  if (mode != kCausal) return 0;
  const int below = first_key - (first_row + STEP - 1);  // rows of the block before the first useful step
  return below > 0 ? (below + STEP - 1) / STEP : 0;
}

// How a workgroup of the dK/dV kernel works: NKG key groups of 32 keys (of one KV block) with two waves
// each, G groups of such waves that share the steps (step n is group n % G's) and add up at the end, STEP
// query rows per step.  QB, KB: the block sizes, 0 where they are not known at compile time.
template <bool BF16_, bool CAP_, int D_, int QB_, int KB_, int NKG_, int G_, int STEP_>
struct BwdDkdvShape {
  static constexpr bool BF16 = BF16_, CAP = CAP_;
  static constexpr int D = D_, QB = QB_, KB = KB_, G = G_;
  static constexpr int kKeyGroups = NKG_;          // 32 keys per wave
  static constexpr int kKeys = NKG_ * 32;          // keys of the workgroup
  static constexpr int kRoleThreads = kKeys * 2;   // one wave per key group in each of the two roles
  static constexpr int kGroupThreads = kKeys * 4;
  static constexpr int kThreads = kGroupThreads * G;
  static constexpr int kStep = STEP_;
  static constexpr int kSub = kStep / 32;
  static constexpr int kTileElems = kStep * D;
  // three sets of two tiles (Q, dO) -- the output staging overlaps them
  static constexpr size_t kTileBytes = size_t(6) * kTileElems * sizeof(uint16_t);
  // the weights one role hands to the other, 16-bit and in B-operand order:
  // [2 steps in flight][key group][32-row half][2][64 lanes] 16-byte words
  static constexpr size_t kHandBytes = size_t(2) * kKeyGroups * kSub * 2 * 64 * 16;
  // -delta and the exponent offsets of the rows of three steps
  static constexpr size_t kRowBytes = size_t(6) * kStep * sizeof(float);
  // one mask byte per row and key of a PARTIAL step
  static constexpr size_t kMaskBytes = size_t(kStep) * kKeys;
  static constexpr size_t kGroupBytes = kTileBytes + kHandBytes + kRowBytes + kMaskBytes;
  static constexpr size_t kFixedBytes = kGroupBytes * G;
  static_assert(size_t(G) * (G - 1) * 2 * kKeyGroups * ((D / 8 + G - 1) / G) * 1024 <= kFixedBytes, "merge in LDS");
  // workgroups that a compute unit's registers hold (waves per SIMD: 2 at head_dim 128, 4 at 64, 5 at 32)
  static constexpr int kWavesFit = (D == 128 ? 2 : (D == 64 ? 4 : 5)) * 256 / kThreads;
  static_assert(kWavesFit >= 1 && kFixedBytes + dkdv_word_bytes(64) + kDkdvTail + kDkdvMinTable * 8 <= kLdsOfComputeUnit,
                "a workgroup fits a compute unit");
};
// One workgroup per KV block, all steps in one group.  Query rows per step: at head_dim 128 with
// 128-key blocks 64, worked as two 32-row halves
// whose products and vector work overlap inside a wave (one workgroup of eight waves per
// compute unit, two waves per SIMD).  Elsewhere 32, so that two workgroups share a compute
// unit: a 64-key workgroup has four waves, and at head_dim <= 64 the products of a step are so
// short that four waves per SIMD hide more than longer steps gain (measured at head_dim 64:
// 64-row steps at two waves per SIMD take 1.3 x the time of 32-row steps at four).
template <bool BF16, bool CAP, int D, int QB, int KB>
using BwdDkdvBlockShape = BwdDkdvShape<BF16, CAP, D, QB, KB, KB / 32, 1, (KB == 128 && D == 128) ? 64 : 32>;

// Two 16-bit values of a word -> fp32 (exact).
template <bool BF16>
__device__ __forceinline__ void unpack2(uint32_t w, float& lo, float& hi) {
  if constexpr (BF16) {
    const uint32_t l = w << 16, h = w & 0xffff0000u;
    lo = __builtin_bit_cast(float, l);
    hi = __builtin_bit_cast(float, h);
  } else {
    const f16x2_t v = __builtin_bit_cast(f16x2_t, w);
    lo = float(v[0]);
    hi = float(v[1]);
  }
}

// One workgroup per KV block, two waves per 32 keys with different work, so that two waves
// share each SIMD and the vector work of one runs under the matrix work of the other:
//   the "weight" wave of a key group holds K, computes S = Q.K^T and P for a step, hands P
//   (times the soft-cap derivative factor, when capped) to its partner through LDS -- rounded to
//   16 bits, in the order the partner's product reads it -- and accumulates dV^T += dO^T.P;
//   the "gradient" wave holds V, computes dP - delta = dO.V^T - delta, and one step later
//   dS = P (dP - delta) and dK^T += Q^T.dS.
// The gradient waves run one step behind the weight waves, so one barrier per step orders
// the hand-over, the tile loads (the weight waves load Q, the gradient waves dO, one step ahead)
// and the reuse of the three tile sets.
// A step is kStep query rows.  Its products form one sequence of slots -- first products of the
// 32-row halves, then second products of the halves -- each slot one MFMA, the LDS fetch of
// the operand three slots ahead and a share of the vector work of the half whose first
// product has just finished, with a scheduling fence after each slot: the weights of half u are
// computed under the products of half u + 1 (or under the second products of half 0).
template <class Traits>
__device__ __forceinline__ void bwd_dkdv_walk(const BwdParams& p) {
  constexpr bool BF16 = Traits::BF16, CAP = Traits::CAP;
  constexpr int D = Traits::D;
  constexpr int G = Traits::G;
  constexpr int KT = Traits::kKeys;
  const int QB = Traits::QB != 0 ? Traits::QB : p.QB;
  const int KB = Traits::KB != 0 ? Traits::KB : p.KB;
  constexpr int NKG = Traits::kKeyGroups;
  constexpr int RT = Traits::kRoleThreads;
  constexpr int NW = Traits::kThreads / 64;  // waves of the workgroup
  constexpr int STEP = Traits::kStep;
  constexpr int NSUB = Traits::kSub;
  const int NSTEPS = QB / STEP;      // steps per query block
  constexpr int KS = D / 16;         // products of a 32-row half: KS for S (or dP) ...
  constexpr int DT = D / 32;
  constexpr int NTR = 2 * DT;        // ... and as many for dV^T (or dK^T)
  constexpr int NS = 2 * NSUB * KS;  // slots of a step
  constexpr int SPC = 16 / KS;       // scores of a half whose vector work goes beside one product
  constexpr int TILE = Traits::kTileElems;
  constexpr int PF = 3 < NS ? 3 : NS;  // operand fetch distance in slots
  constexpr bool PRIO = KT == 64 || G > 1;  // raise the wave priority around the products (it pays
                                       // with two workgroups per compute unit)
  static_assert(NTR == KS && 16 % KS == 0, "slot layout");

  extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
  const int w_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int group = G == 1 ? 0 : w_all / (2 * NKG);     // group of the wave (wave-uniform)
  const int w = G == 1 ? w_all : w_all % (2 * NKG);     // wave of the group
  uint8_t* const lds_group = lds_raw + size_t(group) * Traits::kGroupBytes;
  uint16_t* const lds16 = reinterpret_cast<uint16_t*>(lds_group);  // [3 sets][Q, dO][TILE]
  // (byte addresses in LDS are integers: a pointer that goes through the generic address space is checked for null)
  const uint32_t lds_tiles = lds_offset_of(lds_raw) + uint32_t(group) * uint32_t(Traits::kGroupBytes);
  const uint32_t lds_hand = lds_tiles + uint32_t(Traits::kTileBytes);
  const uint32_t lds_nd = lds_hand + uint32_t(Traits::kHandBytes);  // [3 sets][STEP] -delta
  const uint32_t lds_l2 = lds_nd + 3u * STEP * 4u;                  // [3 sets][STEP] exponent offsets
  const uint32_t lds_masks = lds_nd + uint32_t(Traits::kRowBytes);  // [key groups][STEP][32]
  uint64_t* const sMatch = reinterpret_cast<uint64_t*>(lds_raw + Traits::kFixedBytes);

  // Workgroup -> (slab, KV block): XCD x takes the slabs bh with bh % n_xcd == x in groups, first KV
  // blocks (the longest walks of a causal mask) first, so the workgroups that run together on an XCD
  // read the Q and dO rows of a few slabs and share them through that XCD's L2.
  const int tiles = G == 1 ? p.Tk : p.Tk * (KB / KT);
  const Dealt deal = deal_slab(p, p.slab_group, p.flat_first != 0);
  if (deal.slab < 0) return;
  const int bh = deal.slab >> p.deal.part_shift;
  const int kt = (deal.rank << p.deal.part_shift) + deal.slab - (bh << p.deal.part_shift);
  const int key0 = kt * KT;  // first key of this workgroup
  if (kt >= tiles || (G > 1 && key0 >= p.S)) return;
  const int kvb = G == 1 ? kt : key0 >> (KB == 128 ? 7 : 6);
  const int tid = G == 1 ? threadIdx.x : threadIdx.x - group * Traits::kGroupThreads;  // thread of the group
  const int lane = tid & 63;
  const bool grad_role = w >= NKG;        // wave-uniform
  const int kg = grad_role ? w - NKG : w;  // key group of the wave
  const int rtid = tid - (grad_role ? RT : 0);
  const int g = lane >> 5, c = lane & 31;

  // Rows at or beyond the sequence are never read: the resources of Q and dO end there, so
  // those rows arrive as zeros whatever the caller left in them.
  const size_t slab = size_t(bh) * size_t(p.S) * D;
  const uint32_t q_pitch = p.q_at.row * 2u, do_pitch = p.dout_at.row * 2u;  // bytes from row to row
  const i32x4_t rQ = row_resource<D>(p.q, p.q_at, bh, p.H, p.deal.heads, p.seqlen);
  const i32x4_t rD = row_resource<D>(p.dout, p.dout_at, bh, p.H, p.deal.heads, p.seqlen);
  const i32x4_t rNd = make_buffer_resource(p.ws + size_t(bh) * p.S, uint32_t(p.S) * 4u);
  const i32x4_t rL2 = make_buffer_resource(p.ws + size_t(p.n_slabs) * p.S + size_t(bh) * p.S, uint32_t(p.S) * 4u);
  const int key_wave_min = key0 + 32 * kg;
  const int kcol = key_wave_min - kvb * KB;  // ... inside its block
  const int key = key_wave_min + c;  // this lane's key row inside the slab
  const bool key_live = key < p.seqlen;
  const size_t meta_slab = size_t(bh) * p.Tq;
  const int chunks = (p.max_blocks + 63) / 64;  // 64-slot words per query block
  const int n_words = p.Tq * chunks;
  const int win_words = p.win_words;  // words of the bitmap held in LDS at a time
  int32_t* const sFirst = reinterpret_cast<int32_t*>(sMatch + win_words);
  typedef __attribute__((ext_vector_type(2))) int32_t i32x2_t;
  // one entry per step: first query row; mode in the low two bits, tile index above
  i32x2_t* const sSteps = reinterpret_cast<i32x2_t*>(sFirst + ((win_words + 1) & ~1));
  const int table_steps = p.table_steps;

  // This lane's key as B operand: K for a weight wave, V for a gradient wave (zeros for a key
  // beyond the sequence).
  u32x4_t bop[KS];
  {
    const RowStrides& at = grad_role ? p.v_at : p.k_at;
    const i32x4_t rB = row_resource<D>(grad_role ? p.v : p.k, at, bh, p.H, p.deal.heads, p.seqlen);
    const uint32_t lane_off = key_live ? uint32_t(key) * (at.row * 2u) + 16u * uint32_t(g) : kNoRow<D>;
#pragma unroll
    for (int s = 0; s < KS; ++s) bop[s] = buffer_load_b128(rB, lane_off, 32 * s);
  }

  // The scan: which (query block, slot) pairs list this KV block (after the forward's clamping of
  // the block index) with a type the forward would visit?  One 64-bit word per query block and 64
  // slots.  Mode and tile index of a word's first match are
  // kept beside it (a list names a block once, except for duplicates and clamped indices).  The
  // words [base, end) of the slab go to entries 0 .. end - base of the window; every wave of the
  // workgroup calls this at the same point (the barriers are the workgroup's).
  auto scan_window = [&](auto scan_c, const auto& pp, int base, int end) {
    __syncthreads();  // nobody reads the previous window any more
    const bool has_partial = pp.partial_idx != nullptr;
    // A wave takes SCAN consecutive words per pass and has the loads of all of them in flight
    // together (every slot inside the list's width is loaded; kv_num_blocks cuts afterwards).
    // The first window, scanned while few registers are live, takes four; later ones one.
    constexpr int SCAN = decltype(scan_c)::value;
    for (int word0 = base + w_all * SCAN; word0 < end; word0 += NW * SCAN) {
      int32_t raw[SCAN], ty[SCAN], pid[SCAN], nbv[SCAN];
#pragma unroll
      for (int u = 0; u < SCAN; ++u) {
        const int word = word0 + u < end ? word0 + u : end - 1;  // (a repeat of the last word: ignored below)
        const int qb = word / chunks, ch = word - qb * chunks;
        const int slot = ch * 64 + lane;
        const size_t o = (meta_slab + qb) * pp.max_blocks + (slot < pp.max_blocks ? slot : pp.max_blocks - 1);
        raw[u] = pp.kv_indices[o];
        ty[u] = pp.types[o];
        pid[u] = has_partial ? pp.partial_idx[o] : -1;
        nbv[u] = pp.kv_num_blocks[meta_slab + qb];
      }
#pragma unroll
      for (int u = 0; u < SCAN; ++u) {
        const int word = word0 + u;
        if (word >= end) break;
        const int ch = word % chunks;
        const int nb = nbv[u] < 0 ? 0 : (nbv[u] > pp.max_blocks ? pp.max_blocks : nbv[u]);
        const int32_t idx = raw[u] < 0 ? 0 : (raw[u] >= pp.Tk ? pp.Tk - 1 : raw[u]);
        const int32_t mode = bwd_slot_mode(ty[u], pid[u], has_partial, pp.num_partial);
        const bool hit = ch * 64 + lane < nb && idx == kvb && mode != kMasked;
        const int32_t info = (mode == kPartial ? pid[u] << 2 : 0) | mode;
        const uint64_t bits = __builtin_amdgcn_ballot_w64(hit);
        if (lane == 0) sMatch[word - base] = bits;
        if (bits != 0 && lane == __builtin_ctzll(bits)) sFirst[word - base] = info;
      }
    }
    __syncthreads();
  };

  const f32x16_t zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  f32x16_t acc[DT];  // dV^T of a weight wave, dK^T of a gradient wave
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = zero16;

  // The walk: the matches in ascending (query block, slot) order, each as NSTEPS steps of STEP query
  // rows, skipping steps beyond the sequence and CAUSAL steps entirely above the diagonal (both cut a
  // match's steps from one end).  The first wave turns the window's bitmap into a table of steps, a
  // lane per word, so that the loop gets a step with one LDS read, requested an iteration ahead
  // (a generator that found the next step from the bitmap cost every wave 500 - 700 cycles per
  // step).  A table holds table_steps of them, a piece of the window's walk.  Returns their number;
  // behind the table stay the word that the next piece begins with (or `end`), the number of the window's
  // steps before that word, and that of the next piece's first step.
  int32_t* const s_table = reinterpret_cast<int32_t*>(sSteps + table_steps);  // steps, word, before, next
  auto steps_of = [&](int32_t info, int first_row, int& sub0) {
    sub0 = bwd_first_step<STEP>(info & 3, key0, first_row);
    const int rows = p.seqlen - first_row;
    const int subs = rows <= 0 ? 0 : (rows + STEP - 1) / STEP;
    const int n = (subs < NSTEPS ? subs : NSTEPS) - sub0;
    return n > 0 ? n : 0;
  };
  auto build_table = [&](const auto& pp, int base, int end, bool first_piece) {
    if (w_all == 0) {
      const bool has_partial = pp.partial_idx != nullptr;
      int w0 = base, n = 0, first = 0;
      if (!first_piece) {
        w0 = s_table[1];
        n = s_table[2];
        first = s_table[3];
      }
      for (; w0 < end; w0 += 64) {
        const int word = w0 + lane;
        uint64_t bits = word < end ? sMatch[word - base] : 0;
        const int qb = word / chunks, ch = word - qb * chunks;
        const int first_row = qb * QB;
        // information of the match that is the lowest bit of `left`
        auto info_of = [&](uint64_t left) {
          if (left == bits) return sFirst[word - base];
          const size_t o = (meta_slab + qb) * pp.max_blocks + ch * 64 + __builtin_ctzll(left);
          const int32_t pid = has_partial ? pp.partial_idx[o] : -1;
          const int32_t mode = bwd_slot_mode(pp.types[o], pid, has_partial, pp.num_partial);
          return (mode == kPartial ? pid << 2 : 0) | mode;
        };
        int count = 0, sub0;
        for (uint64_t left = bits; left != 0; left &= left - 1) count += steps_of(info_of(left), first_row, sub0);
        int upto = count;  // inclusive sum over the lanes
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
          const int other = __shfl_up(upto, d, 64);
          upto += lane >= d ? other : 0;
        }
        int at = n + upto - count - first;  // entry of this lane's first step
        for (uint64_t left = bits; left != 0 && at < table_steps; left &= left - 1) {
          const int32_t info = info_of(left);
          const int k = steps_of(info, first_row, sub0);
          for (int i = 0; i < k; ++i, ++at)
            if (at >= 0 && at < table_steps) sSteps[at] = i32x2_t{first_row + (sub0 + i) * STEP, info};
        }
        const int all = __builtin_amdgcn_readfirstlane(__shfl(upto, 63, 64));
        if (n + all - first > table_steps) break;  // (these words have steps of the next piece)
        n += all;
      }
      if (lane == 0) {
        s_table[0] = w0 < end ? table_steps : n - first;
        s_table[1] = w0 < end ? w0 : end;
        s_table[2] = n;
        s_table[3] = first + table_steps;
      }
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(s_table[0]);
  };
  int win_base = 0, win_end = win_words < n_words ? win_words : n_words;  // the words of the slab the window holds
  scan_window(IntC<4>{}, p, 0, win_end);
  int n_steps = build_table(p, 0, win_end, true);
  const uint32_t hand_lane = lds_hand + uint32_t(kg) * (NSUB * 2048u) + uint32_t(lane) * 16u;
  auto tile_at = [&](int set, int which) { return lds_tiles + uint32_t(set * 2 + which) * (TILE * 2u); };
  // the four words of half `half` of 32-row half u of the step with parity par
  auto hand_at = [&](int par, int u, int half) {
    return hand_lane + uint32_t(par) * (NKG * NSUB * 2048u) + uint32_t(u) * 2048u + uint32_t(half) * 1024u;
  };
  struct Step {
    int row0, info;
    bool valid;
  };
  // The rows of step j + 1 are loaded during iteration j: Q and the exponent offsets by the
  // weight waves, dO and -delta by the gradient waves.
  auto load_q = [&](const Step& st, int set) {
    bwd_load_tile<D, RT, STEP>(rQ, q_pitch, st.row0, tile_at(set, 0), rtid, kg);
    if (rtid < STEP)
      buffer_to_lds_b32(rL2, uint32_t(rtid) * 4u, uint32_t(st.row0) * 4u, lds_l2 + uint32_t(set * STEP) * 4u);
  };
  auto load_do = [&](const Step& st, int set) {
    bwd_load_tile<D, RT, STEP>(rD, do_pitch, st.row0, tile_at(set, 1), rtid, kg);
    if (rtid < STEP)
      buffer_to_lds_b32(rNd, uint32_t(rtid) * 4u, uint32_t(st.row0) * 4u, lds_nd + uint32_t(set * STEP) * 4u);
  };
  const uint32_t row_lane = bwd_row_lane<D>(g, c);
  const uint32_t tr_lo = bwd_tr_lane<D>(g, c, 0);

  // Operand n of a step's slot sequence, from the tile read row-wise (first products: rows
  // 32 u + lane of the tile at k-step s) or transposed (second products: columns 32 dt .. +31
  // at rows 32 u + 16 ts .. +15).
  auto operand = [&](auto nc, uint32_t a_rows, uint32_t a_tr0) {
    constexpr int n = decltype(nc)::value;
    constexpr int ch = n / KS, s = n % KS;
    if constexpr (ch < NSUB) {
      return lds_b128_at((a_rows ^ uint32_t(32 * s)) + uint32_t(ch) * (32u * D * 2u));
    } else {
      constexpr int u = ch - NSUB, ts = s / DT, dt = s % DT;
      constexpr uint32_t off = uint32_t(2 * u + ts) * (16u * D * 2u);
      return lds_tr_frag<D>(a_tr0, uint32_t(64 * dt), off);
    }
  };

  // Weight wave, one step: S = Q.K^T (lane = key, registers = query rows), P, dV^T += dO^T.P.
  // The accumulator of a half's scores starts at the rows' offsets -LSE * sqrt(D) -- at -inf where
  // the step's mask (`masked`, wave-uniform: the words kw are only looked at then) forbids the
  // pair -- so a weight is exp2(score * sl2) and the mask costs nothing inside the slots.  A
  // soft-capped score is not linear in the product: there the accumulator starts at zero, the
  // offsets are fetched when the weights are computed and the mask is applied to the weights.
  auto weight_step = [&](int set, int par, const uint32_t (&kw)[NSUB], bool masked) {
    const uint32_t aQ = tile_at(set, 0) + row_lane, tD0 = tile_at(set, 1) + tr_lo;
    // The row offsets of the workspace: registers 4 i .. +3 of a half are its query rows
    // 8 i + 4 g .. +3.
    auto row_offsets = [&](int u, int i4) {
      return lds_f32x4_at(lds_l2 + uint32_t(set * STEP + 32 * u + 8 * i4) * 4u + 16u * g);
    };
    // 0 or ~0: may register r of half u keep its value?  (kw is already shifted by 4 g: bit
    // 8 (r / 4) + r % 4 is the row of register r)
    auto keep_bits = [&](auto uc, auto rc) {
      constexpr int u = decltype(uc)::value, r = decltype(rc)::value;
      return uint32_t(__builtin_amdgcn_sbfe(int(kw[u]), 8 * (r >> 2) + (r & 3), 1));
    };
    f32x16_t sc[NSUB];
    u32x4_t pb[NSUB][2];   // P packed to 16 bits, B-operand order
    u32x4_t hb[NSUB][2];   // what the partner gets when capped: P times the soft-cap factor
    f32x4_t lq = {0.f, 0.f, 0.f, 0.f};
    auto weights = [&](auto uc, auto ic) {
      constexpr int u = decltype(uc)::value, i = decltype(ic)::value;
      static_for<SPC / 2>([&](auto jc) {
        constexpr int r = SPC * i + 2 * decltype(jc)::value;
        float w0, w1;
        if constexpr (CAP) {
          if constexpr ((r & 3) == 0) lq = row_offsets(u, r >> 2);
          const float d0 = capped_d(sc[u][r], p.cap_c2), d1 = capped_d(sc[u][r + 1], p.cap_c2), t0 = 1.f - d0, t1 = 1.f - d1;
          w0 = __builtin_amdgcn_exp2f(capped_exponent(t0, p.cap_l2, lq[r & 3]));
          w1 = __builtin_amdgcn_exp2f(capped_exponent(t1, p.cap_l2, lq[(r + 1) & 3]));
          hb[u][r >> 3][(r & 7) >> 1] = pack2<BF16>(w0 * capped_slope(d0, t0), w1 * capped_slope(d1, t1));
        } else {  // the scores already carry their row's offset and the mask
          w0 = __builtin_amdgcn_exp2f(sc[u][r] * p.sl2);
          w1 = __builtin_amdgcn_exp2f(sc[u][r + 1] * p.sl2);
        }
        pb[u][r >> 3][(r & 7) >> 1] = pack2<BF16>(w0, w1);
      });
      if constexpr (((i + 1) * SPC) % 8 == 0) {  // four words are complete: to the partner
        constexpr int half = (i + 1) * SPC / 8 - 1;
        if constexpr (CAP) {
          if (masked)
            static_for<4>([&](auto jc) {
              constexpr int j = decltype(jc)::value;
              const uint32_t a = pb[u][half][j], b = hb[u][half][j];
              pb[u][half][j] = keep_pair<8 * half + 2 * j>(a, kw[u]);
              hb[u][half][j] = keep_pair<8 * half + 2 * j>(b, kw[u]);
            });
          *(__attribute__((address_space(3))) u32x4_t*)(hand_at(par, u, half)) = hb[u][half];
        } else {
          *(__attribute__((address_space(3))) u32x4_t*)(hand_at(par, u, half)) = pb[u][half];
        }
      }
    };
    u32x4_t opq[PF];
    static_for<PF>([&](auto nc) { opq[decltype(nc)::value] = operand(nc, aQ, tD0); });
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(1);
    static_for<NS>([&](auto nc) {
      constexpr int n = decltype(nc)::value;
      constexpr int ch = n / KS, s = n % KS;
      if constexpr (ch < NSUB) {
        if constexpr (s == 0) {
          if constexpr (CAP) {
            sc[ch] = zero16;
          } else {
            static_for<4>([&](auto ic) {
              constexpr int i4 = decltype(ic)::value;
              const f32x4_t o4 = row_offsets(ch, i4);
              sc[ch][4 * i4 + 0] = o4[0];
              sc[ch][4 * i4 + 1] = o4[1];
              sc[ch][4 * i4 + 2] = o4[2];
              sc[ch][4 * i4 + 3] = o4[3];
            });
            if (masked) {
              static_for<16>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                const uint32_t keep = keep_bits(IntC<ch>{}, rc);
                const uint32_t bits = __builtin_bit_cast(uint32_t, float(sc[ch][r]));
                sc[ch][r] = __builtin_bit_cast(float, (bits & keep) | (0xff800000u & ~keep));
              });
            }
          }
        }
        sc[ch] = mfma_32x32x16<BF16>(opq[n % PF], bop[s], sc[ch]);
      } else {
        constexpr int u = ch - NSUB, ts = s / DT, dt = s % DT;
        acc[dt] = mfma_32x32x16<BF16>(opq[n % PF], pb[u][ts], acc[dt]);
      }
      if constexpr (n + PF < NS) opq[n % PF] = operand(IntC<n + PF>{}, aQ, tD0);
      // the weights of half ch - 1 go beside the products of chain ch
      if constexpr (NSUB > 1 && ch >= 1 && ch <= NSUB) weights(IntC<ch - 1>{}, IntC<s>{});
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (NSUB == 1 && n == KS - 1) {  // a one-half step: nothing to put them under
        if constexpr (PRIO) __builtin_amdgcn_s_setprio(0);
        static_for<KS>([&](auto ic) { weights(IntC<0>{}, ic); });
        if constexpr (PRIO) __builtin_amdgcn_s_setprio(1);
        __builtin_amdgcn_sched_barrier(0);
      }
    });
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(0);
  };
  // Gradient wave, one step: dP - delta = dO.V^T - delta (the accumulator starts at -delta),
  // dS = P (dP - delta) with the partner's P, dK^T += Q^T.dS.
  auto grad_step = [&](int set, int par) {
    const uint32_t aD = tile_at(set, 1) + row_lane, tQ0 = tile_at(set, 0) + tr_lo;
    f32x16_t dp[NSUB];
    u32x4_t hand[NSUB][2], dsb[NSUB][2];
    static_for<4 * NSUB>([&](auto ic) {
      constexpr int u = decltype(ic)::value / 4, i4 = decltype(ic)::value % 4;
      const f32x4_t nd = lds_f32x4_at(lds_nd + uint32_t(set * STEP + 32 * u + 8 * i4) * 4u + 16u * g);
      dp[u][4 * i4 + 0] = nd[0];
      dp[u][4 * i4 + 1] = nd[1];
      dp[u][4 * i4 + 2] = nd[2];
      dp[u][4 * i4 + 3] = nd[3];
    });
    auto score_grads = [&](auto uc, auto ic) {
      constexpr int u = decltype(uc)::value, i = decltype(ic)::value;
      static_for<SPC / 2>([&](auto jc) {
        constexpr int r = SPC * i + 2 * decltype(jc)::value;
        float h0, h1;
        unpack2<BF16>(hand[u][r >> 3][(r & 7) >> 1], h0, h1);
        dsb[u][r >> 3][(r & 7) >> 1] = pack2<BF16>(h0 * dp[u][r], h1 * dp[u][r + 1]);
      });
    };
    u32x4_t opq[PF];
    static_for<PF>([&](auto nc) { opq[decltype(nc)::value] = operand(nc, aD, tQ0); });
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(1);
    static_for<NS>([&](auto nc) {
      constexpr int n = decltype(nc)::value;
      constexpr int ch = n / KS, s = n % KS;
      if constexpr (ch < NSUB) {
        if constexpr (s == 0) {
          hand[ch][0] = lds_b128_at(hand_at(par, ch, 0));
          hand[ch][1] = lds_b128_at(hand_at(par, ch, 1));
        }
        dp[ch] = mfma_32x32x16<BF16>(opq[n % PF], bop[s], dp[ch]);
      } else {
        constexpr int u = ch - NSUB, ts = s / DT, dt = s % DT;
        acc[dt] = mfma_32x32x16<BF16>(opq[n % PF], dsb[u][ts], acc[dt]);
      }
      if constexpr (n + PF < NS) opq[n % PF] = operand(IntC<n + PF>{}, aD, tQ0);
      if constexpr (NSUB > 1 && ch >= 1 && ch <= NSUB) score_grads(IntC<ch - 1>{}, IntC<s>{});
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (NSUB == 1 && n == KS - 1) {
        if constexpr (PRIO) __builtin_amdgcn_s_setprio(0);
        static_for<KS>([&](auto ic) { score_grads(IntC<0>{}, ic); });
        if constexpr (PRIO) __builtin_amdgcn_s_setprio(1);
        __builtin_amdgcn_sched_barrier(0);
      }
    });
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(0);
  };

  // PARTIAL steps: the mask of a weight wave's 32 keys, as bytes or packed words, is requested with its rows,
  // straight into LDS (writer and reader are the same wave).
  const uint32_t lds_mask = lds_masks + uint32_t(kg) * (STEP * 32u);
  auto request_mask = [&](const Step& st) {
    const auto& pp = params_again();
    int l = lane;  // (addresses are worked out here, not kept in registers over the walk)
    asm volatile("" : "+v"(l));
    const uint32_t first = uint32_t(st.row0 & (QB - 1));  // row of the tile
    if (pp.partial_bits != nullptr) {
      const uint32_t words = uint32_t(QB) * uint32_t(KB / 32);
      const i32x4_t rM = make_buffer_resource(pp.partial_bits + size_t(st.info >> 2) * words, words * 4u);
      if (l < STEP)
        buffer_to_lds_b32(rM, uint32_t(l) * uint32_t(KB / 8), (first * uint32_t(KB / 32) + uint32_t(kcol / 32)) * 4u,
                          lds_mask);
    } else {
      const i32x4_t rM = make_buffer_resource(pp.partial_masks + size_t(st.info >> 2) * size_t(QB * KB), uint32_t(QB * KB));
#pragma unroll
      for (int u = 0; u < NSUB; ++u)
        buffer_to_lds_b128(rM, uint32_t(l / 2) * uint32_t(KB) + uint32_t(l % 2) * 16u,
                           (first + 32 * u) * uint32_t(KB) + uint32_t(kcol), lds_mask + uint32_t(u) * 1024u);
    }
  };
  // Bits of half u for this lane's key: bit j = its row j attends the key.  Collected from the 32 rows, unless
  // none of those inside the sequence leaves a key out (with a length that is no multiple of the block, all blocks
  // of the last list are PARTIAL because of the rows beyond it).
  auto mask_column = [&](int u, int row0) {
    const auto& pp = params_again();
    int l = lane & 31;
    asm volatile("" : "+v"(l));
    uint32_t roww;
    if (pp.partial_bits != nullptr) {
      roww = lds_u32_at(lds_mask + uint32_t(32 * u + l) * 4u);
    } else {
      const uint32_t at = lds_mask + uint32_t(32 * u + l) * 32u;
      roww = pack_mask_bytes(lds_b128_at(at), lds_b128_at(at + 16u));
    }
    if (__builtin_amdgcn_ballot_w64(roww != 0xffffffffu && row0 + 32 * u + l < p.seqlen) == 0) return 0xffffffffu;
    uint32_t col = 0;
    static_for<32>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      const uint32_t r = uint32_t(__builtin_amdgcn_readlane(int(roww), j));
      col |= ((r >> c) & 1u) << j;
    });
    return col;
  };

  // Iteration j: the weight waves do step j, the gradient waves step j - 1.  The two roles
  // run separate copies of the loop (same trip count, one barrier per trip), so that each keeps
  // its accumulators in place.  Metadata of more words than the bitmap holds takes several
  // windows: the steps of a window are worked off completely before the next one is scanned.
  auto run = [&](auto role_c) {
    constexpr bool GRAD = decltype(role_c)::value;
    // A round is G steps, one of each group.  A window's last round may have fewer: the next
    // window's first one goes on with the group whose turn it is.
    int turn = 0;
    for (;;) {
      const int rounds = (n_steps + turn + G - 1) / G;
      auto index_of = [&](int j) { return j * G + group - turn; };  // of this group's step of round j
      auto request = [&](int j) {
        const int t = index_of(j);
        return sSteps[t < 0 || t >= n_steps ? 0 : t];
      };
      auto receive = [&](i32x2_t e, int j) {
        const int t = index_of(j);
        const int e0 = e[0], e1 = e[1];
        return Step{__builtin_amdgcn_readfirstlane(e0), __builtin_amdgcn_readfirstlane(e1), t >= 0 && t < n_steps};
      };
      Step prev = {0, kMasked, false}, cur = receive(request(0), 0);
      i32x2_t coming = request(1);
      int s_prev = 2, s_cur = 0, s_nxt = 1;  // tile sets of steps j - 1, j, j + 1
      if (cur.valid) {
        if constexpr (!GRAD) {
          load_q(cur, 0);
          if ((cur.info & 3) == kPartial) request_mask(cur);
        } else {
          load_do(cur, 0);
        }
      }
      const int iterations = rounds > 0 ? rounds + 1 : 0;
      for (int j = 0; j < iterations; ++j) {
        const Step nxt = receive(coming, j + 1);
        coming = request(j + 2);
        wait_loads();  // the tile (and mask) this wave loaded has landed
        // mask words of this lane's key: bit i of word u = query row row0 + 32 u + i attends it
        uint32_t kw[NSUB];
        bool masked = false;  // (wave-uniform) something is left out
        if constexpr (!GRAD) {
          const int mode = cur.info & 3;
          if (__builtin_expect(cur.valid && !(mode == kFull && key_wave_min + 32 <= p.seqlen), 0)) {
            uint32_t all = 0xffffffffu;
#pragma unroll
            for (int u = 0; u < NSUB; ++u) {
              uint32_t m = key_live ? 0xffffffffu : 0u;
              if (mode == kCausal) {  // rows at or after the key
                const int n = key - (cur.row0 + 32 * u);
                m &= n <= 0 ? 0xffffffffu : (n >= 32 ? 0u : (0xffffffffu << (n & 31)));
              }
              if (mode == kPartial) m &= mask_column(u, cur.row0);
              all &= m;
              kw[u] = m >> (4 * g);
            }
            masked = __builtin_amdgcn_ballot_w64(all != 0xffffffffu) != 0;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (read before the next request overwrites it)
          }
        }
        __syncthreads();  // ... everybody's have; the hand-over of step j - 1 is written; the set
                          // about to be overwritten (step j - 2) is no longer read
        if constexpr (!GRAD) {
          if (nxt.valid) {
            load_q(nxt, s_nxt);
            if (__builtin_expect((nxt.info & 3) == kPartial, 0)) request_mask(nxt);
          }
          if (cur.valid) weight_step(s_cur, j & 1, kw, masked);
        } else {
          if (nxt.valid) load_do(nxt, s_nxt);
          if (prev.valid) grad_step(s_prev, (j + 1) & 1);
        }
        prev = cur;
        cur = nxt;
        const int t3 = s_prev;
        s_prev = s_cur;
        s_cur = s_nxt;
        s_nxt = t3;
      }
      const bool window_done = __builtin_amdgcn_readfirstlane(s_table[1]) >= win_end;
      if (__builtin_expect(window_done && win_end >= n_words, 1)) break;
      // more steps, or more words of metadata, than LDS holds: the next piece of the window, or the next window
      turn = (turn + n_steps) % G;
      if (window_done) {
        win_base = win_end;
        win_end = win_base + win_words < n_words ? win_base + win_words : n_words;
        scan_window(IntC<1>{}, params_again(), win_base, win_end);
      } else {
        __syncthreads();  // nobody reads the table any more
      }
      n_steps = build_table(params_again(), win_base, win_end, window_done);
    }
    __syncthreads();
    if constexpr (G > 1) {
      const size_t row = slab + size_t(key < p.S ? key : 0) * D;
      bwd_merge_store<BF16, D, G, 2 * NKG>(acc, GRAD ? p.scale : 1.f, lds_raw, group, w, lane,
                                           (GRAD ? p.dk : p.dv) + row, key < p.S);
      return;
    }
    uint16_t* stage = lds16 + size_t(w) * 32 * D;
    if constexpr (!GRAD) {
      bwd_store_rows<BF16, D>(acc, 1.f, stage, p.dv + slab, key_wave_min, p.S, lane);
    } else {
      bwd_store_rows<BF16, D>(acc, p.scale, stage, p.dk + slab, key_wave_min, p.S, lane);
    }
  };
  if (grad_role) {
    run(std::integral_constant<bool, true>{});
  } else {
    run(std::integral_constant<bool, false>{});
  }
}

template <bool BF16, bool CAP, int D, int QB, int KB>
__global__ void __launch_bounds__(KB * 4, D == 128 ? 2 : 4) bwd_dkdv_kernel(const BwdParams p) {
  bwd_dkdv_walk<BwdDkdvBlockShape<BF16, CAP, D, QB, KB>>(p);
}
// The query rows of a KV block shared by the groups of a workgroup.
template <bool BF16, bool CAP, int D, int NKG, int G>
__global__ void __launch_bounds__(NKG * 128 * G, D == 128 ? 2 : 4) bwd_dkdv_split(const BwdParams p) {
  bwd_dkdv_walk<BwdDkdvShape<BF16, CAP, D, 0, 0, NKG, G, 32>>(p);
}

// Launch of one backward kernel; its dynamic-LDS limit is raised once per device.
template <auto Kernel>
int launch_bwd_kernel(const BwdParams& p, int tiles, int threads, size_t lds, size_t max_lds, hipStream_t stream) {
  static std::atomic<bool> lds_limit_set[kMaxDevices];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return int(e);
  const bool cached = dev >= 0 && dev < kMaxDevices;
  if (!cached || !lds_limit_set[dev].load(std::memory_order_acquire)) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                            int(max_lds));
    if (e != hipSuccess) return int(e);
    if (cached) lds_limit_set[dev].store(true, std::memory_order_release);
  }
  const unsigned slabs_per_xcd = unsigned(p.n_slabs * p.parts + p.n_xcd - 1) / unsigned(p.n_xcd);
  const dim3 grid(unsigned(p.n_xcd) * slabs_per_xcd * (unsigned(tiles + p.parts - 1) / unsigned(p.parts)));
  BwdParams params = p;
  params.deal = plan_deal(p.n_slabs, p.parts, p.n_xcd, p.slab_group, tiles, p.H);
  void* args[] = {&params};
  return int(hipLaunchKernel(reinterpret_cast<const void*>(Kernel), grid, dim3(threads), args, lds, stream));
}

template <bool BF16, bool CAP, int D, int QB, int KB>
int launch_dq(const BwdParams& p, hipStream_t stream) {
  if constexpr (QB == 64 && D == 128) {
    if (p.dq_step == 32) {
      using Shape = BwdDqShape<BF16, CAP, D, QB, KB, QB, 1, 32>;
      return launch_bwd_kernel<bwd_dq_short<BF16, CAP, D, QB, KB>>(p, p.Tq, Shape::kThreads, Shape::kLdsBytes,
                                                                   Shape::kLdsBytes, stream);
    }
  }
  using Shape = BwdDqShape<BF16, CAP, D, QB, KB, QB, 1, 64>;
  return launch_bwd_kernel<bwd_dq_kernel<BF16, CAP, D, QB, KB>>(p, p.Tq, Shape::kThreads, Shape::kLdsBytes,
                                                                Shape::kLdsBytes, stream);
}
template <bool BF16, bool CAP, int D, int QT, int KG, int STEP>
int launch_dq_ksplit(const BwdParams& p, hipStream_t stream) {
  using Shape = BwdDqShape<BF16, CAP, D, 0, 0, QT, KG, STEP>;
  return launch_bwd_kernel<bwd_dq_ksplit<BF16, CAP, D, QT, KG, STEP>>(p, p.Tq * (p.QB / QT), Shape::kThreads,
                                                                      Shape::kLdsBytes, Shape::kLdsBytes, stream);
}

template <class Shape, auto Kernel>
int launch_dkdv_shape(const BwdParams& p, int tiles, hipStream_t stream) {
  const long long n_words = (long long)p.Tq * ((p.max_blocks + 63) / 64);
  const DkdvPlan plan = dkdv_plan(Shape::kFixedBytes, Shape::kWavesFit, n_words, p.QB / Shape::kStep);
  BwdParams with = p;
  with.win_words = plan.words;
  with.table_steps = plan.steps;
  return launch_bwd_kernel<Kernel>(with, tiles, Shape::kThreads, plan.bytes, kLdsOfComputeUnit, stream);
}
template <bool BF16, bool CAP, int D, int QB, int KB>
int launch_dkdv(const BwdParams& p, hipStream_t stream) {
  return launch_dkdv_shape<BwdDkdvBlockShape<BF16, CAP, D, QB, KB>, bwd_dkdv_kernel<BF16, CAP, D, QB, KB>>(p, p.Tk,
                                                                                                          stream);
}
template <bool BF16, bool CAP, int D, int NKG, int G>
int launch_dkdv_split(const BwdParams& p, hipStream_t stream) {
  return launch_dkdv_shape<BwdDkdvShape<BF16, CAP, D, 0, 0, NKG, G, 32>, bwd_dkdv_split<BF16, CAP, D, NKG, G>>(
      p, p.Tk * (p.KB / (32 * NKG)), stream);
}

template <bool BF16, bool CAP, int D, int QB, int KB>
int launch_bwd_cap(const BwdParams& p, hipStream_t stream) {
  int e;
  switch (p.dq_split) {
    case FwdSplit::kRows32x4: e = launch_dq_ksplit<BF16, CAP, D, 32, 4, 32>(p, stream); break;
    case FwdSplit::kRows64x2: e = launch_dq_ksplit<BF16, CAP, D, 64, 2, 64>(p, stream); break;
    default: e = launch_dq<BF16, CAP, D, QB, KB>(p, stream); break;
  }
  if (e != 0) return e;
  if constexpr (D != 128) {
    if (p.dkdv_split == DkdvSplit::kKeys32x4) return launch_dkdv_split<BF16, CAP, D, 1, 4>(p, stream);
  }
  if (p.dkdv_split == DkdvSplit::kKeys64x2) return launch_dkdv_split<BF16, CAP, D, 2, 2>(p, stream);
  return launch_dkdv<BF16, CAP, D, QB, KB>(p, stream);
}

// The soft-capped instances are separate kernels: the extra arithmetic per score would
// otherwise cost the plain ones registers.
template <bool BF16, int D, int QB, int KB>
int launch_bwd(const BwdParams& p, hipStream_t stream) {
  return p.softcap > 0.f ? launch_bwd_cap<BF16, true, D, QB, KB>(p, stream)
                         : launch_bwd_cap<BF16, false, D, QB, KB>(p, stream);
}

}  // namespace omni_attn
