// The forward for shapes the tuned kernel has no instance for.
//
// The reference's correctness kernel omni_attn_simple_kernel_impl
// (omni-attn-mma/mma/attn_naive.cu:21-302, launcher :305-408) takes any Q_BLOCK / KV_BLOCK and
// any head_dim up to 256 (`float out[256]`, :189-190); its MMA kernels take only
// {64, 128}^2 x {32, 64, 128}.  This kernel keeps that generality and the slot rules, on the matrix
// cores, at the precision of a scalar kernel: products of 16-bit operands summed in fp32, and
// weights that enter the second product with (at least) 22 significant bits.
//
// One workgroup owns up to 32 query rows of one query block; its four waves share the keys of the
// block's list: the listed keys are one sequence of positions, slot * KB + offset; step n is the
// positions 32 n .. 32 n + 31 (of one block or of several, for any KB) and wave w takes the steps
// w, w + 4, ...  A wave has its own running maximum, sum and O^T accumulators; they are merged
// through LDS at the end.  No workgroup barrier until then.
//
// S^T = K.Q^T and O^T = V^T.P^T with v_mfma_f32_32x32x16 as in the tuned forward: a lane owns a query
// row.  K fragments come straight from global memory into registers (a step's rows are used by one
// wave only, so LDS would share nothing), V goes through a wave-private LDS tile for its transposed
// read.  A weight is a sum of 16-bit parts with one product each: two for fp16 (scaled by 2^14
// first, so that small weights stay out of the subnormals), three for bf16.
//
// Bound by the latency of a step (loads, two matrix chains, the softmax and the split of the weights
// on the vector pipe) times a quarter of the steps of the longest list.  B=1 H=8 S=2048 D=96 fp16,
// causal in 32x32 blocks: 33 us; one wave per row with vector arithmetic and two passes took 1938 us.
#include "../../include/omni_attn_gfx950.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <cmath>
#include <utility>

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
constexpr int kWaves = 4;

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
  int adv_slot, adv_off;  // 32 kWaves positions = adv_slot blocks of kb_eff keys + adv_off keys
  int q_tiles;        // 32-row tiles per query block
  int o_vec;          // rows of o start on 8-byte boundaries and D is a multiple of 8
  int mask_words;     // four keys of a tile row may be read as one 32-bit word
  unsigned n_slabs;   // B * H
  float scale, sl2, softcap;
};

// Columns are worked in chunks of 8, chunk i at columns 8 i .. 8 i + 7.  Where D is not a multiple of
// 8 the last chunk holds the columns D - 8 .. D - 1 instead, and so do the chunks beyond it: every
// read is 16 bytes inside its row (at any alignment), Q is zero where a chunk repeats a column, and
// the repeated columns of the result are not stored.
__device__ __forceinline__ int chunk_start(int d0, int D) { return d0 + 8 <= D ? d0 : D - 8; }

// The chunk of `row` at column d0.  SMALL: head dimensions below 8, zeros behind the row.
template <bool SMALL>
__device__ __forceinline__ u32x4_t load8(const uint16_t* row, int d0, int D) {
  u32x4_t r;
  if constexpr (SMALL) {
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

// One 16-bit part of a pair of values; the values become what is left of them (exact).
template <bool BF16>
__device__ __forceinline__ uint32_t split_part(float& lo, float& hi) {
  if constexpr (BF16) {
    const __bf16 a = (__bf16)lo, b = (__bf16)hi;
    lo -= float(a);
    hi -= float(b);
    const bf16x2_t v = {a, b};
    return __builtin_bit_cast(uint32_t, v);
  } else {
    const _Float16 a = (_Float16)lo, b = (_Float16)hi;
    lo -= float(a);
    hi -= float(b);
    const f16x2_t v = {a, b};
    return __builtin_bit_cast(uint32_t, v);
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

// The other half-wave's value (lane ^ 32).
__device__ __forceinline__ float other_half(float x) { return __shfl_xor(x, 32, 64); }

// DT: 32-column tiles of the head dimension.
template <int DT>
struct GenericTraits {
  static constexpr int kRowBytes = 64 * (DT | 1);  // an odd multiple of 64: four consecutive rows
                                                   // of a transposed read lie on different banks
  static constexpr int kVBytes = 32 * kRowBytes;
  static constexpr int kGroup = DT < kWaves ? DT : kWaves;  // output tiles merged per pass
  static constexpr size_t kMergeBytes = size_t(kWaves) * kGroup * 4096;
  static constexpr size_t kTiles = size_t(kWaves) * kVBytes > kMergeBytes ? size_t(kWaves) * kVBytes : kMergeBytes;
  // From 128 columns on Q lives in LDS (shared by the waves) instead of in registers, of which the
  // rows of the next step and the accumulators leave too few.
  static constexpr bool kQInLds = DT >= 4;
  static constexpr size_t kQBytes = kQInLds ? size_t(kVBytes) : 0;
  // behind the tiles: Q; per wave, compare key, offset inside the block and tile of 32 keys; and
  // the maximum and sum of 32 rows
  static constexpr size_t kLdsBytes = kTiles + kQBytes + kWaves * (32 * 12 + 32 * 8);
};

template <bool BF16, int DT, bool SMALL>
__global__ void __launch_bounds__(64 * kWaves, DT <= 4 ? 2 : 1) fwd_generic_kernel(const GenericParams p) {
  using Traits = GenericTraits<DT>;
  constexpr int KS = 2 * DT;
  constexpr int RS = Traits::kRowBytes;
  constexpr int PARTS = BF16 ? 3 : 2;
  constexpr float kShift = BF16 ? 0.f : 14.f;  // log2 of the factor on the weights
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

  const unsigned wg = blockIdx.x;
  const unsigned rank = wg / p.n_slabs;
  const size_t bh = wg - rank * p.n_slabs;
  const unsigned tile = unsigned(p.Tq) * unsigned(p.q_tiles) - 1 - rank;  // longest lists of a causal mask first
  const int qb = int(tile / unsigned(p.q_tiles));
  const int row0 = int(tile - unsigned(qb) * unsigned(p.q_tiles)) * 32;  // first row inside the block
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 5, c = lane & 31;
  const int q_local = row0 + c;
  const int q_idx = qb * p.QB + q_local;
  const bool q_here = q_local < p.QB && q_idx < p.S;  // a row of this tile
  const bool q_live = q_here && q_idx < p.seqlen;

  uint8_t* const sV = lds + size_t(w) * Traits::kVBytes;
  uint8_t* const sQ = lds + Traits::kTiles;
  int32_t* const sKey = reinterpret_cast<int32_t*>(lds + Traits::kTiles + Traits::kQBytes) + w * 96;
  int32_t* const sOff = sKey + 32;
  int32_t* const sPid = sKey + 64;
  float* const sStat = reinterpret_cast<float*>(lds + Traits::kTiles + Traits::kQBytes + kWaves * 384);  // [2][kWaves][32]

  const int64_t b = int64_t(bh) / p.H, h = int64_t(bh) - b * p.H;
  const uint16_t* const q_slab = p.q + b * p.q_at.batch + h * p.q_at.head;
  const uint16_t* const k_slab = p.k + b * p.k_at.batch + h * p.k_at.head;
  const uint16_t* const v_slab = p.v + b * p.v_at.batch + h * p.v_at.head;
  const size_t mrow = bh * p.Tq + qb;
  const size_t moff = mrow * p.max_blocks;
  int nb = p.kv_num_blocks[mrow];
  nb = nb < 0 ? 0 : (nb > p.max_blocks ? p.max_blocks : nb);
  if (qb * p.QB + row0 >= p.seqlen) nb = 0;  // only padding rows: zeros (attn_naive.cu:64-72)
  const bool has_partial = p.partial_idx != nullptr && p.partial_masks != nullptr;

  // chunk (16 bytes) `ch` of row r of a tile: XORed with bits 2 and 3 of the row
  auto tile_at = [](int r, int ch) { return r * RS + ((ch ^ ((r >> 2) & 3)) * 16); };
  // Q as B operand: lane holds Q[row][16 s + 8 g .. +7]
  u32x4_t qf[Traits::kQInLds ? 1 : KS];
  {
    const uint16_t* qrow = q_slab + int64_t(q_live ? q_idx : 0) * p.q_at.row;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (Traits::kQInLds && s % kWaves != w) continue;
      const int d0 = 16 * s + 8 * g;
      u32x4_t x = load8<SMALL>(qrow, d0, p.D);
      if (!q_live || d0 >= p.D) x = u32x4_t{0u, 0u, 0u, 0u};
      if (!SMALL && d0 < p.D) {
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
    if (Traits::kQInLds) __syncthreads();
  }
  auto q_frag = [&](int s) {
    if constexpr (Traits::kQInLds) {
      return *reinterpret_cast<const u32x4_t*>(sQ + tile_at(c, 2 * s + g));
    } else {
      return qf[s];
    }
  };

  // Position of this lane's key (lanes c and c + 32 follow the same key) in the current step, and
  // the block metadata of the step that is loaded next.
  int slot, off;
  {
    const int pos = 32 * w + c;
    slot = pos / p.kb_eff;
    off = pos - slot * p.kb_eff;
  }
  int32_t m_idx = 0, m_type = kMasked, m_pid = -1;
  auto load_meta = [&]() {
    const bool in = slot < nb;
    const size_t o = moff + size_t(in ? slot : 0);
    m_idx = p.kv_indices[o];
    m_type = in ? p.types[o] : int32_t(kMasked);
    m_pid = has_partial ? p.partial_idx[o] : -1;
  };
  // The key of this lane in the step whose metadata has just been loaded.  `cmp`: the key is
  // allowed for the query rows >= cmp (all of them for FULL and PARTIAL, none for a key that does
  // not exist, lies beyond the sequence or belongs to a skipped slot).
  struct Key {
    int row, cmp, off, pid;
    bool live;
  };
  auto resolve = [&]() {
    Key k;
    const int kvb = m_idx < 0 ? 0 : (m_idx >= p.Tk ? p.Tk - 1 : m_idx);
    int mode = m_type;
    if (mode == kPartial && (m_pid < 0 || m_pid >= p.num_partial)) mode = kMasked;  // :119-131
    const long long row = (long long)kvb * p.KB + off;
    k.live = (mode == kCausal || mode == kFull || mode == kPartial) && row < p.seqlen;
    k.row = k.live ? int(row) : 0;
    k.cmp = !k.live ? 0x7fffffff : (mode == kCausal ? int(row) : -1);
    k.pid = (k.live && mode == kPartial) ? m_pid : -1;
    k.off = off;
    return k;
  };
  auto advance = [&]() {
    slot += p.adv_slot;
    off += p.adv_off;
    if (off >= p.kb_eff) {
      off -= p.kb_eff;
      ++slot;
    }
  };

  constexpr bool kPrefetchV = DT < 8;  // (at 256 columns the registers do not hold a step's V rows as well)
  u32x4_t kf[KS], vf[KS];
  auto load_rows = [&](const uint16_t* base, int64_t pitch, const Key& k, u32x4_t (&dst)[KS]) {
    const uint16_t* row = base + int64_t(k.row) * pitch;
#pragma unroll
    for (int s = 0; s < KS; ++s) dst[s] = load8<SMALL>(row, 16 * s + 8 * g, p.D);
  };

  const f32x16_t zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  f32x16_t ot[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) ot[dt] = zero16;
  float m_run = -INFINITY, l_run = 0.f;  // log2 domain; l_run is this lane's share of the row

  // A wave is done when the first position of its step is beyond the list.
  auto more = [&]() { return __builtin_amdgcn_readfirstlane(slot) < nb; };
  bool go = more() && p.seqlen > 0;
  Key cur = {0, 0x7fffffff, 0, -1, false};
  if (go) {
    load_meta();
    cur = resolve();
    load_rows(k_slab, p.k_at.row, cur, kf);
    if (kPrefetchV) load_rows(v_slab, p.v_at.row, cur, vf);
    advance();
    load_meta();
  }
  while (go) {
    if (!kPrefetchV) load_rows(v_slab, p.v_at.row, cur, vf);
    // what the softmax needs to know about the 32 keys, by key
    if (g == 0) {
      sKey[c] = cur.cmp;
      sOff[c] = cur.off;
      sPid[c] = cur.pid;
    }
    const bool any_partial = __builtin_amdgcn_ballot_w64(cur.pid >= 0) != 0;
    f32x16_t st = zero16;
#pragma unroll
    for (int s = 0; s < KS; ++s) st = mfma<BF16>(kf[s], q_frag(s), st);
    // V rows into the wave's tile
#pragma unroll
    for (int s = 0; s < KS; ++s)
      *reinterpret_cast<u32x4_t*>(sV + tile_at(c, 2 * s + g)) = cur.live ? vf[s] : u32x4_t{0u, 0u, 0u, 0u};
    // registers are free: the rows of the wave's next step, and the metadata of the one after it
    go = more();
    Key nxt = cur;
    if (go) {
      nxt = resolve();
      load_rows(k_slab, p.k_at.row, nxt, kf);
      if (kPrefetchV) load_rows(v_slab, p.v_at.row, nxt, vf);
      advance();
      load_meta();
    }
    // scores: register r is key 8 (r / 4) + 4 g + r % 4 of the step
    float mx = -INFINITY;
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const i32x4_t cmp = *reinterpret_cast<const i32x4_t*>(sKey + 8 * r4 + 4 * g);
      uint32_t bits = 0x01010101u;
      if (any_partial) {  // :143-154: any non-zero byte of the tile = attend
        const i32x4_t pid = *reinterpret_cast<const i32x4_t*>(sPid + 8 * r4 + 4 * g);
        const i32x4_t po = *reinterpret_cast<const i32x4_t*>(sOff + 8 * r4 + 4 * g);
        const int ql = q_here ? q_local : 0;
        if (p.mask_words) {  // the four keys are neighbours in one block
          const int p0 = pid[0], o0 = po[0];
          if (p0 >= 0) bits = *reinterpret_cast<const uint32_t*>(p.partial_masks + (size_t(p0) * p.QB + ql) * p.KB + o0);
        } else {
          bits = 0;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int pi = pid[i], oi = po[i];
            const uint32_t byte = pi >= 0 ? p.partial_masks[(size_t(pi) * p.QB + ql) * p.KB + oi] : 1u;
            bits |= byte << (8 * i);
          }
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float s = st[4 * r4 + i];
        if (p.softcap > 0.f) s = tanhf(s * p.scale / p.softcap) * p.softcap;
        s *= p.sl2;
        const int ci = cmp[i];
        s = (ci <= q_idx && ((bits >> (8 * i)) & 0xffu) != 0) ? s : -INFINITY;
        st[4 * r4 + i] = s;
        mx = fmaxf(mx, s);
      }
    }
    mx = fmaxf(mx, other_half(mx));
    const float m_new = fmaxf(m_run, mx);
    const float m_ref = m_new == -INFINITY ? 0.f : m_new;
    if (__builtin_amdgcn_ballot_w64(m_new > m_run) != 0) {
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_ref);
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) ot[dt][r] *= alpha;
      m_run = m_new;
    }
    u32x4_t pb[PARTS][2];
    float sum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      float p0 = __builtin_amdgcn_exp2f(st[r] - (m_ref - kShift));
      float p1 = __builtin_amdgcn_exp2f(st[r + 1] - (m_ref - kShift));
      sum += p0;
      sum += p1;
#pragma unroll
      for (int n = 0; n < PARTS; ++n) pb[n][r >> 3][(r & 7) >> 1] = split_part<BF16>(p0, p1);
    }
    l_run += sum;
    // O^T += V^T.P^T: k-slot e of lane group g in 16-key half ts is key 16 ts + 8 (e / 4) + 4 g + e % 4
    const int i16 = c & 15, j16 = c >> 4;
#pragma unroll
    for (int ts = 0; ts < 2; ++ts) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const int chunk = 2 * (2 * dt + j16) + ((i16 & 3) >> 1);
        const int r0 = 16 * ts + 4 * g + (i16 >> 2), r1 = r0 + 8;
        const uint8_t* a0 = sV + tile_at(r0, chunk) + (i16 & 1) * 8;
        const uint8_t* a1 = sV + tile_at(r1, chunk) + (i16 & 1) * 8;
        const u32x2_t lo = __builtin_bit_cast(
            u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(a0)));
        const u32x2_t hi = __builtin_bit_cast(
            u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(a1)));
        const u32x4_t a = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
        for (int n = 0; n < PARTS; ++n) ot[dt] = mfma<BF16>(a, pb[n][ts], ot[dt]);
      }
    }
    cur = nxt;
  }

  // Merge: row maxima and sums of the waves, then the O^T tiles, kGroup at a time: every wave
  // writes its tiles, wave i adds up and stores tile i of the group.
  l_run += other_half(l_run);
  if (g == 0) {
    sStat[w * 32 + c] = m_run;
    sStat[(kWaves + w) * 32 + c] = l_run;
  }
  __syncthreads();
  float m_all = -INFINITY;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) m_all = fmaxf(m_all, sStat[i * 32 + c]);
  const float m_fin = m_all == -INFINITY ? 0.f : m_all;
  float l_all = 0.f;
#pragma unroll
  for (int i = 0; i < kWaves; ++i)
    l_all += sStat[(kWaves + i) * 32 + c] * __builtin_amdgcn_exp2f(sStat[i * 32 + c] - m_fin);
  const bool some = q_live && l_all > 0.f;
  const float inv = some ? 1.f / l_all : 0.f;  // :283-288; rows without a key: zeros (:177-183)
  const float mine = __builtin_amdgcn_exp2f(m_run - m_fin) * inv;
  if (w == 0 && g == 0 && q_here && p.lse)
    p.lse[bh * p.S + q_idx] = some ? (m_fin + __builtin_amdgcn_logf(l_all) - kShift) * 0.6931471805599453f : -INFINITY;
  float* const stage = reinterpret_cast<float*>(lds);
  constexpr int G = Traits::kGroup;
#pragma unroll
  for (int d0 = 0; d0 < DT; d0 += G) {
    if (d0 > 0) __syncthreads();  // the previous group has been read
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
    __syncthreads();
    if (w < G && d0 + w < DT) {
      uint16_t* orow = p.o + (bh * p.S + q_idx) * p.D;
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        f32x4_t x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < kWaves; ++i)
          x += *reinterpret_cast<const f32x4_t*>(stage + ((size_t(i) * G + w) * 4 + r4) * 256 + lane * 4);
        if (!q_live) x = f32x4_t{0.f, 0.f, 0.f, 0.f};
        const int d = 32 * (d0 + w) + 8 * r4 + 4 * g;
        uint16_t h[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) h[j] = from_float<BF16>(x[j]);
        if (q_here) {
          if (p.o_vec) {  // D is a multiple of 8: four columns are inside together
            if (d < p.D) {
              const u32x2_t two = {uint32_t(h[0]) | uint32_t(h[1]) << 16, uint32_t(h[2]) | uint32_t(h[3]) << 16};
              *reinterpret_cast<u32x2_t*>(orow + d) = two;
            }
          } else {
            const int chunk = d & ~7;
            const int col = SMALL ? d : chunk_start(chunk, p.D) + (d & 7);
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (chunk < p.D && col + j < p.D && col + j >= chunk) orow[col + j] = h[j];
          }
        }
      }
    }
  }
}

constexpr int kMaxDevices = 64;

template <bool BF16, int DT, bool SMALL>
int launch(const GenericParams& p, unsigned grid, hipStream_t stream) {
  auto kern = fwd_generic_kernel<BF16, DT, SMALL>;
  const void* fn = reinterpret_cast<const void*>(kern);
  constexpr int lds = int(GenericTraits<DT>::kLdsBytes);
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
  void* args[] = {&params};
  return int(hipLaunchKernel(fn, dim3(grid), dim3(64 * kWaves), args, lds, stream));
}

template <bool BF16, int... I>
int launch_tiles(const GenericParams& p, unsigned grid, hipStream_t s, std::integer_sequence<int, I...>) {
  if (p.D < 8) return launch<BF16, 1, true>(p, grid, s);
  int rc = int(hipErrorInvalidValue);
  ((((p.D + 31) / 32 == I + 1) ? (void)(rc = launch<BF16, I + 1, false>(p, grid, s)) : (void)0), ...);
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
  if (Tq != (S_pad + QB - 1) / QB) return OMNI_ATTN_ERR_BAD_SHAPE;
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
  p.Tk = (S_pad + KB - 1) / KB;
  p.max_blocks = max_blocks;
  p.QB = QB;
  p.KB = KB;
  p.seqlen = seqlen_orig < S_pad ? seqlen_orig : S_pad;
  p.kb_eff = KB < S_pad ? KB : S_pad;
  p.adv_slot = 32 * kWaves / p.kb_eff;
  p.adv_off = 32 * kWaves % p.kb_eff;
  p.q_tiles = ((QB < S_pad ? QB : S_pad) + 31) / 32;
  p.mask_words = KB % 4 == 0 && p.kb_eff % 4 == 0 && !misaligned(partial_masks_or_null, 4);
  p.n_slabs = unsigned(B) * unsigned(H);
  p.scale = float(1.0 / std::sqrt(double(D)));
  p.softcap = softcap;
  // the factor of the scores in the log2 domain (a soft-capped score is scaled before the cap)
  p.sl2 = softcap > 0.f ? 1.4426950408889634f : float(1.4426950408889634 / std::sqrt(double(D)));
  p.o_vec = D % 8 == 0 && !misaligned(o, 8);
  const long long grid = (long long)B * H * Tq * p.q_tiles;
  if (grid > 0x7fffffffLL) return OMNI_ATTN_ERR_TOO_LARGE;
  const auto tiles = std::make_integer_sequence<int, kMaxD / 32>{};
  const int e = dtype == OMNI_ATTN_DTYPE_BF16
                    ? launch_tiles<true>(p, unsigned(grid), static_cast<hipStream_t>(stream), tiles)
                    : launch_tiles<false>(p, unsigned(grid), static_cast<hipStream_t>(stream), tiles);
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
