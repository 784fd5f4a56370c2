// Block mask of a prefix rule, built on the GPU.
//
// The masks of a mixed text / image batch have the form "row i of batch element b attends the keys
// below R[b, i]" (transfusion_pytorch/transfusion.py:343-356, :496-515: text is causal, a span
// (type, offset, length) also lets every row from its offset on see its end).  What the operator needs
// of it is the typed block list per (b, head, query block) and the tiles of the PARTIAL blocks, in
// (b, query block, slot) order, shared by the heads.  As tensor algebra that is some 80 launches
// over [B, S, S / KB] integers and two read-backs; here it is three kernels and one wait:
//   classify   one wave per (b, query block): the rows' R from the spans, the type of every key
//              block, the list compacted and written for all heads; the number of its PARTIAL tiles
//   number     one wave per (b, query block): the tiles before it, numbers for its PARTIAL slots, a
//              table of what each tile is; the total goes to the host (pinned memory), which waits
//              for it -- the caller's tile arrays have that size
//   tiles      one workgroup per tile: its bytes, and its bits where they are asked for
// All three are bound by their launches and a chain of a few memory latencies; the bytes
// (B=4 H=16 S=8192, 128x128 blocks: 3.1 MB of lists, 2.4 MB of tiles) take a microsecond.  That mask,
// packed: 472 us as tensor algebra, 39 us so (kernels 8 + 4 + 5 us, the rest launches and the wait).
#include "../../include/omni_attn_gfx950.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace omni_attn {
// Keeps the hipError_t behind an OMNI_ATTN_ERR_LAUNCH for omni_attn_last_hip_error() (defined
// beside that function).
void record_hip_error(int hip_error);
}  // namespace omni_attn

namespace {

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

enum : int { kCausal = 1, kFull = 2, kPartial = 3 };

struct MaskParams {
  const int64_t* spans;   // [B, M, 3] rows of (type, offset, length), or null
  const int64_t* prefix;  // [B, q_len] allowed-prefix lengths, or null (one of the two is given)
  int32_t* nb;            // [B, H, Tq]
  int32_t* idx;           // [B, H, Tq, Tk]
  int32_t* types;         // [B, H, Tq, Tk]
  int32_t* pidx;          // [B, H, Tq, Tk]
  int32_t* counts;        // [B * Tq] PARTIAL tiles of a query block
  int32_t* tile_src;      // [B * Tq * Tk] (b, query block, key block) of a tile, as one index
  int32_t* host_total;    // pinned: [0] the number of tiles, [1] the ticket, written after it
  int ticket;
  int B, M, H, Tq, Tk, QB, KB, q_len, kv_len;
};

// Spans of a batch element that are worked at a time: (offset, end) pairs in LDS.
constexpr int kSpanChunk = 64;

// Keys of batch element b that the rows first .. first + QB - 1 attend: a prefix each, its length to
// reach[].  `spans`: 2 kSpanChunk words of LDS.  Called by all NT threads of the workgroup.
template <int NT>
__device__ __forceinline__ void row_reaches(const MaskParams& p, int b, int first, int32_t* reach, int64_t* spans) {
  for (int r = threadIdx.x; r < p.QB; r += NT) {
    const int i = first + r;
    int64_t n = int64_t(i) + 1;
    if (i >= p.q_len) {
      n = 0;
    } else if (p.prefix != nullptr) {
      n = p.prefix[size_t(b) * p.q_len + i];
      n = n < 0 ? 0 : n;
    }
    reach[r] = int(n < p.kv_len ? n : p.kv_len);
  }
  if (p.spans == nullptr) return;
  const int64_t* sp = p.spans + size_t(b) * p.M * 3;
  for (int m0 = 0; m0 < p.M; m0 += kSpanChunk) {
    __syncthreads();
    const int n_spans = p.M - m0 < kSpanChunk ? p.M - m0 : kSpanChunk;
    if (threadIdx.x < n_spans) {
      const int64_t off = sp[3 * (m0 + threadIdx.x) + 1], len = sp[3 * (m0 + threadIdx.x) + 2];
      const int64_t end = len > 0 ? off + len : 0;
      spans[2 * threadIdx.x] = off;
      spans[2 * threadIdx.x + 1] = end < p.kv_len ? end : p.kv_len;
    }
    __syncthreads();
    for (int r = threadIdx.x; r < p.QB; r += NT) {
      const int i = first + r;
      if (i >= p.q_len) continue;
      int64_t n = reach[r];
      for (int m = 0; m < n_spans; ++m)
        if (int64_t(i) >= spans[2 * m] && spans[2 * m + 1] > n) n = spans[2 * m + 1];
      reach[r] = int(n);
    }
  }
}

__device__ __forceinline__ int clamp_to(int x, int hi) { return x < 0 ? 0 : (x > hi ? hi : x); }

__global__ void __launch_bounds__(64) mask_classify_kernel(const MaskParams p) {
  __shared__ int64_t spans[2 * kSpanChunk];
  extern __shared__ int32_t reach[];  // [QB]
  const int lane = threadIdx.x;
  const int row = blockIdx.x;  // (b, query block)
  const int b = row / p.Tq, qb = row - b * p.Tq;
  row_reaches<64>(p, b, qb * p.QB, reach, spans);
  __syncthreads();
  int lo = 0x7fffffff, hi = 0;
  for (int r = lane; r < p.QB; r += 64) {
    const int v = reach[r];
    lo = v < lo ? v : lo;
    hi = v > hi ? v : hi;
  }
  for (int m = 32; m >= 1; m >>= 1) {
    const int l2 = __shfl_xor(lo, m, 64), h2 = __shfl_xor(hi, m, 64);
    lo = l2 < lo ? l2 : lo;
    hi = h2 > hi ? h2 : hi;
  }
  int listed = 0, partial = 0;
  for (int kb0 = 0; kb0 < p.Tk; kb0 += 64) {
    const int kb = kb0 + lane;
    const int k0 = kb * p.KB;
    const bool active = kb < p.Tk && hi > k0;
    const bool full = active && lo >= k0 + p.KB;
    // the few blocks that are neither: CAUSAL if every row's part of the block is what the causal
    // pattern gives it.  A lane looks at rows here, one block at a time.
    uint64_t open = __ballot(active && !full), causal = 0;
    for (uint64_t left = open; left != 0; left &= left - 1) {
      const int j = __builtin_ctzll(left);
      const int kj = (kb0 + j) * p.KB;
      bool same = true;
      for (int r = lane; r < p.QB; r += 64)
        same &= clamp_to(reach[r] - kj, p.KB) == clamp_to(qb * p.QB + r + 1 - kj, p.KB);
      if (__ballot(!same) == 0) causal |= 1ull << j;
    }
    const int type = !active ? 0 : (full ? kFull : ((causal >> lane) & 1 ? kCausal : kPartial));
    const uint64_t act = __ballot(active);
    partial += __popcll(__ballot(type == kPartial));
    const int slot = listed + __popcll(act & ((1ull << lane) - 1));
    listed += __popcll(act);
    if (active)
      for (int h = 0; h < p.H; ++h) {
        const size_t o = ((size_t(b) * p.H + h) * p.Tq + qb) * p.Tk + slot;
        p.idx[o] = kb;
        p.types[o] = type;
      }
  }
  for (int h = 0; h < p.H; ++h) {  // zeros behind the list
    const size_t o = ((size_t(b) * p.H + h) * p.Tq + qb) * p.Tk;
    for (int s = listed + lane; s < p.Tk; s += 64) {
      p.idx[o + s] = 0;
      p.types[o + s] = 0;
    }
  }
  for (int h = lane; h < p.H; h += 64) p.nb[(size_t(b) * p.H + h) * p.Tq + qb] = listed;
  if (lane == 0) p.counts[row] = partial;
}

__global__ void __launch_bounds__(64) mask_number_kernel(const MaskParams p) {
  const int lane = threadIdx.x;
  const int row = blockIdx.x;
  const int b = row / p.Tq, qb = row - b * p.Tq;
  const int n = p.B * p.Tq;
  int before = 0, all = 0;
  for (int i = lane; i < n; i += 64) {
    const int c = p.counts[i];
    all += c;
    before += i < row ? c : 0;
  }
  for (int m = 32; m >= 1; m >>= 1) {
    before += __shfl_xor(before, m, 64);
    all += __shfl_xor(all, m, 64);
  }
  if (row == 0 && lane == 0) {
    __hip_atomic_store(p.host_total, all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(p.host_total + 1, p.ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  const size_t o0 = (size_t(b) * p.H * p.Tq + qb) * p.Tk;  // head 0
  for (int s0 = 0; s0 < p.Tk; s0 += 64) {
    const int s = s0 + lane;
    const bool is_p = s < p.Tk && p.types[o0 + s] == kPartial;
    const uint64_t bits = __ballot(is_p);
    const int pid = before + __popcll(bits & ((1ull << lane) - 1));
    before += __popcll(bits);
    if (is_p) p.tile_src[pid] = row * p.Tk + p.idx[o0 + s];
    if (s < p.Tk)
      for (int h = 0; h < p.H; ++h) p.pidx[o0 + size_t(h) * p.Tq * p.Tk + s] = is_p ? pid : -1;
  }
}

__global__ void __launch_bounds__(256) mask_tiles_kernel(const MaskParams p, uint8_t* __restrict__ tiles,
                                                         uint32_t* __restrict__ bits) {
  __shared__ int64_t spans[2 * kSpanChunk];
  extern __shared__ int32_t reach[];  // [QB]
  const int src = p.tile_src[blockIdx.x];
  const int row = src / p.Tk, kb = src - row * p.Tk;
  const int b = row / p.Tq, qb = row - b * p.Tq;
  row_reaches<256>(p, b, qb * p.QB, reach, spans);
  __syncthreads();
  const int k0 = kb * p.KB;
  uint8_t* const tile = tiles + size_t(blockIdx.x) * p.QB * p.KB;
  if (p.KB % 16 == 0) {
    const int per_row = p.KB / 16;
    for (int i = threadIdx.x; i < p.QB * per_row; i += 256) {
      const int r = i / per_row, c0 = (i - r * per_row) * 16;
      const int n = clamp_to(reach[r] - k0 - c0, 16);
      u32x4_t x;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int m = clamp_to(n - 4 * j, 4);
        x[j] = m == 0 ? 0u : 0x01010101u >> (8 * (4 - m));
      }
      *reinterpret_cast<u32x4_t*>(tile + size_t(i) * 16) = x;
    }
  } else {
    for (int i = threadIdx.x; i < p.QB * p.KB; i += 256) {
      const int r = i / p.KB;
      tile[i] = k0 + (i - r * p.KB) < reach[r] ? 1 : 0;
    }
  }
  if (bits != nullptr) {
    const int words = p.KB / 32;
    uint32_t* const out = bits + size_t(blockIdx.x) * p.QB * words;
    for (int i = threadIdx.x; i < p.QB * words; i += 256) {
      const int r = i / words;
      const int n = clamp_to(reach[r] - k0 - (i - r * words) * 32, 32);
      out[i] = n == 32 ? 0xffffffffu : (1u << n) - 1u;
    }
  }
}

int bad_shape(int B, int M, int H, int q_len, int kv_len, int QB, int KB) {
  if (B <= 0 || M < 0 || H <= 0 || q_len <= 0 || kv_len <= 0 || QB <= 0 || KB <= 0) return OMNI_ATTN_ERR_BAD_SHAPE;
  if (QB > OMNI_ATTN_MASK_MAX_QB || (long long)q_len + QB > 0x7fffffffLL || (long long)kv_len + KB > 0x7fffffffLL)
    return OMNI_ATTN_ERR_TOO_LARGE;
  const long long Tq = ((long long)q_len + QB - 1) / QB, Tk = ((long long)kv_len + KB - 1) / KB;
  if (B * Tq > 0x7fffffffLL || (long long)B * Tq > 0x7fffffffLL / Tk) return OMNI_ATTN_ERR_TOO_LARGE;
  return OMNI_ATTN_OK;
}

MaskParams common(const int64_t* spans, const int64_t* prefix, void* workspace, int B, int M, int H, int q_len,
                  int kv_len, int QB, int KB) {
  MaskParams p = {};
  p.spans = spans;
  p.prefix = prefix;
  p.B = B;
  p.M = M;
  p.H = H;
  p.QB = QB;
  p.KB = KB;
  p.q_len = q_len;
  p.kv_len = kv_len;
  p.Tq = (q_len + QB - 1) / QB;
  p.Tk = (kv_len + KB - 1) / KB;
  p.counts = static_cast<int32_t*>(workspace);
  p.tile_src = p.counts + size_t(B) * p.Tq;
  return p;
}

int launched(hipError_t e) {
  if (e == hipSuccess) return OMNI_ATTN_OK;
  omni_attn::record_hip_error(int(e));
  return OMNI_ATTN_ERR_LAUNCH;
}

}  // namespace

extern "C" size_t omni_attn_mask_workspace_bytes(int B, int q_len, int kv_len, int QB, int KB) {
  if (bad_shape(B, 0, 1, q_len, kv_len, QB, KB) != OMNI_ATTN_OK) return 0;
  const size_t Tq = size_t((q_len + QB - 1) / QB), Tk = size_t((kv_len + KB - 1) / KB);
  return (size_t(B) * Tq + size_t(B) * Tq * Tk) * sizeof(int32_t);
}

extern "C" int omni_attn_mask_lists_gfx950(const int64_t* spans_or_null, const int64_t* prefix_or_null,
                                           int32_t* kv_num_blocks, int32_t* kv_indices, int32_t* block_mask_types,
                                           int32_t* partial_idx, void* workspace, int32_t* host_total, int ticket,
                                           int B, int M, int H, int q_len, int kv_len, int QB, int KB, void* stream) {
  if ((!spans_or_null == !prefix_or_null) || !kv_num_blocks || !kv_indices || !block_mask_types || !partial_idx ||
      !workspace || !host_total)
    return OMNI_ATTN_ERR_NULL_POINTER;
  if (const int rc = bad_shape(B, M, H, q_len, kv_len, QB, KB)) return rc;
  MaskParams p = common(spans_or_null, prefix_or_null, workspace, B, M, H, q_len, kv_len, QB, KB);
  p.nb = kv_num_blocks;
  p.idx = kv_indices;
  p.types = block_mask_types;
  p.pidx = partial_idx;
  p.host_total = host_total;
  p.ticket = ticket;
  const dim3 grid(unsigned(B) * unsigned(p.Tq));
  void* args[] = {&p};
  hipError_t e = hipLaunchKernel(reinterpret_cast<const void*>(mask_classify_kernel), grid, dim3(64), args,
                                 size_t(QB) * sizeof(int32_t), static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return launched(e);
  e = hipLaunchKernel(reinterpret_cast<const void*>(mask_number_kernel), grid, dim3(64), args, 0,
                      static_cast<hipStream_t>(stream));
  return launched(e);
}

extern "C" int omni_attn_mask_tiles_gfx950(const int64_t* spans_or_null, const int64_t* prefix_or_null,
                                           void* workspace, uint8_t* partial_masks, uint32_t* partial_bits_or_null,
                                           int num_partial, int B, int M, int H, int q_len, int kv_len, int QB, int KB,
                                           void* stream) {
  if (num_partial == 0) return OMNI_ATTN_OK;
  if ((!spans_or_null == !prefix_or_null) || !workspace || !partial_masks) return OMNI_ATTN_ERR_NULL_POINTER;
  if (const int rc = bad_shape(B, M, H, q_len, kv_len, QB, KB)) return rc;
  if (num_partial < 0 || (partial_bits_or_null && KB % 32 != 0)) return OMNI_ATTN_ERR_BAD_SHAPE;
  if ((reinterpret_cast<uintptr_t>(partial_masks) & 15) != 0 || (reinterpret_cast<uintptr_t>(partial_bits_or_null) & 3) != 0)
    return OMNI_ATTN_ERR_MISALIGNED;
  MaskParams p = common(spans_or_null, prefix_or_null, workspace, B, M, H, q_len, kv_len, QB, KB);
  if ((long long)num_partial > (long long)B * p.Tq * p.Tk) return OMNI_ATTN_ERR_BAD_SHAPE;
  void* args[] = {&p, &partial_masks, &partial_bits_or_null};
  return launched(hipLaunchKernel(reinterpret_cast<const void*>(mask_tiles_kernel), dim3(unsigned(num_partial)),
                                  dim3(256), args, size_t(QB) * sizeof(int32_t), static_cast<hipStream_t>(stream)));
}
