// Block mask of a prefix rule, built on the GPU.
//
// The masks of a mixed text / image batch have the form "row i of batch element b attends the keys
// below R[b, i]" (transfusion_pytorch/transfusion.py:343-356, :496-515: text is causal, a span
// (type, offset, length) also lets every row from its offset on see its end).  What the operator needs
// of it is the typed block list per (b, head, query block) and the tiles of the PARTIAL blocks, in
// (b, query block, slot) order, shared by the heads.  As tensor algebra that is some 80 launches
// over [B, S, S / KB] integers and two read-backs; here it is two kernels and one wait between them:
//   classify   one workgroup per (b, query block): the rows' R from the spans; the blocks below the smallest are FULL,
//              the blocks from the largest on are not listed, and the few between get their type from a look at
//              the rows.  Each sends the number of its PARTIAL tiles to the host (one word of pinned memory), which
//              adds them up -- the caller's tile arrays have that size -- while the lists are allocated
//   write      one workgroup per (b, query block) and four heads, a head per wave, writes the list and the tile
//              numbers (the tiles before the query block are a sum over the counts), and one per tile, which finds
//              its query block by a scan of the counts, writes its bytes, and its bits where they are asked for
// With many query blocks a sum and a scan per workgroup, and a word per query block over the bus, are what a call takes;
// there a kernel of one workgroup sums up the counts once (and sends their total): a call, us, B=32 H=16 S=65536
// 1097 -> 415, B=64 H=4 S=65536 3739 -> 416, B=64 H=16 S=8192 127 -> 54 (the host's share of that: a word instead of 4096).
// Both are bound by their launches and a chain of a few memory latencies; the bytes
// (B=4 H=16 S=8192, 128x128 blocks: 3.1 MB of lists, 2.4 MB of tiles) take a microsecond.  That mask,
// packed, in calls back to back: 472 us as tensor algebra; 38 us as three kernels (8.2, 3.9 and 5.0 us)
// with the wait behind the second; 32 us so (4.9 and 5.8 us; 20 us of a call pass between the first launch and its last
// count on the host).
#include "../../include/omni_attn_gfx950.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

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
  int32_t* full;          // [B * Tq] leading FULL blocks of its list
  int32_t* listed;        // [B * Tq] blocks of its list: 0, 1, ...
  int32_t* before;        // [B * Tq] PARTIAL tiles of the query blocks before it; null: summed up where needed
  int32_t* open;          // [B * Tq * Tk] types of the blocks full .. listed - 1
  int32_t* reach;         // [B * Tq * QB] keys that a row attends
  uint32_t* posted;       // pinned, or null: [B * Tq] tag in the upper 12 bits, count in the lower 20
  int32_t* host_total;    // pinned, or null: [0] the number of tiles, [1] the ticket
  int ticket;
  int num_partial;        // tiles that there is room for
  int head_groups;        // workgroups per query block that write lists
  int B, M, H, Tq, Tk, QB, KB, q_len, kv_len;
};

constexpr int kPostedCountBits = OMNI_ATTN_MASK_POSTED_COUNT_BITS;
// Query blocks up to which the lists and tiles sum the counts up where they need them: every workgroup reads the counts
// before its own, and another launch costs 3 us.  In calls back to back, us, with and without that launch: 1024 query
// blocks (B=16 H=16 S=8192) 40.9 / 37.6, 2048 (S=16384) 62.0 / 65.7, 4096 (B=64 S=8192) 98 / 129.
constexpr int kSumRows = 1024;

// Spans of a batch element that are worked at a time: (offset, end) pairs in LDS.
constexpr int kSpanChunk = 64;

__device__ __forceinline__ int clamp_to(int x, int hi) { return x < 0 ? 0 : (x > hi ? hi : x); }

// Smallest (or largest) x of a wave, for x >= 0: through the lanes of the vector pipe, without LDS.
template <bool MAX>
__device__ __forceinline__ int wave_extreme(int x) {
  auto step = [&](auto ctrl) {
    const int other = __builtin_amdgcn_update_dpp(x, x, decltype(ctrl)::value, 0xf, 0xf, false);
    x = (MAX ? other > x : other < x) ? other : x;
  };
  step(std::integral_constant<int, 0x111>{});  // row_shr 1, 2, 4, 8
  step(std::integral_constant<int, 0x112>{});
  step(std::integral_constant<int, 0x114>{});
  step(std::integral_constant<int, 0x118>{});
  step(std::integral_constant<int, 0x142>{});  // row_bcast 15, 31
  step(std::integral_constant<int, 0x143>{});
  return __builtin_amdgcn_readlane(x, 63);
}

// One workgroup per (b, query block), a thread per row (and every 256th after it).
__global__ void __launch_bounds__(256) mask_classify_kernel(const MaskParams p) {
  __shared__ int2 spans[kSpanChunk];
  __shared__ int lows[4], highs[4];
  __shared__ uint64_t partials[4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int row = blockIdx.x;  // (b, query block)
  const int b = row / p.Tq, qb = row - b * p.Tq;
  const int first = qb * p.QB;
  int32_t* const reach = p.reach + size_t(row) * p.QB;  // (a thread reads what it has written itself)
  int mine = 0;  // of the first of its rows
  int lo = 0x7fffffff, hi = 0;
  for (int r = threadIdx.x; r < p.QB; r += 256) {
    const int i = first + r;
    int64_t n = int64_t(i) + 1;
    if (i >= p.q_len) {
      n = 0;
    } else if (p.prefix != nullptr) {
      n = p.prefix[size_t(b) * p.q_len + i];
      n = n < 0 ? 0 : n;
    }
    const int own = int(n < p.kv_len ? n : p.kv_len);
    if (r < 256) mine = own;
    if (p.spans == nullptr || r >= 256) reach[r] = own;
  }
  if (p.spans != nullptr) {
    const int64_t* sp = p.spans + size_t(b) * p.M * 3;
    for (int m0 = 0; m0 < p.M; m0 += kSpanChunk) {
      if (m0 > 0) __syncthreads();
      const int n_spans = p.M - m0 < kSpanChunk ? p.M - m0 : kSpanChunk;
      if (threadIdx.x < n_spans) {
        const int64_t off = sp[3 * (m0 + threadIdx.x) + 1], len = sp[3 * (m0 + threadIdx.x) + 2];
        const int64_t end = len > 0 ? off + len : 0;
        // (rows are below 2^31 - 1)
        spans[threadIdx.x] = {int(off < 0 ? 0 : (off < 0x7fffffff ? off : 0x7fffffff)),
                              int(end < 0 ? 0 : (end < p.kv_len ? end : p.kv_len))};
      }
      __syncthreads();
      for (int r = threadIdx.x; r < p.QB; r += 256) {
        const int i = first + r;
        if (i >= p.q_len) continue;
        int n = r < 256 ? mine : reach[r];
#pragma unroll 4
        for (int m = 0; m < n_spans; ++m) {
          const int2 span = spans[m];
          if (i >= span.x && span.y > n) n = span.y;
        }
        if (r < 256) mine = n; else reach[r] = n;
      }
    }
    if (threadIdx.x < p.QB) reach[threadIdx.x] = mine;
  }
  for (int r = threadIdx.x; r < p.QB; r += 256) {
    const int v = r < 256 ? mine : reach[r];
    lo = v < lo ? v : lo;
    hi = v > hi ? v : hi;
  }
  lo = wave_extreme<false>(lo);
  hi = wave_extreme<true>(hi);
  if (lane == 0) {
    lows[w] = lo;
    highs[w] = hi;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    lo = lows[i] < lo ? lows[i] : lo;
    hi = highs[i] > hi ? highs[i] : hi;
  }
  const int full = lo / p.KB, listed = (hi + p.KB - 1) / p.KB;
  // The few blocks that are neither FULL nor left out: CAUSAL if every row's part of the block is what the causal
  // pattern gives it.  A row that attends R keys where causal is c differs from that in the blocks between the two.
  int partial = 0;
  for (int kb0 = full; kb0 < listed; kb0 += 64) {
    const int n = listed - kb0 < 64 ? listed - kb0 : 64;
    uint64_t differ = 0;  // (wave-uniform)
    for (int r0 = 0; r0 < p.QB; r0 += 256) {
      const int r = r0 + threadIdx.x;
      int from = 0, to = 0;
      if (r < p.QB) {
        const int v = r < 256 ? mine : reach[r], c = first + r + 1;
        const int a = v < c ? v : c, z = v < c ? c : v;
        if (a != z) {
          from = a / p.KB;
          to = (z - 1) / p.KB + 1;
        }
      }
      for (int i = 0; i < n; ++i)
        if (__ballot(kb0 + i >= from && kb0 + i < to) != 0) differ |= 1ull << i;
    }
    if (kb0 > full) __syncthreads();
    if (lane == 0) partials[w] = differ;
    __syncthreads();
    differ = partials[0] | partials[1] | partials[2] | partials[3];
    partial += __popcll(differ);
    if (threadIdx.x < n) p.open[size_t(row) * p.Tk + kb0 + threadIdx.x] = (differ >> threadIdx.x) & 1 ? kPartial : kCausal;
  }
  if (threadIdx.x == 0) {
    if (p.posted != nullptr)
      __hip_atomic_store(p.posted + row, uint32_t(p.ticket) << kPostedCountBits | uint32_t(partial), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_SYSTEM);
    p.counts[row] = partial;
    p.full[row] = full;
    p.listed[row] = listed;
  }
}

// Sum over a workgroup of four waves; `part`: 4 words of LDS.
__device__ __forceinline__ int sum_of_256(int x, int32_t* part) {
  for (int m = 32; m >= 1; m >>= 1) x += __shfl_xor(x, m, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = x;
  __syncthreads();
  return part[0] + part[1] + part[2] + part[3];
}

// The tiles before each query block, by one workgroup, a wave per run of query blocks; their number goes to the host as
// one word where that is asked for.
__global__ void __launch_bounds__(1024) mask_number_kernel(const MaskParams p) {
  __shared__ int32_t part[16];
  const unsigned lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const unsigned n = unsigned(p.B) * unsigned(p.Tq);
  const unsigned run = ((n + 63) / 64 + 15) / 16 * 64;  // query blocks of a wave
  const unsigned first = w * run, last = first + run < n ? first + run : n;
  int sum = 0;
  for (unsigned i = first + lane; i < last; i += 64) sum += p.counts[i];
  for (int m = 32; m >= 1; m >>= 1) sum += __shfl_xor(sum, m, 64);
  if (lane == 0) part[w] = sum;
  __syncthreads();
  int upto = 0, all = 0;
  for (unsigned i = 0; i < 16; ++i) {
    upto += i < w ? part[i] : 0;
    all += part[i];
  }
  for (unsigned i0 = first; i0 < last; i0 += 64) {
    const unsigned i = i0 + lane;
    const int own = i < last ? p.counts[i] : 0;
    int here = own;  // inclusive sum over the lanes
    for (unsigned d = 1; d < 64; d <<= 1) {
      const int other = __shfl_up(here, d, 64);
      here += lane >= d ? other : 0;
    }
    if (i < last) p.before[i] = upto + here - own;
    upto += __shfl(here, 63, 64);
  }
  if (threadIdx.x == 0 && p.host_total != nullptr) {
    __hip_atomic_store(p.host_total, all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(p.host_total + 1, p.ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// One tile: its bytes, and its bits.
__device__ __forceinline__ void write_tile(const MaskParams& p, const int32_t* reach, int k0, uint8_t* tile, uint32_t* bits) {
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
    for (int i = threadIdx.x; i < p.QB * words; i += 256) {
      const int r = i / words;
      const int n = clamp_to(reach[r] - k0 - (i - r * words) * 32, 32);
      bits[i] = n == 32 ? 0xffffffffu : (1u << n) - 1u;
    }
  }
}

// The workgroups 0 .. num_partial - 1 write a tile each, the others the lists of four heads in a query block each.
__global__ void __launch_bounds__(256) mask_write_kernel(const MaskParams p, uint8_t* __restrict__ tiles,
                                                         uint32_t* __restrict__ bits) {
  __shared__ int32_t part[4];
  __shared__ int32_t found[2];  // query block of the tile, and which of its PARTIAL blocks
  extern __shared__ int32_t reach[];  // [QB]
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int n_rows = p.B * p.Tq;
  if (int(blockIdx.x) < p.num_partial) {
    const int tile = blockIdx.x;
    int row = 0, left;
    if (p.before != nullptr) {
      for (int n = n_rows; n > 1;) {  // it is one of the query blocks row .. row + n - 1: 256 looks at a time
        const int step = (n + 255) / 256, at = int(threadIdx.x) * step;
        const int c = __syncthreads_count(at < n && p.before[row + at] <= tile) - 1;
        row += c * step;
        n = n - c * step < step ? n - c * step : step;
      }
      left = tile - p.before[row];
      if (left >= p.counts[row]) return;  // there is room for more tiles than the mask has
    } else {
      // a thread looks at `per` neighbouring query blocks
      const int per = (n_rows + 255) / 256, r0 = threadIdx.x * per, r1 = r0 + per < n_rows ? r0 + per : n_rows;
      int mine = 0;
      for (int r = r0; r < r1; ++r) mine += p.counts[r];
      int upto = mine;  // inclusive sum over the threads
      for (int d = 1; d < 64; d <<= 1) {
        const int other = __shfl_up(upto, d, 64);
        upto += lane >= d ? other : 0;
      }
      if (lane == 63) part[w] = upto;
      if (threadIdx.x == 0) found[0] = -1;
      __syncthreads();
      for (int i = 0; i < w; ++i) upto += part[i];
      left = tile - (upto - mine);
      if (left >= 0 && left < mine) {
        int r = r0;
        for (int c = p.counts[r]; left >= c; c = p.counts[++r]) left -= c;
        found[0] = r;
        found[1] = left;
      }
      __syncthreads();
      row = found[0];
      if (row < 0) return;  // (as above)
      left = found[1];
    }
    for (int r = threadIdx.x; r < p.QB; r += 256) reach[r] = p.reach[size_t(row) * p.QB + r];
    const int listed = p.listed[row];
    int kb = p.full[row];
    for (;; kb += 64) {  // (the block is in the list)
      const bool is = kb + lane < listed && p.open[size_t(row) * p.Tk + kb + lane] == kPartial;
      uint64_t partials = __ballot(is);
      const int n = __popcll(partials);
      if (left < n) {
        for (; left > 0; --left) partials &= partials - 1;
        kb += __builtin_ctzll(partials);
        break;
      }
      left -= n;
      if (kb + 64 >= listed) return;
    }
    __syncthreads();
    const size_t at = size_t(tile) * p.QB * p.KB;
    write_tile(p, reach, kb * p.KB, tiles + at, bits != nullptr ? bits + at / 32 : nullptr);
    return;
  }
  const int item = blockIdx.x - p.num_partial;
  const int row = item / p.head_groups, group = item - row * p.head_groups;
  const int b = row / p.Tq, qb = row - b * p.Tq;
  const int full = p.full[row], listed = p.listed[row];
  int before;  // tiles of the query blocks before this one
  if (p.before != nullptr) {
    before = p.before[row];
  } else {
    int x = 0;
    for (int i = threadIdx.x; i < row; i += 256) x += p.counts[i];
    before = sum_of_256(x, part);
  }
  for (int s0 = 0; s0 < p.Tk; s0 += 64) {
    const int s = s0 + lane;
    int type = s < full ? kFull : 0;
    if (s >= full && s < listed) type = p.open[size_t(row) * p.Tk + s];
    const uint64_t partials = __ballot(type == kPartial);
    const int pid = type == kPartial ? before + __popcll(partials & ((1ull << lane) - 1)) : -1;
    before += __popcll(partials);
    if (s >= p.Tk) continue;
    for (int h = group * 4 + w; h < p.H; h += p.head_groups * 4) {
      const size_t o = ((size_t(b) * p.H + h) * p.Tq + qb) * p.Tk + s;
      p.idx[o] = s < listed ? s : 0;
      p.types[o] = type;
      p.pidx[o] = pid;
    }
  }
  for (int h = group * 4 + w; h < p.H; h += p.head_groups * 4)
    if (lane == 0) p.nb[(size_t(b) * p.H + h) * p.Tq + qb] = listed;
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
  const size_t rows = size_t(B) * p.Tq;
  p.counts = static_cast<int32_t*>(workspace);
  p.full = p.counts + rows;
  p.listed = p.full + rows;
  p.before = p.listed + rows;
  p.open = p.before + rows;
  p.reach = p.open + rows * p.Tk;
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
  return size_t(B) * Tq * (4 + Tk + QB) * sizeof(int32_t);
}

namespace {
int launch_classify(const MaskParams& params, hipStream_t stream) {
  MaskParams p = params;
  void* args[] = {&p};
  return launched(hipLaunchKernel(reinterpret_cast<const void*>(mask_classify_kernel), dim3(unsigned(p.B) * unsigned(p.Tq)),
                                  dim3(256), args, 0, stream));
}
int launch_number(const MaskParams& params, hipStream_t stream) {
  MaskParams p = params;
  void* args[] = {&p};
  return launched(hipLaunchKernel(reinterpret_cast<const void*>(mask_number_kernel), dim3(1), dim3(1024), args, 0, stream));
}
// Lists (where p.nb is given) and tiles (where there are any), in one launch.
int launch_write(const MaskParams& params, uint8_t* tiles, uint32_t* bits, hipStream_t stream) {
  MaskParams p = params;
  const long long rows = (long long)p.B * p.Tq, room = 0x7fffffffLL - p.num_partial;
  const long long by_four = (p.H + 3) / 4;
  p.head_groups = p.nb == nullptr ? 0 : int(by_four * rows <= room ? by_four : (room / rows > 1 ? room / rows : 1));
  const long long grid = p.num_partial + rows * p.head_groups;
  if (grid > 0x7fffffffLL) return OMNI_ATTN_ERR_TOO_LARGE;
  void* args[] = {&p, &tiles, &bits};
  return launched(hipLaunchKernel(reinterpret_cast<const void*>(mask_write_kernel), dim3(unsigned(grid)), dim3(256), args,
                                  p.num_partial > 0 ? size_t(p.QB) * sizeof(int32_t) : 0, stream));
}
int check_tiles(const uint8_t* partial_masks, const uint32_t* partial_bits_or_null, int num_partial, const MaskParams& p) {
  if (num_partial < 0 || (partial_bits_or_null && p.KB % 32 != 0)) return OMNI_ATTN_ERR_BAD_SHAPE;
  if ((reinterpret_cast<uintptr_t>(partial_masks) & 15) != 0 || (reinterpret_cast<uintptr_t>(partial_bits_or_null) & 3) != 0)
    return OMNI_ATTN_ERR_MISALIGNED;
  return (long long)num_partial > (long long)p.B * p.Tq * p.Tk ? OMNI_ATTN_ERR_BAD_SHAPE : OMNI_ATTN_OK;
}
}  // namespace

extern "C" int omni_attn_mask_classify_gfx950(const int64_t* spans_or_null, const int64_t* prefix_or_null,
                                              void* workspace, uint32_t* posted, int tag, int B, int M, int q_len,
                                              int kv_len, int QB, int KB, void* stream) {
  if ((!spans_or_null == !prefix_or_null) || !workspace || !posted) return OMNI_ATTN_ERR_NULL_POINTER;
  if (const int rc = bad_shape(B, M, 1, q_len, kv_len, QB, KB)) return rc;
  MaskParams p = common(spans_or_null, prefix_or_null, workspace, B, M, 1, q_len, kv_len, QB, KB);
  if (p.Tk >> kPostedCountBits != 0 || tag < 0 || tag >> (32 - kPostedCountBits) != 0) return OMNI_ATTN_ERR_TOO_LARGE;
  p.posted = posted;
  p.ticket = tag;
  return launch_classify(p, static_cast<hipStream_t>(stream));
}

extern "C" int omni_attn_mask_finish_gfx950(int32_t* kv_num_blocks, int32_t* kv_indices, int32_t* block_mask_types,
                                            int32_t* partial_idx, void* workspace, uint8_t* partial_masks_or_null,
                                            uint32_t* partial_bits_or_null, int num_partial, int B, int H, int q_len,
                                            int kv_len, int QB, int KB, void* stream) {
  if (!kv_num_blocks || !kv_indices || !block_mask_types || !partial_idx || !workspace ||
      (num_partial > 0 && !partial_masks_or_null))
    return OMNI_ATTN_ERR_NULL_POINTER;
  if (const int rc = bad_shape(B, 0, H, q_len, kv_len, QB, KB)) return rc;
  MaskParams p = common(nullptr, nullptr, workspace, B, 0, H, q_len, kv_len, QB, KB);
  if (const int rc = check_tiles(partial_masks_or_null, partial_bits_or_null, num_partial, p)) return rc;
  p.nb = kv_num_blocks;
  p.idx = kv_indices;
  p.types = block_mask_types;
  p.pidx = partial_idx;
  p.num_partial = num_partial;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (p.B * p.Tq <= kSumRows) {
    p.before = nullptr;
  } else if (const int rc = launch_number(p, s)) {
    return rc;
  }
  return launch_write(p, partial_masks_or_null, partial_bits_or_null, s);
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
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (const int rc = launch_classify(p, s)) return rc;
  if (const int rc = launch_number(p, s)) return rc;
  return launch_write(p, nullptr, nullptr, s);
}

extern "C" int omni_attn_mask_tiles_gfx950(const int64_t* spans_or_null, const int64_t* prefix_or_null,
                                           void* workspace, uint8_t* partial_masks, uint32_t* partial_bits_or_null,
                                           int num_partial, int B, int M, int H, int q_len, int kv_len, int QB, int KB,
                                           void* stream) {
  if (num_partial == 0) return OMNI_ATTN_OK;
  if ((!spans_or_null == !prefix_or_null) || !workspace || !partial_masks) return OMNI_ATTN_ERR_NULL_POINTER;
  if (const int rc = bad_shape(B, M, H, q_len, kv_len, QB, KB)) return rc;
  MaskParams p = common(spans_or_null, prefix_or_null, workspace, B, M, H, q_len, kv_len, QB, KB);
  if (const int rc = check_tiles(partial_masks, partial_bits_or_null, num_partial, p)) return rc;
  p.num_partial = num_partial;
  return launch_write(p, partial_masks, partial_bits_or_null, static_cast<hipStream_t>(stream));
}
