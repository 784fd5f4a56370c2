// Python module `omni_attn`: the operator surface the reference exports from
// omni-attn-mma/pybind/omni_attn.cc:70-77 (five functions, one 13-argument positional
// signature, :10-68), rebuilt over the gfx950 C ABI.  All five names run the same
// kernel; `omni_attn_preftech` is the name the reference's own wrapper tries to import
// (omni-attn-mma/omni_attn_torch.py:978), and `omni_attn_forward` additionally returns
// the row logsumexp.
//
// Host-only C++: the device code lives behind include/omni_attn_gfx950.h.
#include <torch/extension.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <stdexcept>
#include <string>
#include <vector>

#include "omni_attn_gfx950.h"
#include "omni_attn_host_counts.hpp"

namespace {

void check_qkvo(const torch::Tensor& t, const char* name, const torch::Tensor& q) {
  if (!t.is_cuda()) throw std::runtime_error(std::string(name) + " must be a GPU tensor");
  if (t.dim() != 4) throw std::runtime_error(std::string(name) + " must have shape [B, H, S, D]");
  if (t.scalar_type() != q.scalar_type())
    throw std::runtime_error(std::string("Tensor dtype mismatch: ") + name +
                             " must have the dtype of Q (torch.float16 or torch.bfloat16)");
  if (t.sizes() != q.sizes())
    throw std::runtime_error(std::string(name) + " must have the shape of Q");
  if (t.device() != q.device())
    throw std::runtime_error(std::string(name) + " must be on the device of Q");
}

void check_meta(const torch::Tensor& t, const char* name, const torch::Tensor& q) {
  if (t.scalar_type() != torch::kInt32)
    throw std::runtime_error(std::string("Tensor dtype mismatch: ") + name + " must be torch.int32");
  if (t.device() != q.device())
    throw std::runtime_error(std::string(name) + " must be on the device of Q");
}

void forward_impl(const torch::Tensor& Q, const torch::Tensor& K, const torch::Tensor& V,
                  torch::Tensor& O, float* lse, const torch::Tensor& kv_num_blocks,
                  const torch::Tensor& kv_indices, const torch::Tensor& block_mask_types,
                  int Q_BLOCK_SIZE, int KV_BLOCK_SIZE, int seqlen_orig,
                  const torch::Tensor& partial_block_mask_indices,
                  const torch::Tensor& partial_block_masks, bool has_partial, bool packed = false,
                  double softcap = 0.0, bool generic_fallback = false) {
  if (Q.scalar_type() != torch::kHalf && Q.scalar_type() != torch::kBFloat16)
    throw std::runtime_error("Tensor dtype mismatch: Q must be torch.float16 or torch.bfloat16");
  check_qkvo(Q, "Q", Q);
  check_qkvo(K, "K", Q);
  check_qkvo(V, "V", Q);
  check_qkvo(O, "O", Q);
  if (!Q.is_contiguous() || !K.is_contiguous() || !V.is_contiguous() || !O.is_contiguous())
    throw std::runtime_error(
        "Q, K, V, O tensors must be contiguous. Call .contiguous() before calling this function.");
  check_meta(kv_num_blocks, "kv_num_blocks", Q);
  check_meta(kv_indices, "kv_indices", Q);
  check_meta(block_mask_types, "block_mask_types", Q);
  if (!kv_num_blocks.is_contiguous() || !kv_indices.is_contiguous() ||
      !block_mask_types.is_contiguous())
    throw std::runtime_error(
        "Block mask tensors must be contiguous. Call .contiguous() before calling this function.");

  const int64_t B = Q.size(0), H = Q.size(1), S = Q.size(2), D = Q.size(3);
  if (kv_num_blocks.dim() != 3 || kv_indices.dim() != 4 || block_mask_types.dim() != 4)
    throw std::runtime_error(
        "kv_num_blocks must be [B, H, num_q_blocks]; kv_indices and block_mask_types "
        "[B, H, num_q_blocks, max_blocks]");
  const int64_t num_q_blocks = kv_num_blocks.size(2);
  const int64_t max_blocks = kv_indices.size(3);
  if (Q_BLOCK_SIZE <= 0 || KV_BLOCK_SIZE <= 0)
    throw std::runtime_error("Q_BLOCK_SIZE and KV_BLOCK_SIZE must be positive");
  const int64_t expected = (S + Q_BLOCK_SIZE - 1) / Q_BLOCK_SIZE;
  if (num_q_blocks != expected)
    throw std::runtime_error("Block mask num_q_blocks (" + std::to_string(num_q_blocks) +
                             ") does not match expected value (" + std::to_string(expected) +
                             ") based on seqlen=" + std::to_string(S) +
                             " and Q_BLOCK_SIZE=" + std::to_string(Q_BLOCK_SIZE));
  if (kv_num_blocks.size(0) != B || kv_num_blocks.size(1) != H || kv_indices.size(0) != B ||
      kv_indices.size(1) != H || kv_indices.size(2) != num_q_blocks ||
      block_mask_types.sizes() != kv_indices.sizes())
    throw std::runtime_error("Block mask tensor shapes do not match Q's batch / heads / blocks");

  const int32_t* pidx = nullptr;
  const uint8_t* pmask = nullptr;
  int num_partial = 0;
  if (has_partial) {
    if (partial_block_mask_indices.scalar_type() != torch::kInt32)
      throw std::runtime_error(
          "Tensor dtype mismatch: partial_block_mask_indices must be torch.int32");
    if (!packed && partial_block_masks.scalar_type() != torch::kBool)
      throw std::runtime_error("Tensor dtype mismatch: partial_block_masks must be torch.bool");
    if (packed && partial_block_masks.scalar_type() != torch::kInt32)
      throw std::runtime_error("Tensor dtype mismatch: packed partial tiles must be torch.int32");
    if (!partial_block_mask_indices.is_contiguous() || !partial_block_masks.is_contiguous())
      throw std::runtime_error("Partial block mask tensors must be contiguous.");
    if (partial_block_mask_indices.sizes() != kv_indices.sizes())
      throw std::runtime_error("partial_block_mask_indices must have the shape of kv_indices");
    if (partial_block_masks.dim() != 3 || partial_block_masks.size(1) != Q_BLOCK_SIZE ||
        partial_block_masks.size(2) != (packed ? KV_BLOCK_SIZE / 32 : KV_BLOCK_SIZE))
      throw std::runtime_error(
          packed ? "packed partial tiles must be [num_partial, Q_BLOCK_SIZE, KV_BLOCK_SIZE / 32]"
                 : "partial_block_masks must be [num_partial, Q_BLOCK_SIZE, KV_BLOCK_SIZE]");
    if (partial_block_mask_indices.device() != Q.device() ||
        partial_block_masks.device() != Q.device())
      throw std::runtime_error("Partial block mask tensors must be on the device of Q");
    if (partial_block_masks.size(0) > 0) {
      pidx = partial_block_mask_indices.data_ptr<int32_t>();
      pmask = static_cast<const uint8_t*>(partial_block_masks.data_ptr());
      num_partial = int(partial_block_masks.size(0));
    }
  }

  c10::DeviceGuard guard(Q.device());
  hipStream_t stream = c10::hip::getCurrentHIPStream(Q.device().index()).stream();
  const int dtype = Q.scalar_type() == torch::kBFloat16 ? OMNI_ATTN_DTYPE_BF16 : OMNI_ATTN_DTYPE_F16;
  // The scalar entry point of the reference takes any block size and any head_dim <= 256
  // (omni-attn-mma/mma/attn_naive.cu:189-190, :305-408): shapes without an MFMA instance go to
  // the generic kernel when the caller is that entry point.
  const bool has_instance = (D == 32 || D == 64 || D == 128) && (Q_BLOCK_SIZE == 64 || Q_BLOCK_SIZE == 128) &&
                            (KV_BLOCK_SIZE == 64 || KV_BLOCK_SIZE == 128);
  const int rc =
      (generic_fallback && !has_instance && !packed)
          ? omni_attn_fwd_generic_gfx950(
                Q.data_ptr(), K.data_ptr(), V.data_ptr(), O.data_ptr(), lse,
                kv_num_blocks.data_ptr<int32_t>(), kv_indices.data_ptr<int32_t>(),
                block_mask_types.data_ptr<int32_t>(), pidx, pmask, int(B), int(H), int(S), int(D),
                int(num_q_blocks), int(max_blocks), Q_BLOCK_SIZE, KV_BLOCK_SIZE, num_partial, seqlen_orig,
                dtype, float(softcap), static_cast<void*>(stream))
      : packed ? omni_attn_fwd_packed_gfx950(
                   Q.data_ptr(), K.data_ptr(), V.data_ptr(), O.data_ptr(), lse,
                   kv_num_blocks.data_ptr<int32_t>(), kv_indices.data_ptr<int32_t>(),
                   block_mask_types.data_ptr<int32_t>(), pidx, reinterpret_cast<const uint32_t*>(pmask),
                   int(B), int(H), int(S), int(D), int(num_q_blocks), int(max_blocks), Q_BLOCK_SIZE,
                   KV_BLOCK_SIZE, num_partial, seqlen_orig, dtype, float(softcap), static_cast<void*>(stream))
             : omni_attn_fwd_gfx950(
                   Q.data_ptr(), K.data_ptr(), V.data_ptr(), O.data_ptr(), lse,
                   kv_num_blocks.data_ptr<int32_t>(), kv_indices.data_ptr<int32_t>(),
                   block_mask_types.data_ptr<int32_t>(), pidx, pmask, int(B), int(H), int(S), int(D),
                   int(num_q_blocks), int(max_blocks), Q_BLOCK_SIZE, KV_BLOCK_SIZE, num_partial,
                   seqlen_orig, dtype, float(softcap), static_cast<void*>(stream));
  if (rc != OMNI_ATTN_OK) {
    std::string msg = std::string("omni_attn: ") + omni_attn_status_string(rc);
    if (rc == OMNI_ATTN_ERR_UNSUPPORTED_HEAD_DIM) msg += ", got head_dim=" + std::to_string(D);
    if (rc == OMNI_ATTN_ERR_UNSUPPORTED_BLOCK)
      msg += ", got Q_BLOCK_SIZE=" + std::to_string(Q_BLOCK_SIZE) +
             " KV_BLOCK_SIZE=" + std::to_string(KV_BLOCK_SIZE);
    if (rc == OMNI_ATTN_ERR_LAUNCH)
      msg += " (hipError " + std::to_string(omni_attn_last_hip_error()) + ")";
    throw std::runtime_error(msg);
  }
}

// The reference's signature: tensors by value, void return.
void omni_attn_op(torch::Tensor Q, torch::Tensor K, torch::Tensor V, torch::Tensor O,
                  torch::Tensor kv_num_blocks, torch::Tensor kv_indices,
                  torch::Tensor block_mask_types, int Q_BLOCK_SIZE, int KV_BLOCK_SIZE,
                  int seqlen_orig, torch::Tensor partial_block_mask_indices,
                  torch::Tensor partial_block_masks, bool has_partial) {
  forward_impl(Q, K, V, O, nullptr, kv_num_blocks, kv_indices, block_mask_types, Q_BLOCK_SIZE,
               KV_BLOCK_SIZE, seqlen_orig, partial_block_mask_indices, partial_block_masks,
               has_partial);
}

// omni_attn_simple_kernel: as above, and like the reference's scalar kernel for any Q_BLOCK_SIZE,
// KV_BLOCK_SIZE and head_dim <= 256.
void omni_attn_simple_op(torch::Tensor Q, torch::Tensor K, torch::Tensor V, torch::Tensor O,
                         torch::Tensor kv_num_blocks, torch::Tensor kv_indices,
                         torch::Tensor block_mask_types, int Q_BLOCK_SIZE, int KV_BLOCK_SIZE,
                         int seqlen_orig, torch::Tensor partial_block_mask_indices,
                         torch::Tensor partial_block_masks, bool has_partial) {
  forward_impl(Q, K, V, O, nullptr, kv_num_blocks, kv_indices, block_mask_types, Q_BLOCK_SIZE,
               KV_BLOCK_SIZE, seqlen_orig, partial_block_mask_indices, partial_block_masks,
               has_partial, false, 0.0, true);
}

// Same arguments plus LSE [B, H, S] fp32, written in place.
void omni_attn_forward(torch::Tensor Q, torch::Tensor K, torch::Tensor V, torch::Tensor O,
                       torch::Tensor LSE, torch::Tensor kv_num_blocks, torch::Tensor kv_indices,
                       torch::Tensor block_mask_types, int Q_BLOCK_SIZE, int KV_BLOCK_SIZE,
                       int seqlen_orig, torch::Tensor partial_block_mask_indices,
                       torch::Tensor partial_block_masks, bool has_partial, double softcap) {
  if (LSE.scalar_type() != torch::kFloat32)
    throw std::runtime_error("Tensor dtype mismatch: LSE must be torch.float32");
  if (!LSE.is_contiguous() || LSE.dim() != 3 || Q.dim() != 4 || LSE.size(0) != Q.size(0) ||
      LSE.size(1) != Q.size(1) || LSE.size(2) != Q.size(2) || LSE.device() != Q.device())
    throw std::runtime_error("LSE must be a contiguous [B, H, S] tensor on the device of Q");
  forward_impl(Q, K, V, O, LSE.data_ptr<float>(), kv_num_blocks, kv_indices, block_mask_types,
               Q_BLOCK_SIZE, KV_BLOCK_SIZE, seqlen_orig, partial_block_mask_indices,
               partial_block_masks, has_partial, false, softcap);
}

// PARTIAL tiles [P, QB, KB] bool -> [P, QB, KB / 32] int32 words, packed on the GPU.
torch::Tensor omni_attn_pack_partial_masks(torch::Tensor partial_block_masks) {
  if (!partial_block_masks.is_cuda() || partial_block_masks.scalar_type() != torch::kBool ||
      partial_block_masks.dim() != 3 || !partial_block_masks.is_contiguous())
    throw std::runtime_error("partial_block_masks must be a contiguous [P, Q_BLOCK_SIZE, KV_BLOCK_SIZE] bool GPU tensor");
  const int64_t P = partial_block_masks.size(0), QB = partial_block_masks.size(1), KB = partial_block_masks.size(2);
  if (KB % 32 != 0) throw std::runtime_error("KV_BLOCK_SIZE must be a multiple of 32");
  c10::DeviceGuard guard(partial_block_masks.device());
  torch::Tensor out = torch::empty({P, QB, KB / 32}, partial_block_masks.options().dtype(torch::kInt32));
  hipStream_t stream = c10::hip::getCurrentHIPStream(partial_block_masks.device().index()).stream();
  const int rc = omni_attn_pack_partial_masks_gfx950(
      static_cast<const uint8_t*>(partial_block_masks.data_ptr()),
      reinterpret_cast<uint32_t*>(out.data_ptr<int32_t>()), int(P), int(QB), int(KB), static_cast<void*>(stream));
  if (rc != OMNI_ATTN_OK) throw std::runtime_error(std::string("omni_attn: ") + omni_attn_status_string(rc));
  return out;
}

// omni_attn_forward with packed PARTIAL tiles; LSE may be an empty tensor (no logsumexp).
void omni_attn_forward_packed(torch::Tensor Q, torch::Tensor K, torch::Tensor V, torch::Tensor O,
                              torch::Tensor LSE, torch::Tensor kv_num_blocks, torch::Tensor kv_indices,
                              torch::Tensor block_mask_types, int Q_BLOCK_SIZE, int KV_BLOCK_SIZE,
                              int seqlen_orig, torch::Tensor partial_block_mask_indices,
                              torch::Tensor partial_block_bits, double softcap) {
  float* lse = nullptr;
  if (LSE.numel() > 0) {
    if (LSE.scalar_type() != torch::kFloat32)
      throw std::runtime_error("Tensor dtype mismatch: LSE must be torch.float32");
    if (!LSE.is_contiguous() || LSE.dim() != 3 || Q.dim() != 4 || LSE.size(0) != Q.size(0) ||
        LSE.size(1) != Q.size(1) || LSE.size(2) != Q.size(2) || LSE.device() != Q.device())
      throw std::runtime_error("LSE must be a contiguous [B, H, S] tensor on the device of Q");
    lse = LSE.data_ptr<float>();
  }
  forward_impl(Q, K, V, O, lse, kv_num_blocks, kv_indices, block_mask_types, Q_BLOCK_SIZE, KV_BLOCK_SIZE,
               seqlen_orig, partial_block_mask_indices, partial_block_bits, true, true, softcap);
}

// Backward of omni_attn_forward: dQ, dK, dV written in place (the reference exports no backward).
// PARTIAL tiles as bool bytes or, when `packed`, as the int32 words of omni_attn_pack_partial_masks.
void omni_attn_backward(torch::Tensor Q, torch::Tensor K, torch::Tensor V, torch::Tensor O,
                        torch::Tensor dO, torch::Tensor LSE, torch::Tensor dQ, torch::Tensor dK,
                        torch::Tensor dV, torch::Tensor kv_num_blocks, torch::Tensor kv_indices,
                        torch::Tensor block_mask_types, int Q_BLOCK_SIZE, int KV_BLOCK_SIZE,
                        int seqlen_orig, torch::Tensor partial_block_mask_indices,
                        torch::Tensor partial_tiles, bool has_partial, bool packed, double softcap) {
  if (Q.scalar_type() != torch::kHalf && Q.scalar_type() != torch::kBFloat16)
    throw std::runtime_error("Tensor dtype mismatch: Q must be torch.float16 or torch.bfloat16");
  check_qkvo(Q, "Q", Q);
  check_qkvo(K, "K", Q);
  check_qkvo(V, "V", Q);
  check_qkvo(O, "O", Q);
  check_qkvo(dO, "dO", Q);
  check_qkvo(dQ, "dQ", Q);
  check_qkvo(dK, "dK", Q);
  check_qkvo(dV, "dV", Q);
  for (const torch::Tensor* t : {&Q, &K, &V, &O, &dO, &dQ, &dK, &dV})
    if (!t->is_contiguous())
      throw std::runtime_error("Q, K, V, O, dO, dQ, dK, dV tensors must be contiguous.");
  check_meta(kv_num_blocks, "kv_num_blocks", Q);
  check_meta(kv_indices, "kv_indices", Q);
  check_meta(block_mask_types, "block_mask_types", Q);
  if (!kv_num_blocks.is_contiguous() || !kv_indices.is_contiguous() || !block_mask_types.is_contiguous())
    throw std::runtime_error("Block mask tensors must be contiguous.");
  const int64_t B = Q.size(0), H = Q.size(1), S = Q.size(2), D = Q.size(3);
  if (kv_num_blocks.dim() != 3 || kv_indices.dim() != 4 || block_mask_types.sizes() != kv_indices.sizes() ||
      kv_num_blocks.size(0) != B || kv_num_blocks.size(1) != H || kv_indices.size(0) != B ||
      kv_indices.size(1) != H || kv_indices.size(2) != kv_num_blocks.size(2))
    throw std::runtime_error("Block mask tensor shapes do not match Q's batch / heads / blocks");
  if (LSE.scalar_type() != torch::kFloat32 || !LSE.is_contiguous() || LSE.dim() != 3 || LSE.size(0) != B ||
      LSE.size(1) != H || LSE.size(2) != S || LSE.device() != Q.device())
    throw std::runtime_error("LSE must be the forward's contiguous fp32 [B, H, S] tensor on the device of Q");
  const int32_t* pidx = nullptr;
  const void* tiles = nullptr;
  int num_partial = 0;
  if (has_partial && partial_tiles.numel() > 0) {
    if (partial_block_mask_indices.scalar_type() != torch::kInt32 ||
        partial_block_mask_indices.sizes() != kv_indices.sizes() || !partial_block_mask_indices.is_contiguous() ||
        partial_block_mask_indices.device() != Q.device())
      throw std::runtime_error("partial_block_mask_indices must be a contiguous int32 tensor of the shape of kv_indices");
    if (partial_tiles.scalar_type() != (packed ? torch::kInt32 : torch::kBool) || partial_tiles.dim() != 3 ||
        partial_tiles.size(1) != Q_BLOCK_SIZE || partial_tiles.size(2) != (packed ? KV_BLOCK_SIZE / 32 : KV_BLOCK_SIZE) ||
        !partial_tiles.is_contiguous() || partial_tiles.device() != Q.device())
      throw std::runtime_error("partial tiles must be [num_partial, Q_BLOCK_SIZE, KV_BLOCK_SIZE] bool or packed int32 words");
    pidx = partial_block_mask_indices.data_ptr<int32_t>();
    tiles = partial_tiles.data_ptr();
    num_partial = int(partial_tiles.size(0));
  }
  c10::DeviceGuard guard(Q.device());
  hipStream_t stream = c10::hip::getCurrentHIPStream(Q.device().index()).stream();
  const size_t ws_bytes = omni_attn_bwd_workspace_bytes(int(B), int(H), int(S));
  torch::Tensor workspace = torch::empty({int64_t(ws_bytes)}, Q.options().dtype(torch::kUInt8));
  const int dtype = Q.scalar_type() == torch::kBFloat16 ? OMNI_ATTN_DTYPE_BF16 : OMNI_ATTN_DTYPE_F16;
  const int rc = omni_attn_bwd_gfx950(
      Q.data_ptr(), K.data_ptr(), V.data_ptr(), O.data_ptr(), dO.data_ptr(), LSE.data_ptr<float>(),
      dQ.data_ptr(), dK.data_ptr(), dV.data_ptr(), kv_num_blocks.data_ptr<int32_t>(),
      kv_indices.data_ptr<int32_t>(), block_mask_types.data_ptr<int32_t>(), pidx,
      packed ? nullptr : static_cast<const uint8_t*>(tiles), packed ? static_cast<const uint32_t*>(tiles) : nullptr,
      workspace.data_ptr(), ws_bytes, int(B), int(H), int(S), int(D), int(kv_num_blocks.size(2)),
      int(kv_indices.size(3)), Q_BLOCK_SIZE, KV_BLOCK_SIZE, num_partial, seqlen_orig, dtype, float(softcap),
      static_cast<void*>(stream));
  if (rc != OMNI_ATTN_OK) {
    std::string msg = std::string("omni_attn: ") + omni_attn_status_string(rc);
    if (rc == OMNI_ATTN_ERR_LAUNCH) msg += " (hipError " + std::to_string(omni_attn_last_hip_error()) + ")";
    throw std::runtime_error(msg);
  }
}

struct PinnedWords {
  typedef hipStream_t Stream;
  static void* allocate(size_t bytes) {
    void* mem = nullptr;
    // (portable: memory taken under one device is handed to calls on any)
    const hipError_t e = hipHostMalloc(&mem, bytes, hipHostMallocPortable | hipHostMallocMapped);
    if (e != hipSuccess) throw std::runtime_error(std::string("omni_attn: hipHostMalloc: ") + hipGetErrorString(e));
    return mem;
  }
  static void release(void* memory) { (void)hipHostFree(memory); }
  static bool running(hipStream_t stream) {
    const hipError_t e = hipStreamQuery(stream);
    if (e != hipSuccess && e != hipErrorNotReady)
      throw std::runtime_error(std::string("omni_attn: the mask was not built: ") + hipGetErrorString(e));
    return e == hipErrorNotReady;
  }
  static bool drain(hipStream_t stream) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(stream, &capture) == hipSuccess && capture == hipStreamCaptureStatusNone &&
           hipStreamSynchronize(stream) == hipSuccess;
  }
};
typedef omni_attn::HostCounts<PinnedWords, OMNI_ATTN_MASK_POSTED_COUNT_BITS> HostCounts;

// ---- the operator as one call -----------------------------------------------------------------
// What the wrappers of omni_attn_torch.py do per call, in one native call: look the operands and the
// mask over, allocate the results, launch.  Operands are read at their strides and at their own
// length.  The functions return None for anything out of the ordinary (a mask on another device or
// of other types, sizes that do not fit, an unsupported shape): the wrapper's general path then
// converts, pads or raises.

struct MaskArgs {
  torch::Tensor nb, idx, types, pidx, tiles;  // pidx, tiles: undefined when there are none
  int64_t q_len, kv_len, QB, KB;
  bool packed;
};

int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

bool has_instance(int64_t D, int64_t QB, int64_t KB) {
  return (D == 32 || D == 64 || D == 128) && (QB == 64 || QB == 128) && (KB == 64 || KB == 128);
}

bool plain_meta(const torch::Tensor& t, const torch::Tensor& q) {
  return t.scalar_type() == torch::kInt32 && t.device() == q.device() && t.is_contiguous();
}

// Operands and mask as the kernels take them?
bool ordinary(const torch::Tensor& q, const torch::Tensor& k, const torch::Tensor& v, const MaskArgs& m, bool generic) {
  if (!q.is_cuda() || q.dim() != 4 || (q.scalar_type() != torch::kHalf && q.scalar_type() != torch::kBFloat16)) return false;
  if (k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type() || k.device() != q.device() ||
      v.device() != q.device() || k.sizes() != q.sizes() || v.sizes() != q.sizes() || q.numel() == 0)
    return false;
  const int64_t B = q.size(0), H = q.size(1), S = q.size(2), D = q.size(3);
  if (m.QB <= 0 || m.KB <= 0 || S > 0x3fffffff || round_up(S, m.QB) != m.q_len || round_up(S, m.KB) != m.kv_len ||
      m.kv_len > m.q_len)
    return false;
  if (!has_instance(D, m.QB, m.KB) && !(generic && D <= 256 && !m.packed && m.QB < 0x3fffffff && m.KB < 0x3fffffff))
    return false;
  const int64_t Tq = m.q_len / m.QB;
  if (!plain_meta(m.nb, q) || !plain_meta(m.idx, q) || !plain_meta(m.types, q) || m.nb.dim() != 3 ||
      m.nb.size(0) != B || m.nb.size(1) != H || m.nb.size(2) != Tq || m.idx.dim() != 4 || m.idx.size(0) != B ||
      m.idx.size(1) != H || m.idx.size(2) != Tq || m.types.sizes() != m.idx.sizes())
    return false;
  if (m.tiles.defined()) {
    if (!plain_meta(m.pidx, q) || m.pidx.sizes() != m.idx.sizes() || m.tiles.dim() != 3 ||
        m.tiles.scalar_type() != (m.packed ? torch::kInt32 : torch::kBool) || m.tiles.device() != q.device() ||
        !m.tiles.is_contiguous() || m.tiles.size(1) != m.QB || m.tiles.size(2) != (m.packed ? m.KB / 32 : m.KB))
      return false;
  }
  return true;
}

omni_attn_strides strides_of(const torch::Tensor& t) { return {t.stride(0), t.stride(1), t.stride(2)}; }

// Rows the matrix-core kernels can read in place (16-byte loads, 32-bit byte offsets in a slab)?
bool readable(const torch::Tensor& t, int64_t rows) {
  return t.stride(3) == 1 && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 && t.stride(2) % 8 == 0 &&
         t.stride(2) >= t.size(3) && rows * t.stride(2) * 2 <= 0xffffffffLL &&
         (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
}
torch::Tensor in_rows(const torch::Tensor& t, int64_t rows, bool generic) {
  if (generic ? t.stride(3) == 1 : readable(t, rows)) return t;
  // (clone: contiguous() would return a contiguous but misaligned tensor as it is)
  return t.clone(at::MemoryFormat::Contiguous);
}

[[noreturn]] void fail(int rc) {
  std::string msg = std::string("omni_attn: ") + omni_attn_status_string(rc);
  if (rc == OMNI_ATTN_ERR_LAUNCH) msg += " (hipError " + std::to_string(omni_attn_last_hip_error()) + ")";
  throw std::runtime_error(msg);
}

struct Tiles {
  const int32_t* pidx = nullptr;
  const uint8_t* bytes = nullptr;
  const uint32_t* bits = nullptr;
  int n = 0;
  explicit Tiles(const MaskArgs& m) {
    if (!m.tiles.defined() || m.tiles.size(0) == 0) return;
    pidx = m.pidx.data_ptr<int32_t>();
    n = int(m.tiles.size(0));
    if (m.packed) {
      bits = reinterpret_cast<const uint32_t*>(m.tiles.data_ptr<int32_t>());
    } else {
      bytes = static_cast<const uint8_t*>(m.tiles.data_ptr());
    }
  }
};

int dtype_of(const torch::Tensor& q) {
  return q.scalar_type() == torch::kBFloat16 ? OMNI_ATTN_DTYPE_BF16 : OMNI_ATTN_DTYPE_F16;
}
void* stream_of(const torch::Tensor& q) {
  return static_cast<void*>(c10::hip::getCurrentHIPStream(q.device().index()).stream());
}

// q, k and v become the tensors the kernel has read (copies where it could not read them in place).
torch::Tensor launch_forward(torch::Tensor& q, torch::Tensor& k, torch::Tensor& v, const MaskArgs& m, double softcap,
                             torch::Tensor* lse) {
  const int64_t B = q.size(0), H = q.size(1), S = q.size(2), D = q.size(3);
  const bool generic = !has_instance(D, m.QB, m.KB);
  q = in_rows(q, m.q_len + m.KB, generic);
  k = in_rows(k, m.q_len + m.KB, generic);
  v = in_rows(v, m.q_len + m.KB, generic);
  if (!generic && k.stride(2) != v.stride(2)) {  // one row stride for both (clones: of one row any stride is contiguous)
    k = k.clone(at::MemoryFormat::Contiguous);
    v = v.clone(at::MemoryFormat::Contiguous);
  }
  torch::Tensor out = torch::empty({B, H, S, D}, q.options());
  if (lse) *lse = torch::empty({B, H, S}, q.options().dtype(torch::kFloat32));
  const Tiles t(m);
  const int rc = omni_attn_fwd_strided_gfx950(
      q.data_ptr(), k.data_ptr(), v.data_ptr(), strides_of(q), strides_of(k), strides_of(v), out.data_ptr(),
      lse ? lse->data_ptr<float>() : nullptr, m.nb.data_ptr<int32_t>(), m.idx.data_ptr<int32_t>(),
      m.types.data_ptr<int32_t>(), t.pidx, t.bytes, t.bits, int(B), int(H), int(m.q_len), int(S), int(D),
      int(m.q_len / m.QB), int(m.idx.size(3)), int(m.QB), int(m.KB), t.n, int(S), dtype_of(q), float(softcap), generic,
      stream_of(q));
  if (rc != OMNI_ATTN_OK) fail(rc);
  return out;
}

MaskArgs mask_args(torch::Tensor nb, torch::Tensor idx, torch::Tensor types, int64_t q_len, int64_t kv_len, int64_t QB,
                   int64_t KB, c10::optional<torch::Tensor> pidx, c10::optional<torch::Tensor> tiles, bool packed) {
  MaskArgs m;
  m.nb = std::move(nb);
  m.idx = std::move(idx);
  m.types = std::move(types);
  m.q_len = q_len;
  m.kv_len = kv_len;
  m.QB = QB;
  m.KB = KB;
  m.packed = packed;
  if (pidx && tiles) {
    m.pidx = std::move(*pidx);
    m.tiles = std::move(*tiles);
  }
  return m;
}

// The output, or (output, logsumexp) with `want_lse`.  `any_shape`: the entry point takes any block
// size and head_dim <= 256.
pybind11::object omni_attn_attend(torch::Tensor q, torch::Tensor k, torch::Tensor v, torch::Tensor nb,
                                  torch::Tensor idx, torch::Tensor types, int64_t q_len, int64_t kv_len, int64_t QB,
                                  int64_t KB, c10::optional<torch::Tensor> pidx, c10::optional<torch::Tensor> tiles,
                                  bool packed, bool want_lse, double softcap, bool any_shape) {
  const MaskArgs m = mask_args(std::move(nb), std::move(idx), std::move(types), q_len, kv_len, QB, KB, std::move(pidx),
                               std::move(tiles), packed);
  if (!ordinary(q, k, v, m, any_shape)) return pybind11::none();
  c10::DeviceGuard guard(q.device());
  at::NoGradGuard no_grad;
  torch::Tensor lse;
  torch::Tensor out = launch_forward(q, k, v, m, softcap, want_lse ? &lse : nullptr);
  if (want_lse) return pybind11::make_tuple(std::move(out), std::move(lse));
  return pybind11::cast(std::move(out));
}

// Forward and backward kernels as one differentiable operator.
class AttendFunction : public torch::autograd::Function<AttendFunction> {
 public:
  static torch::Tensor forward(torch::autograd::AutogradContext* ctx, torch::Tensor q, torch::Tensor k,
                               torch::Tensor v, const MaskArgs& m, double softcap) {
    torch::Tensor lse;
    torch::Tensor out = launch_forward(q, k, v, m, softcap, &lse);
    ctx->save_for_backward({q, k, v, out, lse});
    std::vector<torch::Tensor> meta = {m.nb, m.idx, m.types};
    if (m.tiles.defined()) {
      meta.push_back(m.pidx);
      meta.push_back(m.tiles);
    }
    ctx->saved_data["mask"] = std::move(meta);
    ctx->saved_data["sizes"] = std::vector<int64_t>{m.q_len, m.kv_len, m.QB, m.KB, int64_t(m.packed)};
    ctx->saved_data["softcap"] = softcap;
    return out;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const torch::Tensor &q = saved[0], &k = saved[1], &v = saved[2], &out = saved[3], &lse = saved[4];
    const std::vector<torch::Tensor> meta = ctx->saved_data["mask"].toTensorVector();
    const std::vector<int64_t> sizes = ctx->saved_data["sizes"].toIntVector();
    MaskArgs m;
    m.nb = meta[0];
    m.idx = meta[1];
    m.types = meta[2];
    if (meta.size() > 3) {
      m.pidx = meta[3];
      m.tiles = meta[4];
    }
    m.q_len = sizes[0];
    m.kv_len = sizes[1];
    m.QB = sizes[2];
    m.KB = sizes[3];
    m.packed = sizes[4] != 0;
    const int64_t B = q.size(0), H = q.size(1), S = q.size(2), D = q.size(3);
    c10::DeviceGuard guard(q.device());
    torch::Tensor dout = grads[0];
    if (dout.scalar_type() != q.scalar_type()) dout = dout.to(q.scalar_type());
    dout = in_rows(dout, m.q_len + std::max(m.QB, m.KB), false);
    torch::Tensor dq = torch::empty({B, H, S, D}, q.options()), dk = torch::empty({B, H, S, D}, q.options()),
                  dv = torch::empty({B, H, S, D}, q.options());
    const size_t ws_bytes = omni_attn_bwd_workspace_bytes(int(B), int(H), int(S));
    torch::Tensor workspace = torch::empty({int64_t(ws_bytes / 4)}, lse.options());
    const Tiles t(m);
    const int rc = omni_attn_bwd_strided_gfx950(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), dout.data_ptr(), strides_of(q), strides_of(k), strides_of(v),
        strides_of(dout), out.data_ptr(), lse.data_ptr<float>(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
        m.nb.data_ptr<int32_t>(), m.idx.data_ptr<int32_t>(), m.types.data_ptr<int32_t>(), t.pidx, t.bytes, t.bits,
        workspace.data_ptr<float>(), ws_bytes, int(B), int(H), int(m.q_len), int(S), int(D), int(m.q_len / m.QB),
        int(m.idx.size(3)), int(m.QB), int(m.KB), t.n, int(S), dtype_of(q),
        float(ctx->saved_data["softcap"].toDouble()), stream_of(q));
    if (rc != OMNI_ATTN_OK) fail(rc);
    return {dq, dk, dv, torch::Tensor(), torch::Tensor()};
  }
};

pybind11::object omni_attn_attend_autograd(torch::Tensor q, torch::Tensor k, torch::Tensor v, torch::Tensor nb,
                                           torch::Tensor idx, torch::Tensor types, int64_t q_len, int64_t kv_len,
                                           int64_t QB, int64_t KB, c10::optional<torch::Tensor> pidx,
                                           c10::optional<torch::Tensor> tiles, bool packed, double softcap) {
  const MaskArgs m = mask_args(std::move(nb), std::move(idx), std::move(types), q_len, kv_len, QB, KB, std::move(pidx),
                               std::move(tiles), packed);
  if (!ordinary(q, k, v, m, false)) return pybind11::none();
  c10::DeviceGuard guard(q.device());
  return pybind11::cast(AttendFunction::apply(q, k, v, m, softcap));
}

// The block mask of a prefix rule: `source` is [B, M, 3] spans or [B, q_len] prefix lengths, int64 on
// the GPU.  Returns (kv_num_blocks, kv_indices, block_mask_types, partial_block_mask_indices,
// partial_block_masks, partial_block_bits); the last three None where no block is PARTIAL, the
// last one also without `pack`.
pybind11::tuple omni_attn_build_prefix_mask(torch::Tensor source, bool spans, int64_t H, int64_t q_len, int64_t kv_len,
                                            int64_t QB, int64_t KB, bool pack) {
  namespace py = pybind11;
  if (!source.is_cuda() || source.scalar_type() != torch::kInt64 || !source.is_contiguous() ||
      source.dim() != (spans ? 3 : 2) || source.size(1) > 0x7fffffff || (spans && source.size(2) != 3) ||
      (!spans && source.size(1) != q_len))
    throw std::runtime_error("the mask source must be a contiguous int64 GPU tensor: spans [B, M, 3] or prefix lengths [B, q_len]");
  const int64_t B = source.size(0);
  const int64_t M = spans ? source.size(1) : 0;
  c10::DeviceGuard guard(source.device());
  const hipStream_t stream = c10::hip::getCurrentHIPStream(source.device().index()).stream();
  const size_t ws_bytes = omni_attn_mask_workspace_bytes(int(B), int(q_len), int(kv_len), int(QB), int(KB));
  if (ws_bytes == 0) throw std::runtime_error("omni_attn: the block mask's sizes are not positive or too large");
  const int64_t Tq = (q_len + QB - 1) / QB, Tk = (kv_len + KB - 1) / KB;
  const auto i32 = source.options().dtype(torch::kInt32);
  torch::Tensor workspace = torch::empty({int64_t(ws_bytes / 4)}, i32);
  // (a span pointer of an empty [B, 0, 3] tensor may be null: any address, nothing is read through it)
  const int64_t* src = source.numel() > 0 ? source.data_ptr<int64_t>()
                                          : reinterpret_cast<const int64_t*>(workspace.data_ptr<int32_t>());
  const int64_t* sp = spans ? src : nullptr;
  const int64_t* prefix = spans ? nullptr : src;
  const auto refuse = [](int rc) {
    if (rc != OMNI_ATTN_OK) throw std::runtime_error(std::string("omni_attn: ") + omni_attn_status_string(rc));
  };
  int* const ws = workspace.data_ptr<int32_t>();
  torch::Tensor nb, idx, types, pidx, tiles, bits;
  const auto allocate_lists = [&] {
    nb = torch::empty({B, H, Tq}, i32);
    idx = torch::empty({B, H, Tq, Tk}, i32);
    types = torch::empty({B, H, Tq, Tk}, i32);
    pidx = torch::empty({B, H, Tq, Tk}, i32);
  };
  const auto allocate_tiles = [&](int64_t P) {
    if (P > 0x7fffffff) refuse(OMNI_ATTN_ERR_TOO_LARGE);
    if (P == 0) return;
    tiles = torch::empty({P, QB, KB}, source.options().dtype(torch::kBool));
    if (pack) bits = torch::empty({P, QB, KB / 32}, i32);
  };
  const auto tile_bytes = [&] { return tiles.defined() ? static_cast<uint8_t*>(tiles.data_ptr()) : nullptr; };
  const auto tile_words = [&] {
    return bits.defined() ? reinterpret_cast<uint32_t*>(bits.data_ptr<int32_t>()) : nullptr;
  };
  void* const at = static_cast<void*>(stream);
  {
    py::gil_scoped_release release;
    HostCounts counts;
    const int tag = counts.next_tag(stream);
    if (B * Tq <= HostCounts::kWords && (Tk >> OMNI_ATTN_MASK_POSTED_COUNT_BITS) == 0) {
      // The first kernel needs the workspace only, and sends its counts as they are known: the lists are allocated
      // while it runs.
      refuse(omni_attn_mask_classify_gfx950(sp, prefix, ws, counts.memory(), tag, int(B), int(M), int(q_len), int(kv_len),
                                            int(QB), int(KB), at));
      allocate_lists();
      allocate_tiles(counts.wait(tag, int(B * Tq)));
      refuse(omni_attn_mask_finish_gfx950(nb.data_ptr<int32_t>(), idx.data_ptr<int32_t>(), types.data_ptr<int32_t>(),
                                          pidx.data_ptr<int32_t>(), ws, tile_bytes(), tile_words(),
                                          tiles.defined() ? int(tiles.size(0)) : 0, int(B), int(H), int(q_len),
                                          int(kv_len), int(QB), int(KB), at));
    } else {
      allocate_lists();
      refuse(omni_attn_mask_lists_gfx950(sp, prefix, nb.data_ptr<int32_t>(), idx.data_ptr<int32_t>(),
                                         types.data_ptr<int32_t>(), pidx.data_ptr<int32_t>(), ws,
                                         reinterpret_cast<int32_t*>(counts.memory()), HostCounts::word_of(tag), int(B),
                                         int(M), int(H), int(q_len), int(kv_len), int(QB), int(KB), at));
      allocate_tiles(counts.wait_total(tag));
      if (tiles.defined())
        refuse(omni_attn_mask_tiles_gfx950(sp, prefix, ws, tile_bytes(), tile_words(), int(tiles.size(0)), int(B), int(M),
                                           int(H), int(q_len), int(kv_len), int(QB), int(KB), at));
    }
  }
  if (!tiles.defined()) return py::make_tuple(nb, idx, types, py::none(), py::none(), py::none());
  return py::make_tuple(nb, idx, types, pidx, tiles, pack ? py::cast(bits) : py::object(py::none()));
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "gfx950 block-sparse FlashAttention-2 forward (omni-attention operator surface)";
  m.def("omni_attn_mma_stages_split_q_shared_kv", &omni_attn_op,
        "omni_attn_mma_stages_split_q_shared_kv");
  m.def("omni_attn_simple_kernel", &omni_attn_simple_op, "omni_attn_simple_kernel");
  m.def("omni_attn_cp_async", &omni_attn_op, "omni_attn_cp_async");
  m.def("omni_attn_preftech_kernel", &omni_attn_op, "omni_attn_preftech_kernel");
  m.def("omni_attn_preftech", &omni_attn_op, "omni_attn_preftech");
  m.def("omni_attn_mma_stages_split_q_shared_kv_swizzle", &omni_attn_op,
        "omni_attn_mma_stages_split_q_shared_kv_swizzle");
  namespace py = pybind11;
  m.def("omni_attn_forward", &omni_attn_forward, "omni_attn_forward (also writes logsumexp)", py::arg("Q"),
        py::arg("K"), py::arg("V"), py::arg("O"), py::arg("LSE"), py::arg("kv_num_blocks"), py::arg("kv_indices"),
        py::arg("block_mask_types"), py::arg("Q_BLOCK_SIZE"), py::arg("KV_BLOCK_SIZE"), py::arg("seqlen_orig"),
        py::arg("partial_block_mask_indices"), py::arg("partial_block_masks"), py::arg("has_partial"),
        py::arg("softcap") = 0.0);
  m.def("omni_attn_pack_partial_masks", &omni_attn_pack_partial_masks,
        "omni_attn_pack_partial_masks (bool tiles -> 32-bit words)");
  m.def("omni_attn_forward_packed", &omni_attn_forward_packed,
        "omni_attn_forward_packed (PARTIAL tiles as packed words)", py::arg("Q"), py::arg("K"), py::arg("V"),
        py::arg("O"), py::arg("LSE"), py::arg("kv_num_blocks"), py::arg("kv_indices"), py::arg("block_mask_types"),
        py::arg("Q_BLOCK_SIZE"), py::arg("KV_BLOCK_SIZE"), py::arg("seqlen_orig"),
        py::arg("partial_block_mask_indices"), py::arg("partial_block_bits"), py::arg("softcap") = 0.0);
  m.def("omni_attn_backward", &omni_attn_backward, "omni_attn_backward (dQ, dK, dV of omni_attn_forward)",
        py::arg("Q"), py::arg("K"), py::arg("V"), py::arg("O"), py::arg("dO"), py::arg("LSE"), py::arg("dQ"),
        py::arg("dK"), py::arg("dV"), py::arg("kv_num_blocks"), py::arg("kv_indices"), py::arg("block_mask_types"),
        py::arg("Q_BLOCK_SIZE"), py::arg("KV_BLOCK_SIZE"), py::arg("seqlen_orig"),
        py::arg("partial_block_mask_indices"), py::arg("partial_tiles"), py::arg("has_partial"), py::arg("packed"),
        py::arg("softcap") = 0.0);
  m.def("omni_attn_attend", &omni_attn_attend, "omni_attn_attend (the operator as one call)");
  m.def("omni_attn_attend_autograd", &omni_attn_attend_autograd, "omni_attn_attend_autograd (differentiable)");
  m.def("omni_attn_build_prefix_mask", &omni_attn_build_prefix_mask,
        "omni_attn_build_prefix_mask (block mask of spans or prefix lengths)");
  m.def("abi_version", []() { return omni_attn_abi_version(); });
}
