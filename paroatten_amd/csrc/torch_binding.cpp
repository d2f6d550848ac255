// PyTorch-ROCm C++ extension over the C ABI of libparoatten_hip.so (include/paroatten.h).
//
// Host code only: no kernels here.  It registers, under one extension module, three submodules with the
// names, positional signatures, preallocated-output conventions and error behaviour of the reference's
// three CUDA extensions:
//   _qattn_sm80  csrc/qattn/pybind_sm80.cpp:21-27, csrc/qattn/attn_cuda_sm80.h:19-69
//   _fused       csrc/fused/pybind.cpp:21-33,      csrc/fused/fused.h:19-76
//   _rope        csrc/rope/pybind.cpp:5-8,         csrc/rope/rope.h:6
// and a fourth, _ops, which the package's own Python layer calls: whole operators with their argument checks,
// allocations and launches (a call of a few hundred tokens is bound by this host work: 85 us a call at 416 tokens from
// Python over eight launches).
// Checks fail as the reference's do: TORCH_CHECK -> RuntimeError with the texts of csrc/utils.cuh:20-38,
// std::invalid_argument -> ValueError for unsupported layouts, head dims and flags
// (csrc/dispatch_utils.h:23-112).  Unlike the reference's launches (legacy default stream, no device
// guard: paroattention/core.py:168-174 works around it) every call runs under a guard for the tensors'
// device and on torch's current stream of that device.
#include <torch/extension.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <atomic>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include <stdexcept>
#include <string>

#include "../../include/paroatten.h"

namespace {

// NotImplementedError in Python.  An exception of C++, translated once the call has the interpreter lock again: the entry
// points of _ops run without it.
struct Unsupported : std::runtime_error {
  using std::runtime_error::runtime_error;
};

void check_rc(int rc) {
  if (rc == PARO_OK) return;
  const std::string msg = paro_last_error();
  if (rc == PARO_ERR_INVALID_VALUE) throw std::invalid_argument(msg);
  if (rc == PARO_ERR_UNSUPPORTED) throw Unsupported(msg);
  TORCH_CHECK(false, msg);
}

void on_gpu(const torch::Tensor& x, const char* name) { TORCH_CHECK(x.is_cuda(), "Tensor ", name, " must be on CUDA"); }
void contiguous(const torch::Tensor& x, const char* name) { TORCH_CHECK(x.is_contiguous(), "Tensor ", name, " must be contiguous"); }
void lastdim_contiguous(const torch::Tensor& x, const char* name) {
  TORCH_CHECK(x.stride(-1) == 1, "Tensor ", name, " must be contiguous at the last dimension");
}
void dims(const torch::Tensor& x, const char* name, int64_t n) {
  TORCH_CHECK(x.dim() == n, "Tensor ", name, " must have dimension number (", n, ")");
}
void dtype(const torch::Tensor& x, const char* name, at::ScalarType t, const char* tname) {
  TORCH_CHECK(x.scalar_type() == t, "Tensor ", name, " must have dtype (", tname, ")");
}
void shape(const torch::Tensor& x, const char* name, at::IntArrayRef want, const char* text) {
  TORCH_CHECK(x.sizes() == want, "Tensor ", name, " must have shape (", text, ")");
}
int half_code(const torch::Tensor& x, const char* fn) {
  if (x.scalar_type() == at::kHalf) return PARO_DTYPE_F16;
  if (x.scalar_type() == at::kBFloat16) return PARO_DTYPE_BF16;
  TORCH_CHECK(false, fn, " failed to dispatch data type ", x.scalar_type());
  return -1;
}
void* stream_of(const torch::Tensor& x) { return c10::hip::getCurrentHIPStream(x.device().index()).stream(); }

struct Layout { int64_t n_tokens, n_heads, stride_n, stride_h; };
Layout layout_of(const torch::Tensor& x, int tensor_layout) {
  if (tensor_layout == 0) return {x.size(1), x.size(2), x.stride(1), x.stride(2)};
  return {x.size(2), x.size(1), x.stride(2), x.stride(1)};
}

// ---- _qattn_sm80 ------------------------------------------------------------------------------------
// The reference's positional signature has no room for this library's attention flags (PARO_ATTN_* of
// include/paroatten.h: exact exponentials, the float16 P.V product, launch forms).  A process-wide default,
// set_attention_flags(), lets a caller of the compiled module choose them; 0 = the library's defaults.
static std::atomic<int> g_attention_flags{0};
void set_attention_flags(int flags) { g_attention_flags.store(flags); }
int get_attention_flags() { return g_attention_flags.load(); }

torch::Tensor qk_int8_sv_f16_accum_f16_attn(torch::Tensor query, torch::Tensor key, torch::Tensor value,
                                            torch::Tensor output, torch::Tensor query_scale,
                                            torch::Tensor key_scale, int tensor_layout, int is_causal,
                                            int qk_quant_gran, float sm_scale, int return_lse,
                                            torch::Tensor sparse) {
  on_gpu(query, "query"); on_gpu(key, "key"); on_gpu(value, "value"); on_gpu(output, "output");
  on_gpu(query_scale, "query_scale"); on_gpu(key_scale, "key_scale");
  contiguous(query, "query"); contiguous(key, "key");
  lastdim_contiguous(value, "value"); lastdim_contiguous(output, "output");
  contiguous(query_scale, "query_scale"); contiguous(key_scale, "key_scale");
  dtype(query, "query", at::kChar, "torch::kInt8"); dtype(key, "key", at::kChar, "torch::kInt8");
  // the reference takes float16 only; bfloat16 saves the caller's conversion
  TORCH_CHECK(value.scalar_type() == at::kHalf || value.scalar_type() == at::kBFloat16,
              "Tensor value must have dtype (torch::kHalf)");
  dtype(query_scale, "query_scale", at::kFloat, "torch::kFloat32");
  dtype(key_scale, "key_scale", at::kFloat, "torch::kFloat32");
  dims(query, "query", 4); dims(key, "key", 4); dims(value, "value", 4); dims(output, "output", 4);
  dims(query_scale, "query_scale", 3); dims(key_scale, "key_scale", 3);
  if (tensor_layout != 0 && tensor_layout != 1) throw std::invalid_argument("tensor_layout must be 0 or 1");
  const int sn = tensor_layout == 0 ? 1 : 2, sh = tensor_layout == 0 ? 2 : 1;
  const int64_t B = query.size(0), D = query.size(3), H = query.size(sh), Hkv = key.size(sh), Nq = query.size(sn),
                Nk = key.size(sn);
  if (tensor_layout == 0) {
    shape(key, "key", {B, Nk, Hkv, D}, "batch_size, kv_len, num_kv_heads, head_dim");
    shape(value, "value", {B, Nk, Hkv, D}, "batch_size, kv_len, num_kv_heads, head_dim");
  } else {
    shape(key, "key", {B, Hkv, Nk, D}, "batch_size, num_kv_heads, kv_len, head_dim");
    shape(value, "value", {B, Hkv, Nk, D}, "batch_size, num_kv_heads, kv_len, head_dim");
  }
  if (Hkv == 0 || H % Hkv != 0)
    throw std::invalid_argument("num_qo_heads (" + std::to_string(H) + ") must be divisible by num_kv_heads (" +
                                std::to_string(Hkv) + ")");
  if (D != 64 && D != 128) throw std::invalid_argument("Unsupported head dim: " + std::to_string(D));
  if (return_lse != 0 && return_lse != 1)
    throw std::invalid_argument("Unsupported causal mode: " + std::to_string(return_lse));   // sic, as the reference words it
  const int out_code = half_code(output, "qk_int8_sv_f16_accum_f16_attn");
  TORCH_CHECK(output.sizes() == query.sizes(), "Tensor output must have the shape of query");
  const int64_t nbq = (Nq + 63) / 64, nbk = (Nk + 63) / 64;
  if (qk_quant_gran == 2) {
    shape(query_scale, "query_scale", {B, H, nbq * 2},
          "batch_size, num_qo_heads, div_ceil(qo_len, CTA_Q) * (CTA_Q / WARP_Q)");
    shape(key_scale, "key_scale", {B, Hkv, nbk}, "batch_size, num_kv_heads, div_ceil(kv_len, CTA_K) * (CTA_K / WARP_K)");
  } else if (qk_quant_gran == 3) {   // per thread (csrc/qattn/qk_int_sv_f16_cuda_sm80.cu:1034-1038)
    shape(query_scale, "query_scale", {B, H, nbq * 2 * 8},
          "batch_size, num_qo_heads, div_ceil(qo_len, CTA_Q) * (CTA_Q / WARP_Q) * 8");
    shape(key_scale, "key_scale", {B, Hkv, nbk * 4},
          "batch_size, num_kv_heads, div_ceil(kv_len, CTA_K) * (CTA_K / WARP_K) * 4");
  }
  // the reference reads `sparse` through a raw pointer without any check
  on_gpu(sparse, "sparse"); contiguous(sparse, "sparse");
  TORCH_CHECK(sparse.scalar_type() == at::kBool || sparse.scalar_type() == at::kByte,
              "Tensor sparse must have dtype (torch::kBool)");
  int64_t sparse_bs = 0;
  if (sparse.dim() == 4) {
    shape(sparse, "sparse", {B, H, nbq, nbk}, "batch_size, num_qo_heads, num_q_blocks, num_k_blocks");
    sparse_bs = sparse.stride(0);
  } else {
    dims(sparse, "sparse", 3);
    shape(sparse, "sparse", {H, nbq, nbk}, "num_qo_heads, num_q_blocks, num_k_blocks");
  }
  const c10::DeviceGuard guard(query.device());
  torch::Tensor lse = torch::empty({0});
  if (return_lse) lse = torch::empty({B, H, Nq}, query.options().dtype(at::kFloat));
  const int flags = g_attention_flags.load();
  const int64_t ws_bytes = paro_attn_workspace_bytes_for((int)B, (int)Hkv, (int)Nk, (int)D, flags);
  torch::Tensor ws = torch::empty({ws_bytes}, query.options().dtype(at::kByte));
  check_rc(paro_qk_int8_sv_f16_attn(
      query.data_ptr<int8_t>(), key.data_ptr<int8_t>(), value.data_ptr(), half_code(value, "qk_int8_sv_f16_accum_f16_attn"),
      output.data_ptr(), out_code, query_scale.data_ptr<float>(), key_scale.data_ptr<float>(),
      static_cast<const uint8_t*>(sparse.data_ptr()), sparse_bs, return_lse ? lse.data_ptr<float>() : nullptr,
      ws.data_ptr(), ws_bytes, (int)B, (int)H, (int)Hkv, (int)Nq, (int)Nk, (int)D, query.stride(0), query.stride(sh),
      query.stride(sn), key.stride(0), key.stride(sh), key.stride(sn), value.stride(0), value.stride(sh), value.stride(sn),
      output.stride(0), output.stride(sh), output.stride(sn), tensor_layout, is_causal, qk_quant_gran, sm_scale,
      /*smooth_v=*/1, flags, stream_of(query)));
  return lse;
}

torch::Tensor prototype_variant(torch::Tensor, torch::Tensor, torch::Tensor, torch::Tensor, torch::Tensor, torch::Tensor,
                                int, int, int, float, int, torch::Tensor) {
  throw Unsupported("experimental variant of the reference (INT4 Q/K or INT8 P.V) without a working caller; "
                    "use qk_int8_sv_f16_accum_f16_attn");
}

// ---- _fused -----------------------------------------------------------------------------------------
void quant_int8(const char* fn, torch::Tensor input, const torch::Tensor* mean, torch::Tensor output, torch::Tensor scale,
                int group, int64_t groups_per_block, int block_size, int tensor_layout, bool has_sm_scale,
                float sm_scale) {
  on_gpu(input, "input"); on_gpu(output, "output"); on_gpu(scale, "scale");
  if (mean) on_gpu(*mean, "mean");
  dtype(output, "output", at::kChar, "torch::kInt8"); dtype(scale, "scale", at::kFloat, "torch::kFloat");
  dims(input, "input", 4);
  lastdim_contiguous(input, "input"); contiguous(output, "output"); contiguous(scale, "scale");
  dims(output, "output", 4); dims(scale, "scale", 3);
  if (mean) { lastdim_contiguous(*mean, "mean"); dims(*mean, "mean", 3); }
  const int code = half_code(input, fn);
  if (mean) TORCH_CHECK(mean->scalar_type() == input.scalar_type(), "Tensor mean must have dtype (input_dtype)");
  const int64_t B = input.size(0), D = input.size(3);
  const Layout in = layout_of(input, tensor_layout), out = layout_of(output, tensor_layout);
  if (block_size != 64 && block_size != 128) throw std::invalid_argument("Unsupported block_size " + std::to_string(block_size));
  if (D != 64 && D != 128) throw std::invalid_argument("Unsupported head dim: " + std::to_string(D));
  const int64_t n_groups = (in.n_tokens + block_size - 1) / block_size * groups_per_block;
  TORCH_CHECK(output.sizes() == input.sizes(),
              "Tensor output must have shape (input.size(0), input.size(1), input.size(2), input.size(3))");
  shape(scale, "scale", {B, in.n_heads, n_groups}, "batch_size, num_heads, num_groups");
  if (mean) shape(*mean, "mean", {B, in.n_heads, D}, "batch_size, num_heads, head_dim");
  const c10::DeviceGuard guard(input.device());
  check_rc(paro_quant_int8(input.data_ptr(), code, mean ? mean->data_ptr() : nullptr, output.data_ptr<int8_t>(),
                           scale.data_ptr<float>(), (int)B, (int)in.n_heads, (int)in.n_tokens, (int)D, input.stride(0),
                           in.stride_h, in.stride_n, mean ? mean->stride(0) : 0, mean ? mean->stride(1) : 0,
                           output.stride(0), out.stride_h, out.stride_n, scale.stride(0), scale.stride(1), group,
                           (int)n_groups, has_sm_scale ? 1 : 0, sm_scale, stream_of(input)));
}

void quant_per_block_int8_cuda_sm(torch::Tensor input, torch::Tensor output, torch::Tensor scale, float sm_scale,
                                  int block_size, int tensor_layout) {
  quant_int8("quant_per_block_int8_cuda", input, nullptr, output, scale, block_size, 1, block_size, tensor_layout, true, sm_scale);
}
void quant_per_block_int8_cuda(torch::Tensor input, torch::Tensor output, torch::Tensor scale, int block_size,
                               int tensor_layout) {
  quant_int8("quant_per_block_int8_cuda", input, nullptr, output, scale, block_size, 1, block_size, tensor_layout, false, 0.f);
}
void quant_per_block_int8_fuse_sub_mean_cuda(torch::Tensor input, torch::Tensor mean, torch::Tensor output,
                                             torch::Tensor scale, int block_size, int tensor_layout) {
  quant_int8("quant_per_block_int8_fuse_sub_mean_cuda", input, &mean, output, scale, block_size, 1, block_size,
             tensor_layout, false, 0.f);
}
void quant_per_warp_int8_cuda(torch::Tensor input, torch::Tensor output, torch::Tensor scale, int block_size,
                              int warp_block_size, int tensor_layout) {
  if (block_size != 64 && block_size != 128) throw std::invalid_argument("Unsupported block_size " + std::to_string(block_size));
  if (warp_block_size != 16 && warp_block_size != 32)
    throw std::invalid_argument("Unsupported warp_block_size " + std::to_string(warp_block_size));
  quant_int8("quant_per_warp_int8_cuda", input, nullptr, output, scale, warp_block_size, block_size / warp_block_size,
             block_size, tensor_layout, false, 0.f);
}

void sub_mean_cuda(torch::Tensor input, torch::Tensor mean, torch::Tensor output, int tensor_layout) {
  on_gpu(input, "input"); on_gpu(mean, "mean"); on_gpu(output, "output");
  dtype(output, "output", at::kHalf, "torch::kHalf");
  dims(input, "input", 4); dims(mean, "mean", 3); dims(output, "output", 4);
  lastdim_contiguous(input, "input"); lastdim_contiguous(mean, "mean"); lastdim_contiguous(output, "output");
  const int code = half_code(input, "sub_mean_cuda");
  TORCH_CHECK(mean.scalar_type() == input.scalar_type(), "Tensor mean must have dtype (input_dtype)");
  const int64_t B = input.size(0), D = input.size(3);
  const Layout in = layout_of(input, tensor_layout), out = layout_of(output, tensor_layout);
  shape(mean, "mean", {B, in.n_heads, D}, "batch_size, num_heads, head_dim");
  TORCH_CHECK(output.sizes() == input.sizes(),
              "Tensor output must have shape (input.size(0), input.size(1), input.size(2), input.size(3))");
  const c10::DeviceGuard guard(input.device());
  check_rc(paro_sub_mean(input.data_ptr(), code, mean.data_ptr(), output.data_ptr(), (int)B, (int)in.n_heads,
                         (int)in.n_tokens, (int)D, input.stride(0), in.stride_h, in.stride_n, mean.stride(0),
                         mean.stride(1), output.stride(0), out.stride_h, out.stride_n, stream_of(input)));
}

void transpose_pad_permute_cuda(torch::Tensor input, torch::Tensor output, int tensor_layout) {
  on_gpu(input, "input"); on_gpu(output, "output");
  lastdim_contiguous(input, "input"); contiguous(output, "output");
  dims(input, "input", 4); dims(output, "output", 4);
  const int64_t B = input.size(0), D = input.size(3);
  const Layout in = layout_of(input, tensor_layout);
  const int64_t padded = (in.n_tokens + 63) / 64 * 64;
  int64_t os_d, os_h;
  if (tensor_layout == 0) {
    shape(output, "output", {B, D, in.n_heads, padded}, "batch_size, head_dim, num_heads, padded_num_tokens");
    os_d = output.stride(1); os_h = output.stride(2);
  } else {
    shape(output, "output", {B, in.n_heads, D, padded}, "batch_size, num_heads, head_dim, padded_num_tokens");
    os_d = output.stride(2); os_h = output.stride(1);
  }
  TORCH_CHECK(input.scalar_type() == output.scalar_type(), "Input and output must have the same data type");
  const int code = half_code(input, "transpose_pad_permute_cuda");
  if (D != 64 && D != 128) throw std::invalid_argument("Unsupported head dim: " + std::to_string(D));
  const c10::DeviceGuard guard(input.device());
  check_rc(paro_transpose_pad_permute(input.data_ptr(), output.data_ptr(), code, (int)B, (int)in.n_heads, (int)in.n_tokens,
                                      (int)D, input.stride(0), in.stride_h, in.stride_n, output.stride(0), os_h, os_d,
                                      stream_of(input)));
}

void channel_quant(const char* fn, torch::Tensor input, torch::Tensor output, const torch::Tensor* mean, torch::Tensor scale,
                   int num_tokens, float scale_max, int tensor_layout) {
  on_gpu(input, "input"); on_gpu(output, "output");
  if (mean) on_gpu(*mean, "mean");
  on_gpu(scale, "scale");
  if (mean) dtype(*mean, "mean", at::kFloat, "torch::kFloat");
  dtype(scale, "scale", at::kFloat, "torch::kFloat");
  contiguous(input, "input"); contiguous(output, "output");
  if (mean) contiguous(*mean, "mean");
  contiguous(scale, "scale");
  dims(input, "input", 4); dims(output, "output", 4);
  if (mean) dims(*mean, "mean", 3);
  dims(scale, "scale", 3);
  const int64_t B = input.size(0), row_len = input.size(3);
  const int d_dim = tensor_layout == 0 ? 1 : 2, h_dim = tensor_layout == 0 ? 2 : 1;
  const int64_t H = input.size(h_dim), D = input.size(d_dim);
  TORCH_CHECK(output.sizes() == input.sizes(),
              "Tensor output must have shape (input.size(0), input.size(1), input.size(2), input.size(3))");
  if (mean) shape(*mean, "mean", {B, H, D}, "batch_size, num_heads, head_dim");
  shape(scale, "scale", {B, H, D}, "batch_size, num_heads, head_dim");
  const int code = half_code(input, fn);
  TORCH_CHECK(output.element_size() == 1, "Tensor output must have a one-byte dtype (torch.float8_e4m3fn)");
  const c10::DeviceGuard guard(input.device());
  check_rc(paro_channel_quant_fp8(input.data_ptr(), code, static_cast<uint8_t*>(output.data_ptr()),
                                  mean ? mean->data_ptr<float>() : nullptr, scale.data_ptr<float>(), (int)B, (int)H, (int)D,
                                  num_tokens, (int)row_len, scale_max, input.stride(0), input.stride(h_dim),
                                  input.stride(d_dim), output.stride(0), output.stride(h_dim), output.stride(d_dim),
                                  mean ? mean->stride(0) : 0, mean ? mean->stride(1) : 0, scale.stride(0), scale.stride(1),
                                  stream_of(input)));
}
void scale_fuse_quant_cuda(torch::Tensor input, torch::Tensor output, torch::Tensor scale, int num_tokens, float scale_max,
                           int tensor_layout) {
  channel_quant("scale_fuse_quant_cuda", input, output, nullptr, scale, num_tokens, scale_max, tensor_layout);
}
void mean_scale_fuse_quant_cuda(torch::Tensor input, torch::Tensor output, torch::Tensor mean, torch::Tensor scale,
                                int num_tokens, float scale_max, int tensor_layout) {
  channel_quant("mean_scale_fuse_quant_cuda", input, output, &mean, scale, num_tokens, scale_max, tensor_layout);
}

// ---- _rope ------------------------------------------------------------------------------------------
// rope_permutation(Q, K, freq, permutation) -> (QO, KO): Q, K float16 [bs, H, W, dim]; freq float32 [128]
// of (cos, sin) pairs shared by every token and every 128-channel slice; with `permutation` the (H, W) grid
// is written transposed.  The reference's permuting kernel overwrites its inputs and leaves its outputs
// uninitialised (csrc/rope/rope.cuh:49-50); here the inputs stay and the outputs hold the result.
std::vector<torch::Tensor> rope_permutation(torch::Tensor Q, torch::Tensor K, torch::Tensor freq, bool permutation) {
  on_gpu(Q, "Q"); on_gpu(K, "K"); on_gpu(freq, "freq");
  TORCH_CHECK(Q.scalar_type() == at::kHalf && K.scalar_type() == at::kHalf, "expected scalar type Half");
  TORCH_CHECK(freq.scalar_type() == at::kFloat && freq.numel() == 128, "freq must be float32 with 128 entries");
  TORCH_CHECK(Q.dim() == 4 && Q.sizes() == K.sizes() && Q.is_contiguous() && K.is_contiguous(),
              "Q and K must be contiguous [bs, H, W, dim] tensors of the same shape");
  const int64_t bs = Q.size(0), H = Q.size(1), W = Q.size(2), dim = Q.size(3);
  if (dim % 128 != 0) throw std::invalid_argument("Unsupported head dim: " + std::to_string(dim) + " (must be a multiple of 128)");
  const int64_t heads = dim / 128, n = H * W;
  const c10::DeviceGuard guard(Q.device());
  auto cs = freq.view({64, 2});
  auto cos = cs.select(1, 0).repeat_interleave(2).expand({n, 128}).contiguous();
  auto sin = cs.select(1, 1).repeat_interleave(2).expand({n, 128}).contiguous();
  auto orders = torch::full({heads}, permutation ? 1 : 0, Q.options().dtype(at::kInt));
  auto QO = torch::empty({bs, n, dim}, Q.options()), KO = torch::empty({bs, n, dim}, Q.options());
  // [bs, n, heads, 128] seen as (batch, head, token, channel) through strides
  check_rc(paro_rope_permute_fwd(Q.data_ptr(), K.data_ptr(), nullptr, QO.data_ptr(), KO.data_ptr(), nullptr, PARO_DTYPE_F16,
                                 cos.data_ptr<float>(), sin.data_ptr<float>(), orders.data_ptr<int32_t>(), (int)bs, (int)heads,
                                 (int)n, 128, 0, 1, (int)H, (int)W, n * dim, 128, dim, n * dim, 128, dim, stream_of(Q)));
  return {QO, KO};
}

// ---- _ops ---------------------------------------------------------------------------------------------
// the block mask: bool or byte [B,H,nbq,nbk], or [H,nbq,nbk] shared by the batch; returns its batch stride
int64_t check_mask(const torch::Tensor& sparse, int64_t B, int64_t H, int64_t nbq, int64_t nbk) {
  on_gpu(sparse, "sparse");
  TORCH_CHECK(sparse.scalar_type() == at::kBool || sparse.scalar_type() == at::kByte,
              "Tensor sparse must have dtype (torch::kBool)");
  contiguous(sparse, "sparse");
  if (sparse.dim() == 4) {
    TORCH_CHECK(sparse.sizes() == at::IntArrayRef({B, H, nbq, nbk}), "Tensor sparse must have shape (batch_size, num_qo_heads, ",
                nbq, ", ", nbk, "), got ", sparse.sizes());
    return sparse.stride(0);
  }
  TORCH_CHECK(sparse.dim() == 3 && sparse.sizes() == at::IntArrayRef({H, nbq, nbk}),
              "Tensor sparse must have shape ([batch_size,] num_qo_heads, ", nbq, ", ", nbk, "), got ", sparse.sizes());
  return 0;
}

// core.paroattn_qk_int8_pv_fp16_cuda behind its assertions: q, k, v of one 16-bit dtype on one GPU, head size 64 or 128.
// Returns the output, or (output, log-sum-exp).
py::object attn_operator(torch::Tensor q, torch::Tensor k, torch::Tensor v, torch::Tensor sparse, int tensor_layout,
                         bool is_causal, int qk_quant_gran, double sm_scale, bool return_lse, bool smooth_k, bool smooth_v,
                         int flags) {
  dims(q, "query", 4); dims(k, "key", 4); dims(v, "value", 4);
  const int sn = tensor_layout == 0 ? 1 : 2, sh = tensor_layout == 0 ? 2 : 1;
  const int64_t B = q.size(0), D = q.size(3), H = q.size(sh), Hkv = k.size(sh), Nq = q.size(sn), Nk = k.size(sn);
  if (D != 64 && D != 128) throw std::invalid_argument("Unsupported head dim: " + std::to_string(D));
  TORCH_CHECK(k.size(0) == B && k.size(3) == D, "Tensor key must have the batch size and head dim of query");
  TORCH_CHECK(v.sizes() == k.sizes(), "Tensor value must have the shape of key");
  if (Hkv == 0 || H % Hkv != 0)
    throw std::invalid_argument("num_qo_heads (" + std::to_string(H) + ") must be divisible by num_kv_heads (" +
                                std::to_string(Hkv) + ")");
  const int64_t sparse_bs = check_mask(sparse, B, H, (Nq + 63) / 64, (Nk + 63) / 64);
  torch::Tensor out, lse;
  {
    const py::gil_scoped_release unlocked;   // the launches wait while the queue is full: not with the interpreter lock
    const c10::DeviceGuard guard(q.device());
    out = torch::empty(q.sizes(), q.options());
    if (return_lse) lse = torch::empty({B, H, Nq}, q.options().dtype(at::kFloat));
    const int64_t ws_bytes = paro_attn_operator_workspace_bytes((int)B, (int)H, (int)Hkv, (int)Nq, (int)Nk, (int)D, smooth_k,
                                                                return_lse, qk_quant_gran, flags);
    torch::Tensor ws = torch::empty({ws_bytes}, q.options().dtype(at::kByte));
    check_rc(paro_attn_operator(q.data_ptr(), k.data_ptr(), v.data_ptr(), half_code(q, "paroattn"), out.data_ptr(),
                                static_cast<const uint8_t*>(sparse.data_ptr()), sparse_bs,
                                return_lse ? lse.data_ptr<float>() : nullptr, ws.data_ptr(), ws_bytes, (int)B, (int)H, (int)Hkv,
                                (int)Nq, (int)Nk, (int)D, q.stride(0), q.stride(sh), q.stride(sn), k.stride(0), k.stride(sh),
                                k.stride(sn), v.stride(0), v.stride(sh), v.stride(sn), out.stride(0), out.stride(sh),
                                out.stride(sn), is_causal, qk_quant_gran, (float)sm_scale, smooth_k, smooth_v, flags,
                                stream_of(q)));
  }
  if (return_lse) return py::make_tuple(out, lse);
  return py::cast(out);
}

using OptTensor = c10::optional<torch::Tensor>;

void hnd(const torch::Tensor& x, const char* name) {
  TORCH_CHECK(x.is_cuda(), "Tensor ", name, " must be a CUDA tensor");
  dims(x, name, 4);
  TORCH_CHECK(x.scalar_type() == at::kHalf || x.scalar_type() == at::kBFloat16, "Tensor ", name, " must be float16 or bfloat16");
  lastdim_contiguous(x, name);
}
int code_of(const torch::Tensor& x) { return x.scalar_type() == at::kHalf ? PARO_DTYPE_F16 : PARO_DTYPE_BF16; }

void check_orders(const torch::Tensor& orders, int64_t H) {
  TORCH_CHECK(orders.is_cuda(), "Tensor orders must be a CUDA tensor");
  TORCH_CHECK(orders.scalar_type() == at::kInt && orders.dim() == 1 && orders.numel() == H && orders.is_contiguous(),
              "orders must be a contiguous int32 tensor of ", H, " entries (one per head)");
}

struct Tables { const float *cos, *sin; };
Tables check_tables(const OptTensor& cos, const OptTensor& sin, int64_t n_img, int64_t D) {
  if (!cos) return {nullptr, nullptr};
  TORCH_CHECK(sin, "cos and sin must be given together");
  auto one = [&](const torch::Tensor& t, const char* name) {
    TORCH_CHECK(t.is_cuda(), "Tensor ", name, " must be a CUDA tensor");
    TORCH_CHECK(t.scalar_type() == at::kFloat && t.dim() == 2 && t.size(0) == n_img && t.size(1) == D && t.is_contiguous(),
                "Tensor ", name, " must be contiguous float32 of shape (", n_img, ", ", D, ")");
    return t.data_ptr<float>();
  };
  return {one(*cos, "cos"), one(*sin, "sin")};
}

// permute.rope_permute
std::vector<OptTensor> rope_permute(const OptTensor& q, const OptTensor& k, const OptTensor& v, const torch::Tensor& orders,
                                    int F, int Hh, int W, int n_text, const OptTensor& cos, const OptTensor& sin) {
  const OptTensor* in[3] = {&q, &k, &v};
  const torch::Tensor* ref = nullptr;
  for (auto* t : in)
    if (*t) {
      hnd(**t, "input");
      if (!ref) ref = &**t;
      TORCH_CHECK((*t)->sizes() == ref->sizes() && (*t)->strides() == ref->strides() && (*t)->scalar_type() == ref->scalar_type(),
                  "q, k, v must share shape, strides and dtype");
    }
  TORCH_CHECK(ref, "one of q, k, v must be given");
  const int64_t B = ref->size(0), H = ref->size(1), N = ref->size(2), D = ref->size(3);
  check_orders(orders, H);
  const Tables tab = check_tables(cos, sin, (int64_t)F * Hh * W, D);
  const c10::DeviceGuard guard(ref->device());
  std::vector<OptTensor> out(3);
  void *src[3] = {}, *dst[3] = {};
  for (int i = 0; i < 3; i++)
    if (*in[i]) {
      out[i] = torch::empty({B, H, N, D}, ref->options());
      src[i] = (*in[i])->data_ptr();
      dst[i] = out[i]->data_ptr();
    }
  check_rc(paro_rope_permute_fwd(src[0], src[1], src[2], dst[0], dst[1], dst[2], code_of(*ref), tab.cos, tab.sin,
                                 orders.data_ptr<int32_t>(), (int)B, (int)H, (int)N, (int)D, n_text, F, Hh, W, ref->stride(0),
                                 ref->stride(1), ref->stride(2), H * N * D, N * D, D, stream_of(*ref)));
  return out;
}

// permute.permute_inverse
torch::Tensor permute_inverse(const torch::Tensor& o, const torch::Tensor& orders, int F, int Hh, int W, int n_text,
                              const OptTensor& out_) {
  hnd(o, "attn_out");
  const int64_t B = o.size(0), H = o.size(1), N = o.size(2), D = o.size(3);
  check_orders(orders, H);
  const c10::DeviceGuard guard(o.device());
  torch::Tensor out;
  if (out_) {
    out = *out_;
    hnd(out, "out");
    TORCH_CHECK(out.sizes() == o.sizes() && out.scalar_type() == o.scalar_type() && out.device() == o.device(),
                "out must have attn_out's shape, dtype and device");
  } else {
    out = torch::empty({B, H, N, D}, o.options());
  }
  check_rc(paro_permute_inv(o.data_ptr(), out.data_ptr(), code_of(o), orders.data_ptr<int32_t>(), (int)B, (int)H, (int)N, (int)D,
                            n_text, F, Hh, W, o.stride(0), o.stride(1), o.stride(2), out.stride(0), out.stride(1),
                            out.stride(2), stream_of(o)));
  return out;
}

// permute.rope_permute_quant: (q8, q_scale, k8, k_scale, v8, v_scale, v_mean or None, k_mean or None).  km: a K mean that is
// subtracted; compute_km: it is taken in the call.
std::vector<OptTensor> rope_permute_quant(const torch::Tensor& q, const torch::Tensor& k, const torch::Tensor& v,
                                          const torch::Tensor& orders, int F, int Hh, int W, int n_text, const OptTensor& cos,
                                          const OptTensor& sin, OptTensor km, bool compute_km, bool smooth_v) {
  hnd(q, "query");
  hnd(k, "key");
  hnd(v, "value");
  TORCH_CHECK(k.sizes() == q.sizes() && v.sizes() == q.sizes() && k.scalar_type() == q.scalar_type() &&
                  v.scalar_type() == q.scalar_type(),
              "q, k, v must share shape and dtype");
  const int64_t B = q.size(0), H = q.size(1), N = q.size(2), D = q.size(3), nb = (N + 63) / 64;
  check_orders(orders, H);
  const Tables tab = check_tables(cos, sin, (int64_t)F * Hh * W, D);
  const c10::DeviceGuard guard(q.device());
  if (compute_km) km = torch::empty({B, H, 1, D}, q.options());
  if (km) {
    TORCH_CHECK(km->is_cuda(), "Tensor km must be a CUDA tensor");
    TORCH_CHECK(km->scalar_type() == q.scalar_type() && km->sizes() == at::IntArrayRef({B, H, 1, D}) && km->stride(-1) == 1,
                "Tensor km must have shape (", B, ", ", H, ", 1, ", D, ") and the dtype of key");
  }
  const auto i8 = q.options().dtype(at::kChar), u8 = q.options().dtype(at::kByte), f32 = q.options().dtype(at::kFloat);
  torch::Tensor q8 = torch::empty({B, H, N, D}, i8), k8 = torch::empty({B, H, N, D}, i8);
  torch::Tensor q_scale = torch::empty({B, H, nb * 2}, f32), k_scale = torch::empty({B, H, nb}, f32);
  torch::Tensor v8 = torch::empty({paro_v_fp8_bytes((int)B, (int)H, (int)N, (int)D)}, u8);
  torch::Tensor v_scale = torch::empty({B, H, D}, f32), v_mean = torch::empty({B, H, D}, f32);
  const int64_t ws_bytes = compute_km ? paro_prep_smooth_workspace_bytes((int)B, (int)H, (int)N, (int)D)
                                      : paro_prep_workspace_bytes((int)B, (int)H, (int)N, (int)D);
  torch::Tensor ws = torch::empty({ws_bytes}, u8);
  auto call = [&](auto entry) {
    check_rc(entry(q.data_ptr(), k.data_ptr(), v.data_ptr(), code_of(q), tab.cos, tab.sin, orders.data_ptr<int32_t>(),
                   km ? km->data_ptr() : nullptr, q8.data_ptr<int8_t>(), q_scale.data_ptr<float>(), k8.data_ptr<int8_t>(),
                   k_scale.data_ptr<float>(), v8.data_ptr<uint8_t>(), v_scale.data_ptr<float>(), v_mean.data_ptr<float>(),
                   ws.data_ptr(), ws_bytes, (int)B, (int)H, (int)N, (int)D, n_text, F, Hh, W, q.stride(0), q.stride(1),
                   q.stride(2), k.stride(0), k.stride(1), k.stride(2), v.stride(0), v.stride(1), v.stride(2),
                   km ? km->stride(0) : 0, km ? km->stride(1) : 0, smooth_v ? 1 : 0, stream_of(q)));
  };
  if (compute_km) call(&paro_rope_k_mean_permute_quant_fwd);
  else call(&paro_rope_permute_quant_fwd);
  return {q8, q_scale, k8, k_scale, v8, v_scale, smooth_v ? OptTensor(v_mean) : c10::nullopt, compute_km ? km : c10::nullopt};
}

// cogvideox._head_norms: the LayerNorms over the channels of q and k, [B,H,N,D] views of token-major projections, in one launch;
// nothing where the library's own modules have to do it (another type, size or order of rows, or something that
// records or rewrites the operation: autograd in either direction, autocast, a tracer, a mode, a dispatching subclass; the
// subclasses that a tensor's Python type alone tells stay with the caller).
std::vector<torch::Tensor> head_norm(const torch::Tensor& q, const torch::Tensor& k, const OptTensor& q_weight,
                                     const OptTensor& q_bias, double q_eps, const OptTensor& k_weight, const OptTensor& k_bias,
                                     double k_eps) {
  const bool grad = at::GradMode::is_enabled();
  auto plain = [&](const torch::Tensor& x) {
    return x.is_cuda() && x.device() == q.device() && x.scalar_type() == q.scalar_type() && !(grad && x.requires_grad()) &&
           !x.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                                     c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                                     c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor})) &&
           !x._fw_grad(0).defined();   // (a tangent rides on the tensor, with gradients off too)
  };
  if ((q.scalar_type() != at::kHalf && q.scalar_type() != at::kBFloat16) || q.dim() != 4 || !plain(q) || !plain(k)) return {};
  const int64_t B = q.size(0), H = q.size(1), N = q.size(2), D = q.size(3);
  if ((D != 64 && D != 128) || q.numel() == 0 || k.sizes() != q.sizes()) return {};
  for (const OptTensor* w : {&q_weight, &q_bias, &k_weight, &k_bias})
    if (*w && (!plain(**w) || (*w)->dim() != 1 || (*w)->size(0) != D || !(*w)->is_contiguous() || (uintptr_t)(*w)->data_ptr() % 16 != 0))
      return {};
  const torch::Tensor q_rows = q.transpose(1, 2), k_rows = k.transpose(1, 2);
  if (!q_rows.is_contiguous() || !k_rows.is_contiguous() || ((uintptr_t)q.data_ptr() | (uintptr_t)k.data_ptr()) % 16 != 0 ||
      at::autocast::is_autocast_enabled(at::kCUDA) || torch::jit::tracer::isTracing() ||
      c10::impl::TorchDispatchModeTLS::stack_len() > 0 || at::impl::PythonTorchFunctionTLS::stack_len() > 0)
    return {};
  const c10::DeviceGuard guard(q.device());
  torch::Tensor qo = torch::empty({B, N, H, D}, q.options()), ko = torch::empty({B, N, H, D}, q.options());
  auto at_ = [](const OptTensor& w) -> const void* { return w ? w->data_ptr() : nullptr; };
  check_rc(paro_head_norm(q.data_ptr(), k.data_ptr(), qo.data_ptr(), ko.data_ptr(), code_of(q), at_(q_weight), at_(q_bias),
                          at_(k_weight), at_(k_bias), (float)q_eps, (float)k_eps, B * N * H, (int)D, stream_of(q)));
  return {qo.transpose(1, 2), ko.transpose(1, 2)};
}

// _qattn_sm80.attn_sparse_prepacked; unpermute: orders with (F, Hh, W) and n_text, or none
torch::Tensor attn_sparse_prepacked(const torch::Tensor& q8, const torch::Tensor& k8, const torch::Tensor& v8,
                                    const OptTensor& v_scale, const OptTensor& v_mean, const torch::Tensor& output,
                                    const torch::Tensor& q_scale, const torch::Tensor& k_scale, double sm_scale,
                                    const torch::Tensor& sparse, int is_causal, bool return_lse, int flags,
                                    const OptTensor& orders, int F, int Hh, int W, int n_text) {
  const bool pv16 = (flags & PARO_ATTN_PV_F16) != 0;
  auto gpu = [](const torch::Tensor& x, const char* name, bool contig) {
    on_gpu(x, name);
    if (contig) contiguous(x, name);
  };
  gpu(q8, "query", true); gpu(k8, "key", true); gpu(v8, "value", true); gpu(output, "output", false);
  gpu(q_scale, "query_scale", true); gpu(k_scale, "key_scale", true);
  TORCH_CHECK(v_scale || pv16, "Tensor v_scale must be given");
  if (v_scale) gpu(*v_scale, "v_scale", true);
  gpu(sparse, "sparse", true);
  TORCH_CHECK(q8.scalar_type() == at::kChar && k8.scalar_type() == at::kChar, "Tensor query/key must have dtype (torch::kInt8)");
  TORCH_CHECK(q8.dim() == 4 && k8.dim() == 4, "Tensor query/key must have dimension number (4)");
  const int64_t B = q8.size(0), H = q8.size(1), Nq = q8.size(2), D = q8.size(3), Hkv = k8.size(1), Nk = k8.size(2);
  if (D != 64 && D != 128) throw std::invalid_argument("Unsupported head dim: " + std::to_string(D));
  TORCH_CHECK(k8.size(0) == B && k8.size(3) == D, "Tensor key must have the batch size and head dim of query");
  if (Hkv == 0 || H % Hkv != 0)
    throw std::invalid_argument("num_qo_heads (" + std::to_string(H) + ") must be divisible by num_kv_heads (" +
                                std::to_string(Hkv) + ")");
  const int64_t nbq = (Nq + 63) / 64, nbk = (Nk + 63) / 64;
  TORCH_CHECK((int64_t)v8.nbytes() == (pv16 ? paro_v_f16_bytes((int)B, (int)Hkv, (int)Nk, (int)D)
                                            : paro_v_fp8_bytes((int)B, (int)Hkv, (int)Nk, (int)D)),
              "Tensor value has the wrong size for ", pv16 ? "float16" : "FP8", " tiles");
  TORCH_CHECK(q_scale.scalar_type() == at::kFloat && k_scale.scalar_type() == at::kFloat &&
                  q_scale.sizes() == at::IntArrayRef({B, H, nbq * 2}) && k_scale.sizes() == at::IntArrayRef({B, Hkv, nbk}),
              "Tensor query_scale / key_scale must have shapes (B, H, 2*nbq) / (B, Hkv, nbk)");
  const std::vector<int64_t> vs = {B, Hkv, D};
  TORCH_CHECK((!v_scale || (v_scale->sizes() == at::IntArrayRef(vs) && v_scale->scalar_type() == at::kFloat)) &&
                  (!v_mean || (v_mean->sizes() == at::IntArrayRef(vs) && v_mean->scalar_type() == at::kFloat && v_mean->is_cuda())),
              "Tensor v_scale / v_mean must have shape (B, Hkv, head_dim)");
  TORCH_CHECK(output.sizes() == at::IntArrayRef({B, H, Nq, D}) && output.stride(-1) == 1 &&
                  (output.scalar_type() == at::kHalf || output.scalar_type() == at::kBFloat16),
              "Tensor output must be float16/bfloat16 [B,H,N,D] with a contiguous last dimension");
  const int64_t sparse_bs = check_mask(sparse, B, H, nbq, nbk);
  const c10::DeviceGuard guard(q8.device());
  torch::Tensor lse = return_lse ? torch::empty({B, H, Nq}, q8.options().dtype(at::kFloat)) : torch::empty({0});
  float* lse_p = return_lse ? lse.data_ptr<float>() : nullptr;
  const float* vsp = v_scale ? v_scale->data_ptr<float>() : nullptr;
  const float* vmp = v_mean ? v_mean->data_ptr<float>() : nullptr;
  const uint8_t* mask = static_cast<const uint8_t*>(sparse.data_ptr());
  if (orders)
    TORCH_CHECK(orders->is_cuda() && orders->scalar_type() == at::kInt && orders->dim() == 1 && orders->numel() == H &&
                    orders->is_contiguous(),
                "orders must be a contiguous int32 GPU tensor of ", H, " entries");
  const int64_t n_scratch =
      paro_attn_scratch_bytes((int)B, (int)H, (int)Nq, (int)Nk, (int)D, is_causal, return_lse, flags);
  torch::Tensor scratch;
  if (n_scratch > 0) scratch = torch::empty({n_scratch}, q8.options().dtype(at::kByte));
  check_rc(paro_attn_sparse_scratch_fwd(
      q8.data_ptr<int8_t>(), k8.data_ptr<int8_t>(), static_cast<const uint8_t*>(v8.data_ptr()), q_scale.data_ptr<float>(),
      k_scale.data_ptr<float>(), vsp, vmp, mask, sparse_bs, output.data_ptr(), code_of(output), lse_p, (int)B, (int)H, (int)Hkv,
      (int)Nq, (int)Nk, (int)D, q8.stride(0), q8.stride(1), q8.stride(2), k8.stride(0), k8.stride(1), k8.stride(2),
      output.stride(0), output.stride(1), output.stride(2), (float)sm_scale, is_causal, flags,
      orders ? orders->data_ptr<int32_t>() : nullptr, n_text, F, Hh, W, n_scratch > 0 ? scratch.data_ptr() : nullptr,
      stream_of(q8)));
  return lse;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "paroattention's extension modules (_qattn_sm80, _fused, _rope) over libparoatten_hip.so (gfx950)";
  py::register_local_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const Unsupported& e) {
      PyErr_SetString(PyExc_NotImplementedError, e.what());
    }
  });
  m.def("abi_version", &paro_abi_version);
  auto qattn = m.def_submodule("_qattn_sm80");
  qattn.def("qk_int8_sv_f16_accum_f16_attn", &qk_int8_sv_f16_accum_f16_attn, "QK int8 sv f16 accum f16 attn");
  qattn.def("set_attention_flags", &set_attention_flags,
            "process-wide PARO_ATTN_* flags of the attention entry point (1 exact exponentials, 16 float16 P.V product, ...)");
  qattn.def("get_attention_flags", &get_attention_flags);
  qattn.def("qk_int4_sv_f16_accum_f16_attn", &prototype_variant);
  qattn.def("qk_int4_sv_int8_accum_f16_attn", &prototype_variant);
  qattn.def("qk_int8_sv_int8_accum_f16_attn", &prototype_variant);
  auto fused = m.def_submodule("_fused");
  fused.def("quant_per_block_int8_cuda", &quant_per_block_int8_cuda_sm);
  fused.def("quant_per_block_int8_cuda", &quant_per_block_int8_cuda);
  fused.def("quant_per_block_int8_fuse_sub_mean_cuda", &quant_per_block_int8_fuse_sub_mean_cuda);
  fused.def("quant_per_warp_int8_cuda", &quant_per_warp_int8_cuda);
  fused.def("sub_mean_cuda", &sub_mean_cuda);
  fused.def("transpose_pad_permute_cuda", &transpose_pad_permute_cuda);
  fused.def("scale_fuse_quant_cuda", &scale_fuse_quant_cuda);
  fused.def("mean_scale_fuse_quant_cuda", &mean_scale_fuse_quant_cuda);
  auto rope = m.def_submodule("_rope");
  auto ops = m.def_submodule("_ops");
  const py::call_guard<py::gil_scoped_release> unlocked;
  ops.def("attn_operator", &attn_operator);   // releases the lock itself: its result is a Python object
  ops.def("attn_sparse_prepacked", &attn_sparse_prepacked, unlocked);
  ops.def("rope_permute", &rope_permute, unlocked);
  ops.def("rope_permute_quant", &rope_permute_quant, unlocked);
  ops.def("permute_inverse", &permute_inverse, unlocked);
  ops.def("head_norm", &head_norm, unlocked);
  rope.def("rope_permutation", &rope_permutation, "RoPE op with permutation.");
}
