// The whole attention operator on 16-bit q, k, v in one call: INT8 quantisation of Q and K (K's token mean taken off
// first if asked for), the V conversion, block-sparse attention.  Five launches:
//   op_stats     K sums (smooth_k) and V statistics (FP8 product), side by side
//   op_finalize  their second steps
//   op_prep      quantised K and the V tiles, side by side (per-thread scales: quantised Q too)
//   v_residual   (FP8 product with smooth_v)
//   attention    on 16-bit Q, which the q-block's own waves quantise (QRows; per-thread scales: on INT8 Q); the
//                log-sum-exp leaves as the natural one of the scores of q and k as given
// The first four are bound by HBM: at B = 2, H = 48, N = 17776, D = 64 they move 16-bit K and V twice and write their 8-bit
// forms, 1.09 GB.  Q as a pass in op_prep moved 3 bytes per element and the attention launch read a fourth; quantised there,
// behind the requests for the first tiles, start to end of the operator: 1521 -> 1488 us at that shape, 212 -> 205 us at
// N = 8192, B = 1, 502 -> 494 us at N = 9001 with the log-sum-exp, 655 -> 636 us at B = 2, H = 32, Hkv = 8, N = 8192, D = 128, causal,
// 42.4 -> 40.1 us at B = 2, H = 22, N = 1122, D = 128; calls of a few hundred tokens the same.
// op_prep takes the heads in reverse, K and V of a head together, and so finds the last 256 MB of the first pass in the
// memory-side cache: 9 us less at the first of these shapes, 3 us at the second, 23 us at N = 32760, H = 40, D = 128 than
// tensor by tensor (with Q among them).
//
// Stands in for paroattn_qk_int8_pv_fp16_cuda below its argument checks (paroattention/core.py:86-216).
#include "attn_common.hpp"
#include "quant_device.hpp"
#include "stats_device.hpp"
#include "v_pack_device.hpp"

namespace paro {

struct OpParams {
  const unsigned short *q, *k, *v;
  int64_t qs_b, qs_h, qs_n, ks_b, ks_h, ks_n, vs_b, vs_h, vs_n;
  int8_t *q8, *k8;
  float *q_scale, *k_scale;
  uint8_t* v_tiles;             // FP8 or float16 tiles
  float *v_scale, *v_mean, *v_work, *v_resid;
  float* k_partial;
  unsigned short* k_mean;       // nullptr: not smoothed
  float* lse_add;               // per-thread scales: sm_scale * q . k_mean per row; nullptr: not wanted
  int B, H, Hkv, Nq, Nk, nbq, nbk, chunks, smooth_v;
  int stats_k, stats_v;         // which statistics are taken
  int kv_blocks;                // workgroups of op_prep that take K or V; the rest (per-thread scales) take Q
  float sm_scale;
};

template <int DT, int D>
__global__ void __launch_bounds__(256) op_stats_kernel(const OpParams p) {
  // K and V of a head one after the other, in x: y and z keep the whole range of head and batch counts
  const int h = blockIdx.y, b = blockIdx.z;
  const int k_chunks = p.stats_k ? p.chunks : 0;
  if ((int)blockIdx.x < k_chunks)
    v_stats_body<DT, D, true>(p.k, p.k_partial, p.Nk, p.chunks, p.ks_b, p.ks_h, p.ks_n, blockIdx.x, h, b, p.Hkv);
  else
    v_stats_body<DT, D>(p.v, p.v_work + v_stats_offset((int64_t)p.B * p.Hkv, p.Nk, D), p.Nk, p.chunks, p.vs_b, p.vs_h,
                        p.vs_n, (int)blockIdx.x - k_chunks, h, b, p.Hkv);
}

template <int DT, int D>
__global__ void __launch_bounds__(1024) op_finalize_kernel(const OpParams p) {
  const int BH = p.B * p.Hkv;
  if ((int)blockIdx.x < BH * p.stats_k)
    k_mean_finalize_body<DT, D, double>(p.k_partial, p.k_mean, p.Nk, p.chunks, (int64_t)p.Hkv * D, D, p.Hkv, blockIdx.x);
  else
    v_finalize_body<D>(p.v_work, p.v_scale, p.v_mean, p.Nk, p.chunks, p.smooth_v, (int64_t)blockIdx.x - BH * p.stats_k, BH);
}

// PT: per-thread scale granularity.  A workgroup takes one V tile, 256 tokens of K or (PT) 256 tokens of Q.
template <int DT, int D, bool PT, bool F16V>
__global__ void __launch_bounds__(256) op_prep_kernel(const OpParams p) {
  const int wave = threadIdx.x >> 6;
  int i = blockIdx.x;
  if (i < p.kv_blocks) {
    // K and V of a head one after the other, the heads in reverse: the last ones that the statistics have read are
    // still in the memory-side cache
    const int per_k = (p.nbk + 3) / 4, per = p.nbk + per_k;
    const int bh = p.B * p.Hkv - 1 - i / per;
    const int j = i % per;
    if (j < p.nbk) {
      const unsigned short* v = p.v + bh / p.Hkv * p.vs_b + bh % p.Hkv * p.vs_h;
      if constexpr (F16V) v_f16_pack_body<DT, D>(v, (unsigned short*)p.v_tiles, p.Nk, p.nbk, p.vs_n, j, bh);
      else v_pack_body<DT, D>(v, p.v_tiles, p.v_work, p.smooth_v ? p.v_mean : nullptr, p.v_resid, p.Nk, p.nbk, p.vs_n, j, bh);
      return;
    }
    const int g = (j - p.nbk) * 4 + wave;
    if (g >= p.nbk) return;
    const unsigned short* k = p.k + bh / p.Hkv * p.ks_b + bh % p.Hkv * p.ks_h;
    const unsigned short* mean = p.k_mean ? p.k_mean + (int64_t)bh * D : nullptr;
    int8_t* out = p.k8 + (int64_t)bh * p.Nk * D;
    float* scale = p.k_scale + (int64_t)bh * p.nbk * (PT ? 4 : 1);
    if constexpr (PT) {
      if (mean) quant_per_thread_body<DT, D, true, true>(k, mean, out, scale, p.Nk, g, p.ks_n, D);
      else quant_per_thread_body<DT, D, true, false>(k, mean, out, scale, p.Nk, g, p.ks_n, D);
    } else {
      if (mean) quant_group_body<DT, D, 64, true, false>(k, mean, out, scale, p.Nk, g, p.ks_n, D, 0.f);
      else quant_group_body<DT, D, 64, false, false>(k, mean, out, scale, p.Nk, g, p.ks_n, D, 0.f);
    }
    return;
  }
  if constexpr (PT) {
    i -= p.kv_blocks;
    const int per = (p.nbq + 3) / 4, bh = i / per, g = i % per * 4 + wave;
    if (g >= p.nbq) return;
    const int b = bh / p.H, h = bh % p.H;
    float* dot = p.lse_add ? p.lse_add + (int64_t)bh * p.Nq : nullptr;
    const unsigned short* with = p.lse_add ? p.k_mean + ((int64_t)b * p.Hkv + h / (p.H / p.Hkv)) * D : nullptr;
    quant_per_thread_body<DT, D, false, false>(p.q + b * p.qs_b + h * p.qs_h, nullptr, p.q8 + (int64_t)bh * p.Nq * D,
                                               p.q_scale + (int64_t)bh * p.nbq * 16, p.Nq, g, p.qs_n, D, p.sm_scale, dot, with);
  }
}

// Where the intermediate tensors lie in the workspace (256-byte aligned pieces).
struct OpLayout {
  int64_t q8, k8, v_tiles, q_scale, k_scale, v_scale, v_mean, v_work, k_partial, k_mean, bytes;
  OpLayout(int B, int H, int Hkv, int Nq, int Nk, int D, bool smooth_k, bool per_thread, bool f16v) {
    bytes = 0;
    auto take = [&](int64_t n) {
      const int64_t at = bytes;
      bytes += (n + 255) & ~(int64_t)255;
      return at;
    };
    const int64_t nbq = ceil_div(Nq, 64), nbk = ceil_div(Nk, 64), BK = (int64_t)B * Hkv, BQ = (int64_t)B * H;
    q8 = take(per_thread ? BQ * Nq * D : 0);   // (per warp: the attention kernels quantise Q themselves)
    k8 = take(BK * Nk * D);
    v_tiles = take(BK * nbk * 64 * D * (f16v ? 2 : 1));
    q_scale = take(per_thread ? BQ * nbq * 16 * 4 : 0);
    k_scale = take(BK * nbk * (per_thread ? 4 : 1) * 4);
    v_scale = take(f16v ? 0 : BK * D * 4);
    v_mean = take(f16v ? 0 : BK * D * 4);
    v_work = take(f16v ? 0 : paro_v_fp8_partial_floats(B, Hkv, Nk, D) * 4);
    k_partial = take(smooth_k ? BK * ceil_div(Nk, v_chunk(Nk)) * D * 4 : 0);
    k_mean = take(smooth_k ? BK * D * 2 : 0);
  }
};

template <int DT, int D>
static int launch_op_prep(const OpParams& p, bool per_thread, bool f16v, hipStream_t st) {
  if (p.stats_k + p.stats_v > 0) {
    hipLaunchKernelGGL((op_stats_kernel<DT, D>), dim3(p.chunks * (p.stats_k + p.stats_v), p.Hkv, p.B), dim3(256), 0, st, p);
    hipLaunchKernelGGL((op_finalize_kernel<DT, D>), dim3(p.B * p.Hkv * (p.stats_k + p.stats_v)), dim3(1024), 0, st, p);
  }
  const int q_blocks = per_thread ? p.B * p.H * ceil_div(p.nbq, 4) : 0;
  const dim3 grid(p.kv_blocks + q_blocks);
  if (per_thread) hipLaunchKernelGGL((op_prep_kernel<DT, D, true, false>), grid, dim3(256), 0, st, p);
  else if (f16v) hipLaunchKernelGGL((op_prep_kernel<DT, D, false, true>), grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL((op_prep_kernel<DT, D, false, false>), grid, dim3(256), 0, st, p);
  PARO_HIP(hipGetLastError());
  return PARO_OK;
}

}  // namespace paro

extern "C" int64_t paro_attn_operator_workspace_bytes(int B, int H, int Hkv, int Nq, int Nk, int D, int smooth_k,
                                                      int with_lse, int qk_quant_gran, int flags) {
  (void)with_lse;
  return paro::OpLayout(B, H, Hkv, Nq, Nk, D, smooth_k != 0, qk_quant_gran == 3, (flags & PARO_ATTN_PV_F16) != 0).bytes;
}

extern "C" int paro_attn_operator(const void* q, const void* k, const void* v, int dtype, void* out,
                                  const uint8_t* sparse, int64_t sparse_batch_stride, float* lse, void* workspace,
                                  int64_t workspace_bytes, int B, int H, int Hkv, int Nq, int Nk, int D,
                                  int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_n, int64_t k_stride_b,
                                  int64_t k_stride_h, int64_t k_stride_n, int64_t v_stride_b, int64_t v_stride_h,
                                  int64_t v_stride_n, int64_t o_stride_b, int64_t o_stride_h, int64_t o_stride_n,
                                  int is_causal, int qk_quant_gran, float sm_scale, int smooth_k, int smooth_v, int flags,
                                  void* stream) {
  using namespace paro;
  PARO_CHECK(q && k && v && out && sparse, PARO_ERR_RUNTIME, "paro_attn_operator: null tensor pointer");
  PARO_CHECK(B > 0 && H > 0 && Hkv > 0 && Nq > 0 && Nk > 0, PARO_ERR_RUNTIME, "paro_attn_operator: empty shape");
  PARO_CHECK(D == 64 || D == 128, PARO_ERR_INVALID_VALUE, "Unsupported head dim: %d", D);
  PARO_CHECK(H % Hkv == 0, PARO_ERR_INVALID_VALUE, "num_qo_heads (%d) must be divisible by num_kv_heads (%d)", H, Hkv);
  PARO_CHECK(dtype == PARO_DTYPE_F16 || dtype == PARO_DTYPE_BF16, PARO_ERR_RUNTIME,
             "Unsupported input dtype (expect float16 or bfloat16)");
  PARO_CHECK(qk_quant_gran == 2 || qk_quant_gran == 3, PARO_ERR_INVALID_VALUE, "Unsupported quantization granularity: %d",
             qk_quant_gran);
  const bool per_thread = qk_quant_gran == 3, f16v = (flags & PARO_ATTN_PV_F16) != 0;
  PARO_CHECK(!(per_thread && f16v), PARO_ERR_UNSUPPORTED, "per-thread scales do not go with PARO_ATTN_PV_F16");
  PARO_CHECK(B <= MAX_GRID_YZ && H <= MAX_GRID_YZ, PARO_ERR_RUNTIME,
             "paro_attn_operator: batch or head count exceeds %d", MAX_GRID_YZ);
  PARO_CHECK((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) % 16) == 0 &&
                 ((q_stride_b | q_stride_h | q_stride_n | k_stride_b | k_stride_h | k_stride_n | v_stride_b | v_stride_h |
                   v_stride_n) % 8) == 0,
             PARO_ERR_RUNTIME, "Tensor query/key/value must be 16-byte aligned with strides that are multiples of 8");
  const OpLayout at(B, H, Hkv, Nq, Nk, D, smooth_k != 0, per_thread, f16v);
  PARO_CHECK(workspace && ((uintptr_t)workspace % 256) == 0 && workspace_bytes >= at.bytes, PARO_ERR_RUNTIME,
             "paro_attn_operator: workspace of %lld bytes (256-byte aligned) is needed, %lld given", (long long)at.bytes,
             (long long)workspace_bytes);
  uint8_t* ws = (uint8_t*)workspace;
  OpParams p;
  p.q = (const unsigned short*)q; p.k = (const unsigned short*)k; p.v = (const unsigned short*)v;
  p.qs_b = q_stride_b; p.qs_h = q_stride_h; p.qs_n = q_stride_n;
  p.ks_b = k_stride_b; p.ks_h = k_stride_h; p.ks_n = k_stride_n;
  p.vs_b = v_stride_b; p.vs_h = v_stride_h; p.vs_n = v_stride_n;
  p.B = B; p.H = H; p.Hkv = Hkv; p.Nq = Nq; p.Nk = Nk; p.nbq = ceil_div(Nq, 64); p.nbk = ceil_div(Nk, 64);
  PARO_CHECK((int64_t)B * H * p.nbq + 2 * (int64_t)B * Hkv * p.nbk < (int64_t)1 << 31, PARO_ERR_RUNTIME,
             "paro_attn_operator: too many blocks");
  p.q8 = (int8_t*)(ws + at.q8); p.k8 = (int8_t*)(ws + at.k8); p.v_tiles = ws + at.v_tiles;
  p.q_scale = (float*)(ws + at.q_scale); p.k_scale = (float*)(ws + at.k_scale);
  p.v_scale = f16v ? nullptr : (float*)(ws + at.v_scale);
  p.v_mean = f16v ? nullptr : (float*)(ws + at.v_mean);
  p.v_work = (float*)(ws + at.v_work);
  p.smooth_v = smooth_v != 0;
  p.v_resid = !f16v && smooth_v ? p.v_work + v_resid_offset((int64_t)B * Hkv, Nk, D) : nullptr;
  p.k_partial = (float*)(ws + at.k_partial);
  p.k_mean = smooth_k ? (unsigned short*)(ws + at.k_mean) : nullptr;
  p.lse_add = per_thread && smooth_k ? lse : nullptr;   // (the attention kernel adds to what the row holds)
  p.chunks = ceil_div(Nk, v_chunk(Nk));
  p.stats_k = smooth_k != 0; p.stats_v = !f16v;
  p.kv_blocks = B * Hkv * (p.nbk + ceil_div(p.nbk, 4));
  p.sm_scale = sm_scale;
  hipStream_t st = (hipStream_t)stream;
  int rc;
  if (dtype == PARO_DTYPE_F16)
    rc = D == 64 ? launch_op_prep<PARO_DTYPE_F16, 64>(p, per_thread, f16v, st) : launch_op_prep<PARO_DTYPE_F16, 128>(p, per_thread, f16v, st);
  else
    rc = D == 64 ? launch_op_prep<PARO_DTYPE_BF16, 64>(p, per_thread, f16v, st) : launch_op_prep<PARO_DTYPE_BF16, 128>(p, per_thread, f16v, st);
  if (rc) return rc;
  if (p.v_resid)
    if ((rc = v_fp8_add_residual(p.v_resid, p.v_scale, p.v_mean, B, Hkv, Nk, D, st))) return rc;
  AttnExtra extra;
  extra.lse_scale = 0.6931471805599453f;
  extra.lse_add = p.lse_add != nullptr;
  if (!per_thread) {
    extra.q16 = p.q;
    extra.k_mean = p.k_mean;
    extra.lse_dot_scale = sm_scale;
  }
  const int64_t qs_b = per_thread ? (int64_t)H * Nq * D : q_stride_b, qs_h = per_thread ? (int64_t)Nq * D : q_stride_h;
  return attn_sparse_impl(p.q8, p.k8, p.v_tiles, p.q_scale, p.k_scale, p.v_scale, smooth_v ? p.v_mean : nullptr, sparse,
                          sparse_batch_stride, out, dtype, lse, extra, nullptr, B, H, Hkv, Nq, Nk, D, qs_b, qs_h,
                          per_thread ? D : q_stride_n, (int64_t)Hkv * Nk * D, (int64_t)Nk * D, D, o_stride_b, o_stride_h,
                          o_stride_n, sm_scale, is_causal, flags | (per_thread ? PARO_ATTN_QK_PER_THREAD : 0), nullptr, 0, 0, 0,
                          0, stream);
}
