// V -> FP8 (e4m3fn) per-channel quantisation with mean smoothing, written in the fragment order
// of the P.V MFMA (v_mfma_f32_32x32x64_f8f6f4) so that the attention kernel's K-loop copies V
// tiles straight from HBM to LDS and reads each A operand as one contiguous 16-byte piece per lane.
//
// Three launches, all HBM-bound and deterministic (no float atomics):
//   v_stats    : per v_chunk(N)-token chunk, per channel: sum, min, max      (reads V once)
//   v_finalize : per (b,h,channel): mean = sum/N, amax = max(max-mean, mean-min), scale = amax/448,
//                recp = 448/amax
//   v_pack     : per 64-token tile: (v-mean)*recp -> e4m3, fragment order  (reads V once more), and the
//                tile's rounding residual sums per channel
//   v_residual : per (b,h,channel): v_mean += scale * (sum of residuals) / N
// The last step removes the mean error of the codes: rounding (v-mean)/scale to e4m3 is unbiased only if
// the values are spread evenly over the rounding cells, and 16-bit inputs (bfloat16 above all, with its 8
// significant bits) are a lattice that is not; what is left, ~3e-4 of max|v| per channel, does not
// average out over the keys of an attention row, whereas the rounding noise does.
// max|v-mean| over tokens equals max(max-mean, mean-min) exactly because fp32 subtraction is
// monotonic, so no second reduction pass is needed.
// Arithmetic follows MeanScaleKernel of the reference (csrc/fused/fused.cu:316-427) except that the
// mean divides by the true token count.
#include "share_device.hpp"
#include "stats_device.hpp"
#include "v_pack_device.hpp"

namespace paro {

template <int DT, int D>
__global__ void __launch_bounds__(256) v_stats_kernel(const unsigned short* __restrict__ v,
                                                      float* __restrict__ partial, int N, int n_chunks,
                                                      int64_t vs_b, int64_t vs_h, int64_t vs_n) {
  v_stats_body<DT, D>(v, partial, N, n_chunks, vs_b, vs_h, vs_n, blockIdx.x, blockIdx.y, blockIdx.z, gridDim.y);
}

template <int D>
__global__ void __launch_bounds__(1024) v_finalize_kernel(float* work, float* __restrict__ v_scale,
                                                          float* __restrict__ v_mean, int N, int n_chunks,
                                                          int smooth) {
  v_finalize_body<D>(work, v_scale, v_mean, N, n_chunks, smooth, blockIdx.x, gridDim.x);
}

template <int DT, int D>
__global__ void __launch_bounds__(256) v_pack_kernel(const unsigned short* __restrict__ v, uint8_t* __restrict__ v8,
                                                     const float* __restrict__ work, const float* __restrict__ v_mean,
                                                     float* __restrict__ resid, int N, int nb, int64_t vs_b,
                                                     int64_t vs_h, int64_t vs_n) {
  const int h = blockIdx.y, b = blockIdx.z;
  v_pack_body<DT, D>(v + b * vs_b + h * vs_h, v8, work, v_mean, resid, N, nb, vs_n, blockIdx.x, (int64_t)b * gridDim.y + h);
}

// v_mean += v_scale * (sum over tiles and row tiles of the residual sums) / N.  A workgroup has one of PARTS parts of a head's channels;
// a thread takes four of them of every SL-th row (16-byte loads, all independent), the SL partial sums per channel are
// combined through LDS in a fixed order, the same for any PARTS.  What bounds it is the trips to memory one after the other, behind a launch of 4 to
// 5 us in a kernel trace; with one workgroup to a head and four loads in flight per thread instead of eight, 40 heads, D = 128:
// four parts N = 75600 15.0 -> 10.4 us, N = 32760 8.0 -> 6.3 (D = 64, two parts, N = 17776, 96 heads: 5.3 and 5.6).
template <int D, int PARTS>
__global__ void __launch_bounds__(1024 / PARTS) v_residual_kernel(const float* __restrict__ resid,
                                                          const float* __restrict__ v_scale,
                                                          float* __restrict__ v_mean, int N, int n_rows, int heads,
                                                          const ShareLook look) {
  constexpr int CH = D / PARTS, CW = CH / 4;   // a workgroup's channels, and threads per row
  if ((int)blockIdx.x >= heads * PARTS) {
    share_look(look, blockIdx.x - heads * PARTS);
    return;
  }
  constexpr int C4 = D / 4;
  constexpr int SL = 1024 / C4;      // rows in flight per pass
  __shared__ v4f red[SL][CW];
  const int c4 = threadIdx.x % CW, sl = threadIdx.x / CW, part = blockIdx.x % PARTS;
  const int64_t bh = blockIdx.x / PARTS;
  const v4f* p = reinterpret_cast<const v4f*>(resid + bh * n_rows * D) + part * CW + c4;
  v4f s = {0.f, 0.f, 0.f, 0.f};
  // (what the sum goes into is asked for here: behind it, it was one more trip)
  const int64_t ch = bh * D + part * CH + (threadIdx.x & (CH - 1));
  const float mean = v_mean[ch], scale = v_scale[ch];
  // (a batch at a time also where less of it is left, since a loop unrolled by eight takes the remainder one by one; but no more than
  // a thread has rows: eight throughout, a layer of 20 heads, N = 2192, D = 64 39.4 us, so 38.4)
  auto add = [&](auto batch) __attribute__((always_inline)) {
    constexpr int U = decltype(batch)::value;
    for (int r = sl; r < n_rows; r += U * SL) {
      v4f x[U];
#pragma unroll
      for (int u = 0; u < U; u++) x[u] = p[(int64_t)min(r + u * SL, n_rows - 1) * C4];
#pragma unroll
      for (int u = 0; u < U; u++)
        if (r + u * SL < n_rows) s += x[u];
    }
  };
  if (n_rows <= SL) add(std::integral_constant<int, 1>{});
  else if (n_rows <= 2 * SL) add(std::integral_constant<int, 2>{});
  else if (n_rows <= 4 * SL) add(std::integral_constant<int, 4>{});
  else add(std::integral_constant<int, 8>{});
  red[sl][c4] = s;
  __syncthreads();
  if (threadIdx.x < CH) {
    float t = 0.f;
#pragma unroll 8
    for (int i = 0; i < SL; i++) t += red[i][threadIdx.x >> 2][threadIdx.x & 3];
    v_mean[ch] = mean + scale * (t / (float)N);
  }
}

int v_fp8_add_residual(const float* resid, const float* v_scale, float* v_mean, int B, int Hkv, int N, int D,
                       hipStream_t st, const ShareLook* look) {
  const int n_rows = ceil_div(N, 64) * 2, heads = B * Hkv;
  const ShareLook l = look ? *look : ShareLook{};
  auto launch = [&](auto kern, int parts) {
    hipLaunchKernelGGL(kern, dim3(heads * parts + l.heads), dim3(1024 / parts), 0, st, resid, v_scale, v_mean, N, n_rows, heads, l);
    PARO_HIP(hipGetLastError());
    return PARO_OK;
  };
  if (D == 128) return launch(v_residual_kernel<128, 4>, 4);
  // (a workgroup per head / two, layer, replayed graphs, us: 14 heads, N = 630 22.60 / 22.78, 1024 24.42 / 24.57, 2048 30.79 / 30.90, 3 heads,
  // 4096 29.36 / 29.49; from 8192 tokens on two are ahead, 3 heads 43.77 / 43.58, 48 188.3 / 188.1)
  return n_rows <= 128 ? launch(v_residual_kernel<64, 1>, 1) : launch(v_residual_kernel<64, 2>, 2);
}

template <int DT, int D>
static int run_v_stats(const void* v, float* v_scale, float* v_mean, float* partial, int B, int Hkv, int N,
                       int64_t vs_b, int64_t vs_h, int64_t vs_n, int smooth, hipStream_t st) {
  const int n_chunks = ceil_div(N, v_chunk(N));
  hipLaunchKernelGGL((v_stats_kernel<DT, D>), dim3(n_chunks, Hkv, B), dim3(256), 0, st, (const unsigned short*)v,
                     partial + v_stats_offset((int64_t)B * Hkv, N, D), N, n_chunks, vs_b, vs_h, vs_n);
  PARO_HIP(hipGetLastError());
  hipLaunchKernelGGL((v_finalize_kernel<D>), dim3(B * Hkv), dim3(1024), 0, st, partial, v_scale, v_mean, N,
                     n_chunks, smooth);
  PARO_HIP(hipGetLastError());
  return PARO_OK;
}

int v_fp8_stats(const void* v, int dtype, float* v_scale, float* v_mean, float* partial, int B, int Hkv, int N,
                int D, int64_t vs_b, int64_t vs_h, int64_t vs_n, int smooth, hipStream_t st) {
  if (dtype == PARO_DTYPE_F16) {
    if (D == 64) return run_v_stats<PARO_DTYPE_F16, 64>(v, v_scale, v_mean, partial, B, Hkv, N, vs_b, vs_h, vs_n, smooth, st);
    return run_v_stats<PARO_DTYPE_F16, 128>(v, v_scale, v_mean, partial, B, Hkv, N, vs_b, vs_h, vs_n, smooth, st);
  }
  if (D == 64) return run_v_stats<PARO_DTYPE_BF16, 64>(v, v_scale, v_mean, partial, B, Hkv, N, vs_b, vs_h, vs_n, smooth, st);
  return run_v_stats<PARO_DTYPE_BF16, 128>(v, v_scale, v_mean, partial, B, Hkv, N, vs_b, vs_h, vs_n, smooth, st);
}

template <int DT, int D>
static int run_v_pack(const void* v, uint8_t* v8, float* partial, float* v_scale, float* v_mean, int B, int Hkv,
                      int N, int64_t vs_b, int64_t vs_h, int64_t vs_n, hipStream_t st) {
  const int nb = ceil_div(N, 64);
  // without smoothing there is no mean to correct
  float* resid = v_mean ? partial + v_resid_offset((int64_t)B * Hkv, N, D) : nullptr;
  hipLaunchKernelGGL((v_pack_kernel<DT, D>), dim3(nb, Hkv, B), dim3(256), 0, st, (const unsigned short*)v, v8,
                     partial, v_mean, resid, N, nb, vs_b, vs_h, vs_n);
  PARO_HIP(hipGetLastError());
  if (resid) return v_fp8_add_residual(resid, v_scale, v_mean, B, Hkv, N, D, st);
  return PARO_OK;
}

// out_f16 = fp16(v - mean): SubMeanKernel of the reference (csrc/fused/fused.cu:200-260); for bf16
// input the subtraction is rounded to bf16 before the conversion to fp16, as there.
template <int DT, int D>
__global__ void __launch_bounds__(256) sub_mean_kernel(const unsigned short* __restrict__ v,
                                                       const unsigned short* __restrict__ mean,
                                                       unsigned short* __restrict__ out, int N, int64_t vs_b,
                                                       int64_t vs_h, int64_t vs_n, int64_t ms_b, int64_t ms_h,
                                                       int64_t os_b, int64_t os_h, int64_t os_n) {
  constexpr int LPR = D / 8;
  const int t = threadIdx.x;
  const int tok = blockIdx.x * (256 / LPR) + t / LPR;
  if (tok >= N) return;
  const int h = blockIdx.y, b = blockIdx.z, col = (t % LPR) * 8;
  const v4i raw = *reinterpret_cast<const v4i*>(v + b * vs_b + h * vs_h + (int64_t)tok * vs_n + col);
  const v4i mr = *reinterpret_cast<const v4i*>(mean + b * ms_b + h * ms_h + col);
  v4i o;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    unsigned short r2[2];
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const unsigned short xv = (unsigned short)(((unsigned)raw[j] >> (16 * q)) & 0xffffu);
      const unsigned short mv = (unsigned short)(((unsigned)mr[j] >> (16 * q)) & 0xffffu);
      float d = F16x<DT>::to_f32(xv) - F16x<DT>::to_f32(mv);
      if constexpr (DT == PARO_DTYPE_BF16) d = F16x<PARO_DTYPE_BF16>::to_f32(F16x<PARO_DTYPE_BF16>::from_f32(d));
      r2[q] = F16x<PARO_DTYPE_F16>::from_f32(d);
    }
    o[j] = (int)((unsigned)r2[0] | ((unsigned)r2[1] << 16));
  }
  *reinterpret_cast<v4i*>(out + b * os_b + h * os_h + (int64_t)tok * os_n + col) = o;
}

}  // namespace paro

extern "C" int64_t paro_v_fp8_bytes(int B, int Hkv, int N, int D) {
  return (int64_t)B * Hkv * paro::ceil_div(N, 64) * 64 * D;
}
extern "C" int64_t paro_v_fp8_partial_floats(int B, int Hkv, int N, int D) {
  // see v_resid_offset: statistics (sum, min, max per chunk and channel), residual sums per row tile
  return (int64_t)B * Hkv * ((int64_t)paro::ceil_div(N, paro::V_CHUNK) * 3 + (int64_t)paro::ceil_div(N, 64) * 2) * D;
}

extern "C" int paro_v_fp8_pack(const void* v, int dtype, uint8_t* v8, float* v_scale, float* v_mean,
                               float* partial, int B, int Hkv, int N, int D, int64_t v_stride_b,
                               int64_t v_stride_h, int64_t v_stride_n, int smooth, void* stream) {
  using namespace paro;
  PARO_CHECK(v && v8 && v_scale && partial, PARO_ERR_RUNTIME, "paro_v_fp8_pack: null tensor pointer");
  PARO_CHECK(!smooth || v_mean, PARO_ERR_RUNTIME, "paro_v_fp8_pack: smoothing needs a v_mean buffer");
  PARO_CHECK(B > 0 && Hkv > 0 && N > 0, PARO_ERR_RUNTIME, "paro_v_fp8_pack: empty shape");
  PARO_CHECK(B <= MAX_GRID_YZ && Hkv <= MAX_GRID_YZ, PARO_ERR_RUNTIME, "paro_v_fp8_pack: batch or head count exceeds %d",
             MAX_GRID_YZ);
  PARO_CHECK(D == 64 || D == 128, PARO_ERR_INVALID_VALUE, "Unsupported head dim: %d", D);
  PARO_CHECK(dtype == PARO_DTYPE_F16 || dtype == PARO_DTYPE_BF16, PARO_ERR_RUNTIME,
             "Unsupported input dtype (expect float16 or bfloat16)");
  PARO_CHECK(v_stride_n % 8 == 0 && v_stride_h % 8 == 0 && v_stride_b % 8 == 0 && ((uintptr_t)v % 16) == 0,
             PARO_ERR_RUNTIME, "Tensor value must be 16-byte aligned with strides that are multiples of 8");
  PARO_CHECK(((uintptr_t)v8 % 16) == 0, PARO_ERR_RUNTIME, "paro_v_fp8_pack: v8 must be 16-byte aligned");
  hipStream_t st = (hipStream_t)stream;
  if (int rc = v_fp8_stats(v, dtype, v_scale, v_mean, partial, B, Hkv, N, D, v_stride_b, v_stride_h, v_stride_n,
                           smooth, st))
    return rc;
  float* mean = smooth ? v_mean : nullptr;
  if (dtype == PARO_DTYPE_F16) {
    if (D == 64) return run_v_pack<PARO_DTYPE_F16, 64>(v, v8, partial, v_scale, mean, B, Hkv, N, v_stride_b, v_stride_h, v_stride_n, st);
    return run_v_pack<PARO_DTYPE_F16, 128>(v, v8, partial, v_scale, mean, B, Hkv, N, v_stride_b, v_stride_h, v_stride_n, st);
  }
  if (D == 64) return run_v_pack<PARO_DTYPE_BF16, 64>(v, v8, partial, v_scale, mean, B, Hkv, N, v_stride_b, v_stride_h, v_stride_n, st);
  return run_v_pack<PARO_DTYPE_BF16, 128>(v, v8, partial, v_scale, mean, B, Hkv, N, v_stride_b, v_stride_h, v_stride_n, st);
}

extern "C" int paro_sub_mean(const void* v, int dtype, const void* mean, void* out_f16, int B, int H, int N,
                             int D, int64_t v_stride_b, int64_t v_stride_h, int64_t v_stride_n,
                             int64_t mean_stride_b, int64_t mean_stride_h, int64_t out_stride_b,
                             int64_t out_stride_h, int64_t out_stride_n, void* stream) {
  using namespace paro;
  PARO_CHECK(v && mean && out_f16, PARO_ERR_RUNTIME, "paro_sub_mean: null tensor pointer");
  PARO_CHECK(B > 0 && H > 0 && N > 0 && B <= MAX_GRID_YZ && H <= MAX_GRID_YZ, PARO_ERR_RUNTIME,
             "paro_sub_mean: empty shape, or batch or head count above %d", MAX_GRID_YZ);
  PARO_CHECK(D == 64 || D == 128, PARO_ERR_INVALID_VALUE, "Unsupported head dim: %d", D);
  PARO_CHECK(dtype == PARO_DTYPE_F16 || dtype == PARO_DTYPE_BF16, PARO_ERR_RUNTIME,
             "Unsupported input dtype (expect float16 or bfloat16)");
  PARO_CHECK(v_stride_n % 8 == 0 && v_stride_h % 8 == 0 && v_stride_b % 8 == 0 && out_stride_n % 8 == 0 &&
                 out_stride_h % 8 == 0 && out_stride_b % 8 == 0 && mean_stride_b % 8 == 0 && mean_stride_h % 8 == 0 &&
                 ((uintptr_t)v % 16) == 0 && ((uintptr_t)out_f16 % 16) == 0 && ((uintptr_t)mean % 16) == 0,
             PARO_ERR_RUNTIME, "paro_sub_mean: tensors must be 16-byte aligned with strides that are multiples of 8");
  hipStream_t st = (hipStream_t)stream;
  const int rows = 256 / (D / 8);
  dim3 grid(ceil_div(N, rows), H, B), block(256);
#define PARO_SM(DTV, DV)                                                                                      \
  hipLaunchKernelGGL((sub_mean_kernel<DTV, DV>), grid, block, 0, st, (const unsigned short*)v,                \
                     (const unsigned short*)mean, (unsigned short*)out_f16, N, v_stride_b, v_stride_h,        \
                     v_stride_n, mean_stride_b, mean_stride_h, out_stride_b, out_stride_h, out_stride_n)
  if (dtype == PARO_DTYPE_F16) {
    if (D == 64) PARO_SM(PARO_DTYPE_F16, 64); else PARO_SM(PARO_DTYPE_F16, 128);
  } else {
    if (D == 64) PARO_SM(PARO_DTYPE_BF16, 64); else PARO_SM(PARO_DTYPE_BF16, 128);
  }
#undef PARO_SM
  PARO_HIP(hipGetLastError());
  return PARO_OK;
}
