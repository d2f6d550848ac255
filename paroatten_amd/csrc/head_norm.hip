// LayerNorm over the channels of a head, for q and k of an attention block in one launch: what CogVideoX's attention does
// between its projections and the rotation (paroattention/cogvideox.py:157-160).
//
// Bound by HBM, 4 bytes an element and tensor.  A row is 64 or 128 channels, so 8 or 16 lanes take one, 16 bytes each, four
// rows in flight per lane, and the two sums of a row stay inside a group of 16 lanes.  (The library's LayerNorm gives each row
// a workgroup of one wave of which most lanes have nothing to do: B = 2, N = 1762, four heads of 64 channels 18.3 us for each
// of q and k in a kernel trace.)  Statistics in fp32 from the row in registers: the mean first, then the squares of
// the differences.
#include "paro_device.hpp"

namespace paro {

struct HeadNormParams {
  const unsigned short* x[2];
  unsigned short* out[2];
  const unsigned short *weight[2], *bias[2];   // null: one, zero
  float eps[2];
  int64_t rows;
};

// the sum over the LPR lanes that share a row, in all of them
template <int LPR> __device__ __forceinline__ float row_sum(float v) {
  v += row_dpp<0xB1>(v);    // lane ^ 1
  v += row_dpp<0x4E>(v);    // lane ^ 2
  v += row_dpp<0x141>(v);   // 7 - lane of eight
  if constexpr (LPR == 16) v += row_dpp<0x140>(v);   // 15 - lane of sixteen
  return v;
}

template <int DT, int D>
__global__ void __launch_bounds__(256) head_norm_kernel(const HeadNormParams p) {
  constexpr int LPR = D / 8, ROWS = 256 / LPR, U = 4;
  const int which = blockIdx.y, t = threadIdx.x, col = (t % LPR) * 8;
  const int64_t row0 = (int64_t)with_args(p, blockIdx.x) * (ROWS * U) + t / LPR;
  const unsigned short* x = p.x[which] + col;
  v4i raw[U];
#pragma unroll
  for (int u = 0; u < U; u++) raw[u] = *reinterpret_cast<const v4i*>(x + min(row0 + u * ROWS, p.rows - 1) * D);
  float w[8], b[8];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    w[j] = 1.f;
    b[j] = 0.f;
  }
  if (p.weight[which]) {
    const v4i r = *reinterpret_cast<const v4i*>(p.weight[which] + col);
#pragma unroll
    for (int j = 0; j < 8; j++) w[j] = elem16_to_f32<DT>(r, j);
  }
  if (p.bias[which]) {
    const v4i r = *reinterpret_cast<const v4i*>(p.bias[which] + col);
#pragma unroll
    for (int j = 0; j < 8; j++) b[j] = elem16_to_f32<DT>(r, j);
  }
  const float eps = p.eps[which];
#pragma unroll
  for (int u = 0; u < U; u++) {
    float f[8], s = 0.f, q = 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++) f[j] = elem16_to_f32<DT>(raw[u], j);
    s = ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
    const float mean = row_sum<LPR>(s) * (1.0f / D);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      f[j] -= mean;
      q = fmaf(f[j], f[j], q);
    }
    const float inv = 1.0f / sqrtf(row_sum<LPR>(q) * (1.0f / D) + eps);
    v4i o;
#pragma unroll
    for (int j = 0; j < 4; j++)
      o[j] = (int)pack2_from_f32<DT>(fmaf(f[2 * j] * inv, w[2 * j], b[2 * j]), fmaf(f[2 * j + 1] * inv, w[2 * j + 1], b[2 * j + 1]));
    const int64_t row = row0 + u * ROWS;
    if (row < p.rows) *reinterpret_cast<v4i*>(p.out[which] + row * D + col) = o;
  }
}

}  // namespace paro

extern "C" int paro_head_norm(const void* q, const void* k, void* q_out, void* k_out, int dtype, const void* q_weight,
                              const void* q_bias, const void* k_weight, const void* k_bias, float q_eps, float k_eps,
                              int64_t rows, int D, void* stream) {
  using namespace paro;
  PARO_CHECK(q && k && q_out && k_out, PARO_ERR_RUNTIME, "paro_head_norm: null tensor pointer");
  PARO_CHECK(D == 64 || D == 128, PARO_ERR_INVALID_VALUE, "Unsupported head dim: %d", D);
  PARO_CHECK(dtype == PARO_DTYPE_F16 || dtype == PARO_DTYPE_BF16, PARO_ERR_RUNTIME,
             "Unsupported input dtype (expect float16 or bfloat16)");
  const int per = 4 * 256 * 8 / D;   // rows a workgroup takes
  PARO_CHECK(rows > 0 && rows <= (int64_t)per * 0x7fffffff, PARO_ERR_RUNTIME, "paro_head_norm: %lld rows", (long long)rows);
  const void* ptrs[8] = {q, k, q_out, k_out, q_weight, q_bias, k_weight, k_bias};
  for (const void* ptr : ptrs)
    PARO_CHECK((uintptr_t)ptr % 16 == 0, PARO_ERR_RUNTIME, "paro_head_norm: tensors must be 16-byte aligned");
  HeadNormParams p;
  p.x[0] = (const unsigned short*)q; p.x[1] = (const unsigned short*)k;
  p.out[0] = (unsigned short*)q_out; p.out[1] = (unsigned short*)k_out;
  p.weight[0] = (const unsigned short*)q_weight; p.weight[1] = (const unsigned short*)k_weight;
  p.bias[0] = (const unsigned short*)q_bias; p.bias[1] = (const unsigned short*)k_bias;
  p.eps[0] = q_eps; p.eps[1] = k_eps;
  p.rows = rows;
  const dim3 grid((unsigned)((rows + per - 1) / per), 2);
  hipStream_t st = (hipStream_t)stream;
  if (dtype == PARO_DTYPE_F16) {
    if (D == 64) hipLaunchKernelGGL((head_norm_kernel<PARO_DTYPE_F16, 64>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((head_norm_kernel<PARO_DTYPE_F16, 128>), grid, dim3(256), 0, st, p);
  } else {
    if (D == 64) hipLaunchKernelGGL((head_norm_kernel<PARO_DTYPE_BF16, 64>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((head_norm_kernel<PARO_DTYPE_BF16, 128>), grid, dim3(256), 0, st, p);
  }
  PARO_HIP(hipGetLastError());
  return PARO_OK;
}
