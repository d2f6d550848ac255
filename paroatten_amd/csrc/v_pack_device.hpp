// Bodies of the two V conversions as device functions (v_fp8.hip, attn_sparse_pv16.hip: V alone; attn_operator.hip:
// next to the quantisation of K, or of Q and K, in one launch).  256 threads take one 64-token block kb of (batch, kv-head)
// bh; v points at the first token of that (batch, kv-head).
#pragma once
#include "paro_device.hpp"

namespace paro {

// FP8 tiles.  work: the work buffer of the V conversion (v_recp_offset); resid (may be null): its second part.
template <int DT, int D>
__device__ __forceinline__ void v_pack_body(const unsigned short* __restrict__ v, uint8_t* __restrict__ v8,
                                            const float* __restrict__ work, const float* __restrict__ v_mean,
                                            float* __restrict__ resid, int N, int nb, int64_t vs_n, int kb, int64_t bh) {
  constexpr int LPR = D / 8;
  constexpr int ROWS = 256 / LPR;
  constexpr int PITCH = D + 8;  // 16-bit elements; +16 bytes keeps rows on different banks
  __shared__ __attribute__((aligned(16))) unsigned short tile[64 * PITCH];
  const int t = threadIdx.x;
  const int col = (t % LPR) * 8;
  const unsigned short* vb = v + col;
#pragma unroll
  for (int r = t / LPR; r < 64; r += ROWS) {
    const int tok = kb * 64 + r;
    const v4i raw = (tok < N) ? __builtin_nontemporal_load(reinterpret_cast<const v4i*>(vb + (int64_t)tok * vs_n))
                              : v4i{0, 0, 0, 0};
    *reinterpret_cast<v4i*>(&tile[r * PITCH + col]) = raw;
  }
  __syncthreads();
  float rs[D / 64];
  pack_v_tile<DT, D, PITCH>(tile, v8 + (bh * nb + kb) * (int64_t)(64 * D), work + v_recp_offset(bh, N, D),
                            v_mean ? v_mean + bh * D : nullptr, kb * 64, N, t, rs);
  if (resid != nullptr && (t & 63) < 32) {
    const int wave = t >> 6;
#pragma unroll
    for (int n = 0; n < D / 64; n++)
      resid[((bh * nb + kb) * 2 + (wave & 1)) * D + 32 * ((wave >> 1) + 2 * n) + (t & 31)] = rs[n];
  }
}

// One block, in LDS as rows of D + 8 elements, as a float16 tile: 256 threads.
template <int DT, int D>
__device__ __forceinline__ void v_f16_store_tile(const unsigned short* tile, unsigned short* __restrict__ dst, int t) {
#pragma unroll
  for (int pl = t; pl < (D / 32) * 4 * 64; pl += 256) {
    const int lane = pl & 63, piece = pl >> 6;
    const int dt = piece >> 2, s = piece & 3;
    const int chn = 32 * dt + (lane & 31);
    unsigned short r[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const int row = 32 * (s >> 1) + 16 * (s & 1) + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
      const unsigned short raw = tile[row * (D + 8) + chn];
      r[e] = DT == PARO_DTYPE_F16 ? raw : F16x<PARO_DTYPE_F16>::from_f32(F16x<PARO_DTYPE_BF16>::to_f32(raw));
    }
    *reinterpret_cast<v4i*>(dst + (int64_t)pl * 8) =
        v4i{(int)(r[0] | ((unsigned)r[1] << 16)), (int)(r[2] | ((unsigned)r[3] << 16)),
            (int)(r[4] | ((unsigned)r[5] << 16)), (int)(r[6] | ((unsigned)r[7] << 16))};
  }
}

// Its way there: 256 threads, rows past the end are zero.
template <int D>
__device__ __forceinline__ void v_f16_load_tile(const unsigned short* __restrict__ v, unsigned short* tile, int N, int64_t vs_n,
                                                int kb, int t) {
  constexpr int CPR = D / 8;   // 16-byte chunks per row
#pragma unroll
  for (int c = t; c < 64 * CPR; c += 256) {
    const int row = c / CPR, ch = c % CPR;
    const int tok = kb * 64 + row;
    v4i x = {0, 0, 0, 0};
    if (tok < N) x = *reinterpret_cast<const v4i*>(v + (int64_t)tok * vs_n + ch * 8);
    *reinterpret_cast<v4i*>(tile + row * (D + 8) + ch * 8) = x;
  }
}

// float16 tiles: the block goes through LDS row by row (16-byte loads) and leaves as D/32 x 4 pieces of 1 KB (16 bytes
// per lane).
template <int DT, int D>
__device__ __forceinline__ void v_f16_pack_body(const unsigned short* __restrict__ v, unsigned short* __restrict__ out,
                                                int N, int nb, int64_t vs_n, int kb, int64_t bh) {
  __shared__ __attribute__((aligned(16))) unsigned short tile[64 * (D + 8)];   // rows padded by 16 bytes
  v_f16_load_tile<D>(v, tile, N, vs_n, kb, threadIdx.x);
  __syncthreads();
  v_f16_store_tile<DT, D>(tile, out + (bh * nb + kb) * (64 * D), threadIdx.x);
}

}  // namespace paro
