// Which heads of a block mask have neighbouring q-blocks that keep the same key blocks, so that the pair kernel
// (attn_sparse.hip) takes them: looked up on the device, where the mask is.  gfx950 only.
#pragma once
#include "paro_common.hpp"

namespace paro {

struct ShareLook {
  const uint8_t* mask;     // [batch][H][nbq][nbk] bytes
  int64_t batch_stride;
  int H, heads;            // heads of the mask: B * H, or H where one mask serves every batch entry
  int nbq, nbk, causal;
  int* share;              // [heads], 1 or 0
};

constexpr int SHARE_THREADS = 256;

// One workgroup (SHARE_THREADS threads or more) per head: 32 columns each of 256 pairs of neighbouring rows.  With U blocks in
// the union of a pair and S in its two lists the pair kernel does the work of 2 U blocks at 0.90 of the time of one (B = 2,
// H = 32, N = 8192, causal: U / S = 0.75 370 / 502 us, 0.5 616 / 573), so that the lines cross at U / S = 0.55; 0.54
// leaves the plain kernel what the sample's noise, 0.005, could get wrong.
__device__ __forceinline__ void share_look(const ShareLook& p, int head) {
  const int t = threadIdx.x, pairs = p.nbq >> 1;   // (pairs of rows that both exist)
  int u = 0, s = 0;
  if (t < SHARE_THREADS && pairs > 0) {
    const int pair = t * pairs / SHARE_THREADS;
    const int cols = p.causal ? min(p.nbk, 2 * pair + 2) : p.nbk;
    if (cols >= 8) {
      const uint8_t* a = p.mask + head / p.H * p.batch_stride + ((int64_t)(head % p.H) * p.nbq + 2 * pair) * p.nbk;
      unsigned seed = (unsigned)t * 2654435761u + 12345u;
      uint64_t xa[4], xb[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        seed = seed * 1664525u + 1013904223u;
        const int c = (int)__umulhi(seed, (unsigned)(cols - 7));
        __builtin_memcpy(&xa[i], a + c, 8);
        __builtin_memcpy(&xb[i], a + p.nbk + c, 8);
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        // (a byte that is not zero -> its top bit)
        const uint64_t low = 0x7f7f7f7f7f7f7f7full;
        const uint64_t ma = (((xa[i] & low) + low) | xa[i]) & ~low, mb = (((xb[i] & low) + low) | xb[i]) & ~low;
        u += __popcll(ma | mb);
        s += __popcll(ma) + __popcll(mb);
      }
    }
  }
  int both = u | (s << 16);   // (at most 2^13 and 2^14)
#pragma unroll
  for (int i = 1; i < 64; i *= 2) both += __shfl_xor(both, i, 64);
  __shared__ int sums[SHARE_THREADS / 64];
  if (t < SHARE_THREADS && (t & 63) == 0) sums[t >> 6] = both;
  __syncthreads();
  if (t == 0) {
    both = sums[0] + sums[1] + sums[2] + sums[3];
    u = both & 0xffff;
    s = both >> 16;
    p.share[head] = s >= 64 && u * 50 <= s * 27;
  }
}

}  // namespace paro
