// Statistics passes of the path as device functions, so that one launch can run several of them side by side:
// per-channel sum / min / max of V (for the FP8 scale and mean) and the mean of the rotated K (for K smoothing).
// The launches that use them: v_fp8.hip (V alone), fused_prep.hip (K alone, or K and V in one launch).
#pragma once
#include "paro_device.hpp"
#include <type_traits>

namespace paro {

// Per-channel sum, minimum and maximum of one v_chunk(N)-token chunk of one (batch, head): 256 threads.  Rows are
// requested in batches of eight, in the last chunk too (rows past the end re-read the last one and are not taken): a
// row at a time, the 738 rows of the last of two chunks took 15.7 us at N = 1762, B = 2, H = 4, D = 64.
// SUM_ONLY: only the sums, [chunk][D] (the mean of an unrotated K).
template <int DT, int D, bool SUM_ONLY = false>
__device__ __forceinline__ void v_stats_body(const unsigned short* __restrict__ v, float* __restrict__ partial, int N,
                                             int n_chunks, int64_t vs_b, int64_t vs_h, int64_t vs_n, int chunk, int h,
                                             int b, int H) {
  constexpr int LPR = D / 8;
  constexpr int ROWS = 256 / LPR;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int col = (t % LPR) * 8;
  const unsigned short* vb = v + b * vs_b + h * vs_h + col;
  float s[8], mn[8], mx[8];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    s[j] = 0.f;
    mn[j] = INFINITY;
    mx[j] = -INFINITY;
  }
  auto take = [&](const v4i raw) {
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const float f = elem16_to_f32<DT>(raw, j);
      s[j] += f;
      if constexpr (!SUM_ONLY) {
        mn[j] = fminf(mn[j], f);
        mx[j] = fmaxf(mx[j], f);
      }
    }
  };
  const int len = v_chunk(N), first = chunk * len, tok0 = first + t / LPR;
  constexpr int VS_BATCH = 8;
  // SUM_ONLY: the eight rows of a batch pairwise, so that a chunk of 1024 tokens has four additions in a row instead of 32.
  // With the chunk sums added up in fp64 the mean of 8192 tokens is 2.7e-8 off before its rounding to 16 bits instead of
  // 6.4e-8 (library reduction 3.7e-8), in the same time
  auto take_sums = [&](const v4i (&raw)[VS_BATCH], int r) {
#pragma unroll
    for (int j = 0; j < 8; j++) {
      float f[VS_BATCH];
#pragma unroll
      for (int u = 0; u < VS_BATCH; u++) f[u] = tok0 + r + u * ROWS < N ? elem16_to_f32<DT>(raw[u], j) : 0.f;
      s[j] += ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
    }
  };
  auto walk = [&](auto whole) {
    for (int r = 0; r < len; r += ROWS * VS_BATCH) {
      if (!decltype(whole)::value && first + r >= N) break;
      v4i raw[VS_BATCH];
#pragma unroll
      for (int u = 0; u < VS_BATCH; u++) {
        // (non-temporal: measured 3-5 us faster per launch of the entry point and of the per-layer sequence
        // than ordinary loads, although the packing pass reads the same tensor right afterwards)
        const int tok = tok0 + r + u * ROWS;
        const v4i* src = reinterpret_cast<const v4i*>(vb + (int64_t)(decltype(whole)::value ? tok : min(tok, N - 1)) * vs_n);
        raw[u] = SUM_ONLY ? *src : __builtin_nontemporal_load(src);
      }
      if constexpr (SUM_ONLY) {
        take_sums(raw, r);
        continue;
      }
#pragma unroll
      for (int u = 0; u < VS_BATCH; u++)
        if (decltype(whole)::value || tok0 + r + u * ROWS < N) take(raw[u]);
    }
  };
  if (first + len <= N) walk(std::true_type{});
  else walk(std::false_type{});
  // lanes that share a column sit LPR apart: 8 lanes round the row (D = 64 only), then lane ^ 16, ^ 32
#pragma unroll
  for (int j = 0; j < 8; j++) {
    float a, b;
    if constexpr (LPR == 8) {
      s[j] += row_dpp<0x128>(s[j]);
      if constexpr (!SUM_ONLY) {
        mn[j] = fminf(mn[j], row_dpp<0x128>(mn[j]));
        mx[j] = fmaxf(mx[j], row_dpp<0x128>(mx[j]));
      }
    }
    with_lane_xor16(s[j], a, b);  s[j] = a + b;
    if constexpr (SUM_ONLY) {
      with_lane_xor32(s[j], a, b);  s[j] = a + b;
      continue;
    }
    with_lane_xor16(mn[j], a, b); mn[j] = fminf(a, b);
    with_lane_xor16(mx[j], a, b); mx[j] = fmaxf(a, b);
    with_lane_xor32(s[j], a, b);  s[j] = a + b;
    with_lane_xor32(mn[j], a, b); mn[j] = fminf(a, b);
    with_lane_xor32(mx[j], a, b); mx[j] = fmaxf(a, b);
  }
  __shared__ float red[4][SUM_ONLY ? 1 : 3][D];
  if (lane < LPR) {
#pragma unroll
    for (int j = 0; j < 8; j++) {
      red[wave][0][col + j] = s[j];
      if constexpr (!SUM_ONLY) {
        red[wave][1][col + j] = mn[j];
        red[wave][2][col + j] = mx[j];
      }
    }
  }
  __syncthreads();
  if (t < D) {
    const float ss = (red[0][0][t] + red[1][0][t]) + (red[2][0][t] + red[3][0][t]);
    if constexpr (SUM_ONLY) {
      partial[((int64_t)(b * H + h) * n_chunks + chunk) * D + t] = ss;
      return;
    }
    constexpr int MN = SUM_ONLY ? 0 : 1, MX = SUM_ONLY ? 0 : 2;
    const float mm = fminf(fminf(red[0][MN][t], red[1][MN][t]), fminf(red[2][MN][t], red[3][MN][t]));
    const float xx = fmaxf(fmaxf(red[0][MX][t], red[1][MX][t]), fmaxf(red[2][MX][t], red[3][MX][t]));
    float* p = partial + (((int64_t)(b * H + h) * n_chunks + chunk) * 3) * D;
    p[t] = ss;
    p[D + t] = mm;
    p[2 * D + t] = xx;
  }
}


// mean, scale and reciprocal scale of one (batch, head) from its chunk statistics: 1024 threads.  `work`: the work
// buffer of the V conversion (v_stats_offset, v_recp_offset).
template <int D>
__device__ __forceinline__ void v_finalize_body(float* work, float* __restrict__ v_scale, float* __restrict__ v_mean,
                                                int N, int n_chunks, int smooth, int64_t bh, int64_t BH) {
  // 1024 / D slices of the chunk range per channel, combined through LDS in a fixed order.  The sums of short chunks are
  // four times as many: added up in fp32 the mean of 8192 tokens was up to 1.4 times as far from 64 bits as with long
  // chunks, in fp64 it is nearer
  constexpr int SL = 1024 / D;
  __shared__ double red_s[SL][D];
  __shared__ float red[2][SL][D];
  const bool wide = v_chunk(N) != V_CHUNK;
  auto add = [wide](double a, double b) { return wide ? a + b : (double)((float)a + (float)b); };
  const int ch = threadIdx.x % D, sl = threadIdx.x / D;
  const float* p = work + v_stats_offset(BH, N, D) + bh * n_chunks * 3 * D;
  double s = 0.0;
  float mn = INFINITY, mx = -INFINITY;
  for (int c = sl; c < n_chunks; c += SL) {
    s = add(s, p[(c * 3 + 0) * D + ch]);
    mn = fminf(mn, p[(c * 3 + 1) * D + ch]);
    mx = fmaxf(mx, p[(c * 3 + 2) * D + ch]);
  }
  red_s[sl][ch] = s;
  red[0][sl][ch] = mn;
  red[1][sl][ch] = mx;
  __syncthreads();
  if (sl == 0) {
    for (int i = 1; i < SL; i++) {
      s = add(s, red_s[i][ch]);
      mn = fminf(mn, red[0][i][ch]);
      mx = fmaxf(mx, red[1][i][ch]);
    }
    const float mean = !smooth ? 0.f : wide ? (float)(s / (double)N) : (float)s / (float)N;
    const float amax = fmaxf(mx - mean, mean - mn);
    v_scale[bh * D + ch] = amax / 448.0f;
    if (v_mean) v_mean[bh * D + ch] = mean;
    // (long chunks: the partials of this (batch, head) are in the same place; every thread of the workgroup has read
    // its own before the barrier above)
    work[v_recp_offset(bh, N, D) + ch] = amax > 0.f ? 448.0f / amax : 0.f;
    work[v_recp_offset(bh, N, D) + D + ch] = mean;
  }
}


// K mean over tokens AFTER the rotation (the permutation does not change a mean): partial sums per
// K_CHUNK-token chunk, then one workgroup per (batch, head) adds them in a fixed order.  A thread keeps
// the table entries of its token piece while it walks over a group of (batch, head) pairs.
constexpr int KM_GROUP = 4;   // measured: 4 beats 8 (too few workgroups at 40 heads) and 2 (tables re-read twice as often)
template <int DT, int D, int KB, int GROUP>
__device__ __forceinline__ void rope_k_sum_body(const unsigned short* __restrict__ k, const float* __restrict__ cos_t,
                                                const float* __restrict__ sin_t, float* __restrict__ partial, int BH,
                                                int H, int N, int n_text, int n_chunks, int64_t ks_b, int64_t ks_h,
                                                int64_t ks_n, int chunk, int bh0) {
  constexpr int LPR = D / 8;
  constexpr int ROWS = 256 / LPR;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int col = (t % LPR) * 8;
  float s[GROUP][8];
#pragma unroll
  for (int g = 0; g < GROUP; g++)
#pragma unroll
    for (int j = 0; j < 8; j++) s[g][j] = 0.f;
  // one step: the rows of one token of the group's heads (table entries first: they are shared by the heads)
  auto add_rows = [&](const v4i (&raw)[GROUP], bool rot, const v4f& c0, const v4f& c1, const v4f& s0, const v4f& s1) {
    float cs[8], sn[8];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      cs[j] = c0[j]; cs[4 + j] = c1[j];
      sn[j] = s0[j]; sn[4 + j] = s1[j];
    }
#pragma unroll
    for (int g = 0; g < GROUP; g++) {
      const v4i x = rot ? rotate8<DT>(raw[g], cs, sn) : raw[g];
#pragma unroll
      for (int j = 0; j < 8; j++) s[g][j] += elem16_to_f32<DT>(x, j);
    }
  };
  const int tok_first = chunk * K_CHUNK;
  // batches of KB tokens per thread: their table pieces and K rows are all requested before the first is used
  // (ordinary loads for K: it was just written by the projection and is read again by the preparation pass).
  // `whole`: every row and head is there and every row rotated alike; otherwise rows and heads past the end re-read
  // the last one, such rows are not added and such heads not stored, and a row says for itself whether it is rotated
  const bool tables = cos_t != nullptr;
  const unsigned short* kp[GROUP];
#pragma unroll
  for (int g = 0; g < GROUP; g++) {
    const int bh = min(bh0 + g, BH - 1), b = bh / H, h = bh - b * H;
    kp[g] = k + b * ks_b + h * ks_h + col;
  }
  auto walk = [&](auto whole_c) {
    constexpr bool whole = decltype(whole_c)::value;
    for (int r = t / LPR; r < K_CHUNK; r += ROWS * KB) {
      if (!whole && tok_first + (r - t / LPR) >= N) break;
      v4f c0[KB], c1[KB], s0[KB], s1[KB];
      v4i raw[KB][GROUP];
#pragma unroll
      for (int u = 0; u < KB; u++) {
        const int tok = whole ? tok_first + r + u * ROWS : min(tok_first + r + u * ROWS, N - 1);
        if (tables) {
          const int64_t o = (int64_t)(whole ? tok - n_text : max(tok - n_text, 0)) * D + col;
          c0[u] = *reinterpret_cast<const v4f*>(cos_t + o); c1[u] = *reinterpret_cast<const v4f*>(cos_t + o + 4);
          s0[u] = *reinterpret_cast<const v4f*>(sin_t + o); s1[u] = *reinterpret_cast<const v4f*>(sin_t + o + 4);
        }
#pragma unroll
        for (int g = 0; g < GROUP; g++) raw[u][g] = *reinterpret_cast<const v4i*>(kp[g] + (int64_t)tok * ks_n);
      }
#pragma unroll
      for (int u = 0; u < KB; u++) {
        const int tok = tok_first + r + u * ROWS;
        if (whole || tok < N) add_rows(raw[u], tables && (whole || tok >= n_text), c0[u], c1[u], s0[u], s1[u]);
      }
    }
  };
  if (tok_first + K_CHUNK <= N && bh0 + GROUP <= BH && (!tables || tok_first >= n_text)) walk(std::true_type{});
  else walk(std::false_type{});
  __shared__ float red[4][GROUP][D];
#pragma unroll
  for (int g = 0; g < GROUP; g++) {
    // lanes that share a column sit LPR apart
#pragma unroll
    for (int j = 0; j < 8; j++) {
      float a, b;
      if constexpr (LPR == 8) s[g][j] += row_dpp<0x128>(s[g][j]);
      with_lane_xor16(s[g][j], a, b);
      s[g][j] = a + b;
      with_lane_xor32(s[g][j], a, b);
      s[g][j] = a + b;
    }
    if (lane < LPR) {
#pragma unroll
      for (int j = 0; j < 8; j++) red[wave][g][col + j] = s[g][j];
    }
  }
  __syncthreads();
  for (int i = t; i < GROUP * D; i += 256) {
    const int g = i / D, ch = i % D;
    if (bh0 + g < BH)
      partial[((int64_t)(bh0 + g) * n_chunks + chunk) * D + ch] =
          (red[0][g][ch] + red[1][g][ch]) + (red[2][g][ch] + red[3][g][ch]);
  }
}

// k_mean[b,h,:] = (sum of the chunk sums, in a fixed order) / N, rounded to the input dtype: 1024 threads.  Acc: what the
// chunk sums are added up in.
template <int DT, int D, typename Acc = float>
__device__ __forceinline__ void k_mean_finalize_body(const float* __restrict__ partial,
                                                     unsigned short* __restrict__ k_mean, int N, int n_chunks,
                                                     int64_t ms_b, int64_t ms_h, int H, int64_t bh) {
  constexpr int SL = 1024 / D;
  __shared__ Acc red[SL][D];
  const int ch = threadIdx.x % D, sl = threadIdx.x / D;
  const float* p = partial + bh * n_chunks * D;
  Acc s = 0;
  // (batches of independent loads: as a plain loop every load waited for the one before it)
  constexpr int FB = 8;
  int c = sl;
  for (; c + (FB - 1) * SL < n_chunks; c += FB * SL) {
    float x[FB];
#pragma unroll
    for (int u = 0; u < FB; u++) x[u] = p[(c + u * SL) * D + ch];
#pragma unroll
    for (int u = 0; u < FB; u++) s += x[u];
  }
  for (; c < n_chunks; c += SL) s += p[c * D + ch];
  red[sl][ch] = s;
  __syncthreads();
  if (sl == 0) {
    for (int i = 1; i < SL; i++) s += red[i][ch];
    const int b = (int)(bh / H), h = (int)(bh % H);
    k_mean[b * ms_b + h * ms_h + ch] = (unsigned short)(pack2_from_f32<DT>((float)(s / (Acc)N), 0.f) & 0xffffu);
  }
}

}  // namespace paro
