// The whole attention operator on 16-bit q, k, v in one call: INT8 quantisation of Q and K (K's token mean taken off
// first if asked for), the V conversion, block-sparse attention.  Two to five launches:
//   op_stats     K sums (smooth_k) and V statistics (FP8 product), side by side
//   op_finalize  their second steps
//   op_prep      quantised K and the V tiles, side by side (op_q_pass: quantised Q too)
//   v_residual   (FP8 product with smooth_v; up to 4096 keys and with few q-blocks the attention launch does it: split_takes_residual)
//   attention    on 16-bit Q, which the q-block's own waves quantise (QRows; op_q_pass: on INT8 Q); the
//                log-sum-exp leaves as the natural one of the scores of q and k as given
// Short sequences take one launch for the first four (op_head: up to 1024 tokens, as many heads as op_head_plan says) or one for
// the second and third (op_prep_short: the rest up to 4096 tokens, op_short).  Calls with nothing to sum up (float16 product
// without smooth_k) have op_prep and the attention alone, and those with per-thread scales all five.
// The first four are bound by HBM where they are long: at B = 2, H = 48, N = 17776, D = 64 they move 16-bit K and V twice and write their 8-bit
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
  float* lse_add;               // with a pass over Q: sm_scale * q . k_mean per row; nullptr: not wanted
  int B, H, Hkv, Nq, Nk, nbq, nbk, chunks, smooth_v;
  int stats_k, stats_v;         // which statistics are taken
  int kv_blocks;                // workgroups of op_prep that take K or V; the rest (q_pass) take Q
  float sm_scale;
  bool q_pass;                  // op_prep quantises Q too (op_q_pass)
  bool one_launch;              // op_head does it all (op_head_plan)
  int k_parts, k_rounds;        // of op_head: workgroups that share the K of a head, 256 tokens they take one after the other
  bool short_prep;              // op_prep_short does what comes after the statistics (op_short)
};

template <int DT, int D>
__global__ void __launch_bounds__(256) op_stats_kernel(const OpParams p) {
  // K and V of a head one after the other, in x: y and z keep the whole range of head and batch counts
  const int h = blockIdx.y, b = blockIdx.z, block = with_args(p, blockIdx.x);
  const int k_chunks = p.stats_k ? p.chunks : 0;
  if (block < k_chunks)
    v_stats_body<DT, D, true>(p.k, p.k_partial, p.Nk, p.chunks, p.ks_b, p.ks_h, p.ks_n, block, h, b, p.Hkv);
  else
    v_stats_body<DT, D>(p.v, p.v_work + v_stats_offset((int64_t)p.B * p.Hkv, p.Nk, D), p.Nk, p.chunks, p.vs_b, p.vs_h,
                        p.vs_n, block - k_chunks, h, b, p.Hkv);
}

template <int DT, int D>
__global__ void __launch_bounds__(1024) op_finalize_kernel(const OpParams p) {
  const int BH = p.B * p.Hkv, block = with_args(p, blockIdx.x);
  if (block < BH * p.stats_k)
    k_mean_finalize_body<DT, D, double>(p.k_partial, p.k_mean, p.Nk, p.chunks, (int64_t)p.Hkv * D, D, p.Hkv, block);
  else
    v_finalize_body<D>(p.v_work, p.v_scale, p.v_mean, p.Nk, p.chunks, p.smooth_v, (int64_t)block - BH * p.stats_k, BH);
}

// PT: per-thread scale granularity.  A workgroup takes one V tile, 256 tokens of K or 128 (PT: 256) tokens of Q.
template <int DT, int D, bool PT, bool F16V>
__global__ void __launch_bounds__(256) op_prep_kernel(const OpParams p) {
  const int wave = threadIdx.x >> 6;
  int i = with_args(p, blockIdx.x);
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
  i -= p.kv_blocks;
  const int groups = PT ? p.nbq : 2 * p.nbq;   // of 64 or 32 tokens
  const int per = (groups + 3) / 4, bh = i / per, g = i % per * 4 + wave;
  if (g >= groups) return;
  const int b = bh / p.H, h = bh % p.H;
  const unsigned short* q = p.q + b * p.qs_b + h * p.qs_h;
  int8_t* out = p.q8 + (int64_t)bh * p.Nq * D;
  float* dot = p.lse_add ? p.lse_add + (int64_t)bh * p.Nq : nullptr;
  const unsigned short* with = p.lse_add ? p.k_mean + ((int64_t)b * p.Hkv + h / (p.H / p.Hkv)) * D : nullptr;
  if constexpr (PT)
    quant_per_thread_body<DT, D, false, false>(q, nullptr, out, p.q_scale + (int64_t)bh * p.nbq * 16, p.Nq, g, p.qs_n, D, p.sm_scale,
                                               dot, with);
  else
    quant_group_body<DT, D, 32, false, false>(q, nullptr, out, p.q_scale + (int64_t)bh * p.nbq * 2, p.Nq, g, p.qs_n, D, p.sm_scale,
                                              dot, with);
}

// Everything in front of the attention launch, up to OP_HEAD_TOKENS tokens, in one launch: such a call consists of launches of
// a few microseconds that wait for each other, not of bytes.  Workgroups of 16 waves that need nothing of each other:
//   V: 32 channels of a (batch, kv-head) over all tokens, read once and kept in LDS for the statistics and the codes.  A lane
//      has two channels of four neighbouring tokens, which are a word of the tiles each.
//   K: four 64-token groups, four waves to each; with smooth_k every workgroup takes the mean over all tokens for itself.
// What bounds it is the vector work and the latencies of one compute unit: with one workgroup to K and one to V of a head the
// launch took 4.7 us longer at N = 416, D = 64, two heads, for adding up across lanes and for the codes of V; this way it
// is 7.1 us (6.6 at the least) in a kernel trace.  The operator, start to end, separate launches / this one, smooth_k, us:
//   D = 64   N = 416   2 heads 19.4 / 13.2   16 heads 20.7 / 13.4     D = 128  N = 512   8 heads 24.9 / 18.4   48 heads 31.5 / 26.0
//            N = 1024  8 heads 22.6 / 19.9   48 heads 29.6 / 24.6              N = 1024  8 heads 29.4 / 25.2   24 heads 34.0 / 31.5
// (which calls: op_head_plan)
constexpr int OP_HEAD_TOKENS = 1024;

template <int DT, int D, bool F16V>
__global__ void __launch_bounds__(1024) op_head_kernel(const OpParams p) {
  constexpr int LPR = D / 8;                // lanes per token row (K)
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int k_parts = p.k_parts, parts = k_parts + (F16V ? (p.nbk + 3) / 4 : D / 32);
  const int block = with_args(p, blockIdx.x), bh = block / parts, b = bh / p.Hkv, h = bh % p.Hkv;
  int part = block % parts;
  const int N = p.Nk;
  constexpr int V_BYTES = F16V ? 4 * 64 * (D + 8) * 2 : OP_HEAD_TOKENS * 64 + 32 * 3 * 32 * 4 + 2 * 32 * 4;
  constexpr int K_BYTES = 16 * D * 4 + D * 2 + 2 * 16 * 4;
  __shared__ __attribute__((aligned(16))) uint8_t smem[V_BYTES > K_BYTES ? V_BYTES : K_BYTES];

  if (part < k_parts) {
    constexpr int RPI = 64 / LPR, CH = 16 / RPI;   // rows per load, loads per lane of a wave's 16 rows
    constexpr int ROWS = 1024 / LPR, BATCH = 8;
    const int col = (lane % LPR) * 8;
    const unsigned short* k = p.k + b * p.ks_b + h * p.ks_h + col;
    int grp = part * 4 * p.k_rounds + (wave >> 2);
    v4i raw[CH];
    auto load = [&]() {
#pragma unroll
      for (int i = 0; i < CH; i++) {
        const int tok = grp * 64 + (wave & 3) * 16 + lane / LPR + i * RPI;
        raw[i] = tok < N ? *reinterpret_cast<const v4i*>(k + (int64_t)tok * p.ks_n) : v4i{0, 0, 0, 0};
      }
    };
    load();
    float mv[8] = {};
    if (p.stats_k) {
      auto* red = reinterpret_cast<float(*)[D]>(smem);
      unsigned short* mean = reinterpret_cast<unsigned short*>(smem + 16 * D * 4);
      float s[8] = {};
      for (int r = t / LPR; r < N; r += ROWS * BATCH) {
        v4i x[BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; u++)
          x[u] = *reinterpret_cast<const v4i*>(k + (int64_t)min(r + u * ROWS, N - 1) * p.ks_n);
#pragma unroll
        for (int j = 0; j < 8; j++) {
          float f[BATCH];
#pragma unroll
          for (int u = 0; u < BATCH; u++) f[u] = r + u * ROWS < N ? elem16_to_f32<DT>(x[u], j) : 0.f;
          s[j] += ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
        }
      }
#pragma unroll
      for (int j = 0; j < 8; j++) {
        float a, c;
        if constexpr (LPR == 8) s[j] += row_dpp<0x128>(s[j]);
        with_lane_xor16(s[j], a, c);
        s[j] = a + c;
        with_lane_xor32(s[j], a, c);
        s[j] = a + c;
      }
      if (lane < LPR) {
#pragma unroll
        for (int j = 0; j < 8; j++) red[wave][col + j] = s[j];
      }
      __syncthreads();
      if (t < D) {
        double sum = 0.0;
#pragma unroll
        for (int w = 0; w < 16; w++) sum += red[w][t];
        mean[t] = (unsigned short)(pack2_from_f32<DT>((float)(sum / (double)N), 0.f) & 0xffffu);
        if (part == 0) p.k_mean[(int64_t)bh * D + t] = mean[t];
      }
      __syncthreads();
      load8_f32<DT>(mean + col, mv);
    }
    // (the rest is quant_group_body, with the maximum of four waves)
    auto* gmax = reinterpret_cast<float(*)[16]>(smem + 16 * D * 4 + D * 2);
    int8_t* out = p.k8 + (int64_t)bh * N * D + col;
    for (int r = 0; r < p.k_rounds; r++) {
      const int tok0 = grp * 64 + (wave & 3) * 16 + lane / LPR;
      float amax = 0.0000001f;
#pragma unroll
      for (int i = 0; i < CH; i++)
        if (tok0 + i * RPI < N) {
#pragma unroll
          for (int j = 0; j < 8; j++) amax = fmaxf(amax, fabsf(elem16_to_f32<DT>(raw[i], j) - mv[j]));
        }
      float* gm = gmax[r & 1];   // (a wave may be one round ahead of the others, not two)
      gm[wave] = wave_max(amax);
      __syncthreads();
      const int w0 = wave & ~3;
      amax = fmaxf(fmaxf(gm[w0], gm[w0 + 1]), fmaxf(gm[w0 + 2], gm[w0 + 3]));
      if (t % 256 == 0 && grp < p.nbk) p.k_scale[(int64_t)bh * p.nbk + grp] = amax / 127.0f;
      const float inv = 127.0f / amax;
#pragma unroll
      for (int i = 0; i < CH; i++) {
        const int tok = tok0 + i * RPI;
        float y[8];
#pragma unroll
        for (int j = 0; j < 8; j++) y[j] = (elem16_to_f32<DT>(raw[i], j) - mv[j]) * inv;
        if (tok < N)
          *reinterpret_cast<v2i*>(out + (int64_t)tok * D) =
              v2i{(int)pack4_rint_i8(y[0], y[1], y[2], y[3]), (int)pack4_rint_i8(y[4], y[5], y[6], y[7])};
      }
      grp += 4;
      if (r + 1 < p.k_rounds) load();
    }
    return;
  }
  part -= k_parts;

  if constexpr (F16V) {
    auto* tiles = reinterpret_cast<unsigned short(*)[64 * (D + 8)]>(smem);
    const int g = t >> 8, tg = t & 255, kb = part * 4 + g;
    const unsigned short* v = p.v + b * p.vs_b + h * p.vs_h;
    v_f16_load_tile<D>(v, tiles[g], N, p.vs_n, kb, tg);
    __syncthreads();
    if (kb < p.nbk) v_f16_store_tile<DT, D>(tiles[g], (unsigned short*)p.v_tiles + ((int64_t)bh * p.nbk + kb) * (64 * D), tg);
  } else {
    // The 32 channels go to LDS once, four tokens of 64 bytes to a group; token q of group a lies at place q ^ (a / 2 % 4), so
    // that both the statistics (four tokens of a group at a time) and the codes (the same token of every other group) read
    // each bank once.  Sums are taken in the order of v_stats_body, v_finalize_body, pack_v_tile and v_residual, to the bit.
    auto* red = reinterpret_cast<float(*)[3][32]>(smem + OP_HEAD_TOKENS * 64);          // [chunk][group][3][32]
    auto* resid = reinterpret_cast<float(*)[2][32]>(smem + OP_HEAD_TOKENS * 64);        // (later) [row tile][lane half][32]
    auto* chan = reinterpret_cast<float(*)[32]>(smem + OP_HEAD_TOKENS * 64 + 32 * 3 * 32 * 4);   // reciprocal scale, mean
    constexpr int U = D / 8, GROUPS = 64 / U;   // tokens that v_stats_body adds up one after the other; groups of four such rows
    const unsigned short* v = p.v + b * p.vs_b + h * p.vs_h + 32 * part;
    v4i raw[OP_HEAD_TOKENS / 256];
#pragma unroll
    for (int i = 0; i < OP_HEAD_TOKENS / 256; i++) {
      const int tok = t / 4 + 256 * i;
      raw[i] = tok < N ? *reinterpret_cast<const v4i*>(v + (int64_t)tok * p.vs_n + t % 4 * 8) : v4i{0, 0, 0, 0};
    }
    auto at = [&](int group, int q) { return smem + group * 256 + ((q ^ (group >> 1)) & 3) * 64; };
#pragma unroll
    for (int i = 0; i < OP_HEAD_TOKENS / 256; i++) {
      const int tok = t / 4 + 256 * i;
      *reinterpret_cast<v4i*>(at(tok >> 2, tok & 3) + t % 4 * 16) = raw[i];
    }
    __syncthreads();
    const int cp = 2 * (lane & 15);
    for (int sc = wave; sc < OP_HEAD_TOKENS / 256 * GROUPS; sc += 16) {
      const int chunk = sc / GROUPS, q = lane >> 4;
      if (256 * chunk >= N) break;
      float s[2] = {0.f, 0.f}, mn[2] = {INFINITY, INFINITY}, mx[2] = {-INFINITY, -INFINITY};
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int group = 64 * chunk + GROUPS * u + sc % GROUPS;
        const unsigned w = *reinterpret_cast<const unsigned*>(at(group, q) + 2 * cp);
        const float f[2] = {lo16_to_f32<DT>(w), hi16_to_f32<DT>(w)};
#pragma unroll
        for (int c = 0; c < 2; c++) {
          s[c] += f[c];
          if (4 * group + q < N) {
            mn[c] = fminf(mn[c], f[c]);
            mx[c] = fmaxf(mx[c], f[c]);
          }
        }
      }
#pragma unroll
      for (int c = 0; c < 2; c++) {
        float x, y;
        with_lane_xor16(s[c], x, y);  s[c] = x + y;
        with_lane_xor16(mn[c], x, y); mn[c] = fminf(x, y);
        with_lane_xor16(mx[c], x, y); mx[c] = fmaxf(x, y);
        with_lane_xor32(s[c], x, y);  s[c] = x + y;
        with_lane_xor32(mn[c], x, y); mn[c] = fminf(x, y);
        with_lane_xor32(mx[c], x, y); mx[c] = fmaxf(x, y);
        if (lane < 16) {
          red[sc][0][cp + c] = s[c];
          red[sc][1][cp + c] = mn[c];
          red[sc][2][cp + c] = mx[c];
        }
      }
    }
    __syncthreads();
    float mean_t = 0.f, scale_t = 0.f;   // threads below 32: their channel's
    if (wave == 0) {
      const int ch = lane & 31;          // lower half: sum and minimum, upper half: maximum
      double sum = 0.0;
      float ext = lane < 32 ? INFINITY : -INFINITY;
#pragma unroll
      for (int c = 0; c < OP_HEAD_TOKENS / 256; c++) {
        if (256 * c >= N) break;
        float x[GROUPS];
#pragma unroll
        for (int g = 0; g < GROUPS; g++) {
          x[g] = red[GROUPS * c + g][0][ch];
          const float e = red[GROUPS * c + g][lane < 32 ? 1 : 2][ch];
          ext = lane < 32 ? fminf(ext, e) : fmaxf(ext, e);
        }
#pragma unroll
        for (int n = 1; n < GROUPS; n *= 2)
#pragma unroll
          for (int g = 0; g < GROUPS; g += 2 * n) x[g] += x[g + n];
        sum += x[0];
      }
      float lo, hi;
      with_lane_xor32(ext, lo, hi);
      mean_t = p.smooth_v ? (float)(sum / (double)N) : 0.f;
      const float amax = fmaxf(hi - mean_t, mean_t - lo);
      scale_t = amax / 448.0f;
      if (lane < 32) {
        chan[0][ch] = amax > 0.f ? 448.0f / amax : 0.f;
        chan[1][ch] = mean_t;
      }
    }
    __syncthreads();
    const float recp[2] = {chan[0][cp], chan[0][cp + 1]}, mean[2] = {chan[1][cp], chan[1][cp + 1]};
    for (int pc = wave; pc < 4 * p.nbk; pc += 16) {
      const int kb = pc >> 2, mt = (pc >> 1) & 1, lh = pc & 1, g = lane >> 4;
      const int group = kb * 16 + mt * 8 + 2 * g + lh;
      float f[2][4];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const unsigned w = *reinterpret_cast<const unsigned*>(at(group, q) + 2 * cp);
        const bool in = 4 * group + q < N;
        f[0][q] = in ? (lo16_to_f32<DT>(w) - mean[0]) * recp[0] : 0.f;
        f[1][q] = in ? (hi16_to_f32<DT>(w) - mean[1]) * recp[1] : 0.f;
      }
      uint8_t* out = p.v_tiles + ((int64_t)bh * p.nbk + kb) * (64 * D) + part * 2048 + mt * 1024 + (lh * 32 + cp) * 16 + 4 * g;
#pragma unroll
      for (int c = 0; c < 2; c++) {
        int w = __builtin_amdgcn_cvt_pk_fp8_f32(f[c][0], f[c][1], 0, false);
        w = __builtin_amdgcn_cvt_pk_fp8_f32(f[c][2], f[c][3], w, true);
        *reinterpret_cast<int*>(out + 16 * c) = w;
        const float e = ((f[c][0] - __builtin_amdgcn_cvt_f32_fp8(w, 0)) + (f[c][1] - __builtin_amdgcn_cvt_f32_fp8(w, 1))) +
                        ((f[c][2] - __builtin_amdgcn_cvt_f32_fp8(w, 2)) + (f[c][3] - __builtin_amdgcn_cvt_f32_fp8(w, 3)));
        // the four words of a piece one after the other (lanes 0..15)
        float own, e1, e2, e3;
        with_lane_xor16(e, own, e1);
        with_lane_xor32(e, own, e2);
        with_lane_xor32(e1, own, e3);
        if (lane < 16) resid[2 * kb + mt][lh][cp + c] = ((e + e1) + e2) + e3;
      }
    }
    __syncthreads();
    if (t < 32) {
      float r = 0.f;
      for (int i = 0; i < 2 * p.nbk; i++) r += resid[i][0][t] + resid[i][1][t];
      const int64_t ch = (int64_t)bh * D + 32 * part + t;
      p.v_scale[ch] = scale_t;
      p.v_mean[ch] = p.smooth_v ? mean_t + scale_t * (r / (float)N) : mean_t;
    }
  }
}

// op_finalize and op_prep in one, for sequences of few statistics chunks: every workgroup adds the chunks up for itself.  256
// threads take one V tile or 256 tokens of K.  To the bit the results of the two launches (sums of short chunks are added up
// in fp64).  (Tried as well: the last V tile of a head to get there adds up the residuals, instead of a launch of its own.
// Rows that other compute units have just written have to be read past the caches: N = 4096, two heads, 31.6 us instead of 25.0.)
template <int DT, int D, bool F16V>
__global__ void __launch_bounds__(256) op_prep_short_kernel(const OpParams p) {
  constexpr int LPR = D / 8, ROWS = 256 / LPR, SL = 256 / D, PITCH = D + 8;
  const int t = threadIdx.x, wave = t >> 6;
  const int per_k = (p.nbk + 3) / 4, per = p.nbk + per_k;
  const int block = with_args(p, blockIdx.x), bh = block / per, j = block % per;
  const int b = bh / p.Hkv, h = bh % p.Hkv, N = p.Nk;
  const int ch = t % D, sl = t / D;
  __shared__ double red_s[SL][D];
  __shared__ __attribute__((aligned(16))) unsigned short tile[64 * PITCH];
  if (j >= p.nbk) {
    unsigned short* mean = tile;
    if (p.stats_k) {
      const float* x = p.k_partial + (int64_t)bh * p.chunks * D + ch;
      double s = 0.0;
      for (int c = sl; c < p.chunks; c += SL) s += x[c * D];
      red_s[sl][ch] = s;
      __syncthreads();
      if (t < D) {
        for (int i = 1; i < SL; i++) s += red_s[i][ch];
        mean[ch] = (unsigned short)(pack2_from_f32<DT>((float)(s / (double)N), 0.f) & 0xffffu);
        if (j == p.nbk) p.k_mean[(int64_t)bh * D + ch] = mean[ch];
      }
      __syncthreads();
    }
    const int g = (j - p.nbk) * 4 + wave;
    if (g >= p.nbk) return;
    const unsigned short* k = p.k + b * p.ks_b + h * p.ks_h;
    int8_t* out = p.k8 + (int64_t)bh * N * D;
    float* scale = p.k_scale + (int64_t)bh * p.nbk;
    if (p.stats_k) quant_group_body<DT, D, 64, true, false>(k, mean, out, scale, N, g, p.ks_n, D, 0.f);
    else quant_group_body<DT, D, 64, false, false>(k, nullptr, out, scale, N, g, p.ks_n, D, 0.f);
    return;
  }
  const unsigned short* v = p.v + b * p.vs_b + h * p.vs_h;
  if constexpr (F16V) {
    v_f16_load_tile<D>(v, tile, N, p.vs_n, j, t);
    __syncthreads();
    v_f16_store_tile<DT, D>(tile, (unsigned short*)p.v_tiles + ((int64_t)bh * p.nbk + j) * (64 * D), t);
  } else {
    __shared__ float red[2][SL][D];
    __shared__ float chan[2][D];        // reciprocal scale, mean
    const int col = (t % LPR) * 8, row = t / LPR;
    v4i raw[64 / ROWS];
#pragma unroll
    for (int u = 0; u < 64 / ROWS; u++) {
      const int tok = j * 64 + row + u * ROWS;
      raw[u] = tok < N ? *reinterpret_cast<const v4i*>(v + (int64_t)tok * p.vs_n + col) : v4i{0, 0, 0, 0};
    }
    const float* x = p.v_work + v_stats_offset((int64_t)p.B * p.Hkv, N, D) + (int64_t)bh * p.chunks * 3 * D + ch;
    double s = 0.0;
    float mn = INFINITY, mx = -INFINITY;
#pragma unroll 4
    for (int c = sl; c < p.chunks; c += SL) {
      s += x[(c * 3 + 0) * D];
      mn = fminf(mn, x[(c * 3 + 1) * D]);
      mx = fmaxf(mx, x[(c * 3 + 2) * D]);
    }
    red_s[sl][ch] = s;
    red[0][sl][ch] = mn;
    red[1][sl][ch] = mx;
#pragma unroll
    for (int u = 0; u < 64 / ROWS; u++) *reinterpret_cast<v4i*>(&tile[(row + u * ROWS) * PITCH + col]) = raw[u];
    __syncthreads();
    if (t < D) {
      for (int i = 1; i < SL; i++) {
        s += red_s[i][ch];
        mn = fminf(mn, red[0][i][ch]);
        mx = fmaxf(mx, red[1][i][ch]);
      }
      const float mean = p.smooth_v ? (float)(s / (double)N) : 0.f;
      const float amax = fmaxf(mx - mean, mean - mn);
      chan[0][ch] = amax > 0.f ? 448.0f / amax : 0.f;
      chan[1][ch] = mean;
      if (j == 0) {
        p.v_scale[(int64_t)bh * D + ch] = amax / 448.0f;
        p.v_mean[(int64_t)bh * D + ch] = mean;
      }
    }
    __syncthreads();
    float rs[D / 64];
    pack_v_tile<DT, D, PITCH>(tile, p.v_tiles + ((int64_t)bh * p.nbk + j) * (64 * D), chan[0], p.smooth_v ? chan[1] : nullptr,
                              j * 64, N, t, rs);
    if (!p.smooth_v) return;
    float* resid = p.v_resid + (int64_t)bh * p.nbk * 2 * D;
    if ((t & 63) < 32) {
#pragma unroll
      for (int n = 0; n < D / 64; n++)
        resid[(j * 2 + (wave & 1)) * D + 32 * ((wave >> 1) + 2 * n) + (t & 31)] = rs[n];
    }
  }
}

// What a launch less is worth, 2 to 3 us, against the chunks (768 bytes per 256 tokens, of V at D = 64) that every workgroup
// reads.  Operator, smooth_k, with op_finalize / without it, us: D = 64 N = 320 256 heads 32.9 / 29.7, N = 1024 100 heads 42.0 /
// 38.5 (D = 128 70.6 / 67.0); N = 1100 2 heads 22.2 / 20.0, 96 heads 44.2 / 41.1;
// N = 4096 2 heads 26.6 / 24.6, 24 heads 63.1 / 59.6, 96 heads 182.2 / 180.5; N = 8192 8 heads 68.9 / 67.2, 48 heads 288.8 / 289.9;
// D = 128 N = 4096 2 heads 35.0 / 33.7, 48 heads 183.6 / 183.8; N = 8192 2 heads 60.2 / 59.2, 24 heads 288.3 / 292.9.
static bool op_short(int64_t BK, int Nk, int D, bool per_thread) {
  return !per_thread && (Nk <= 4096 || (Nk <= 8192 && BK * D <= 512));
}

// Whether Q has a pass of its own, in op_prep.  The attention kernels quantise 16-bit Q at next to no cost where a compute unit
// has other waves to work on meanwhile (QRows); with few q-blocks it is 0.3 us (D = 64) to 2 us on the way of each, while op_prep
// has compute units to spare for it.  Operator, in the attention kernel / in op_prep, shares of the time, by q-blocks:
//                                             up to 64        65 to 128      129 to 256     601 to 1024    above 1536
//   float16 tiles without smooth_k  D = 64   1.01 to 1.04    1.01 to 1.04   0.99 to 0.99   0.96 to 0.99   0.94 to 0.97
//     (N = 8 .. 4000; 9.4 / 9.1 us)  D = 128  1.02 to 1.06    1.01 to 1.02   0.99 to 1.01   0.97 to 1.00   0.95 to 0.97
//   4500 and 9000 keys, FP8         D = 64   0.99 to 1.00    0.99 to 1.00   0.99 to 1.00   0.97 to 0.99   0.97
//                                    D = 128  0.99 to 1.03    1.00 to 1.02   1.00 to 1.01   0.98 to 0.99   0.98
//     with the log-sum-exp          D = 64   0.98 to 1.03    1.00 to 1.02   1.00 to 1.01   0.99 to 1.00   0.98
//                                    D = 128  1.00 to 1.03    1.00 to 1.01   1.01 to 1.02   0.98 to 1.00   0.97 to 0.99
// Calls that have no op_prep keep it in the attention kernel: the launch they lack is worth more.
static bool op_q_pass(int64_t q_blocks, int64_t BK, int Nk, int D, bool smooth_k, bool per_thread, bool f16v) {
  if (per_thread) return true;
  return q_blocks <= 2 * D && !((smooth_k || !f16v) && op_short(BK, Nk, D, false));
}

// Where the intermediate tensors lie in the workspace (256-byte aligned pieces).
struct OpLayout {
  int64_t q8, k8, v_tiles, q_scale, k_scale, v_scale, v_mean, v_work, k_partial, k_mean, resid, bytes;
  OpLayout(int B, int H, int Hkv, int Nq, int Nk, int D, bool smooth_k, bool per_thread, bool f16v) {
    bytes = 0;
    auto take = [&](int64_t n) {
      const int64_t at = bytes;
      bytes += (n + 255) & ~(int64_t)255;
      return at;
    };
    const int64_t nbq = ceil_div(Nq, 64), nbk = ceil_div(Nk, 64), BK = (int64_t)B * Hkv, BQ = (int64_t)B * H;
    const bool q_pass = op_q_pass(BQ * nbq, BK, Nk, D, smooth_k, per_thread, f16v);
    q8 = take(q_pass ? BQ * Nq * D : 0);   // (otherwise the attention kernels quantise Q themselves)
    k8 = take(BK * Nk * D);
    v_tiles = take(BK * nbk * 64 * D * (f16v ? 2 : 1));
    q_scale = take(q_pass ? BQ * nbq * (per_thread ? 16 : 2) * 4 : 0);
    k_scale = take(BK * nbk * (per_thread ? 4 : 1) * 4);
    v_scale = take(f16v ? 0 : BK * D * 4);
    v_mean = take(f16v ? 0 : BK * D * 4);
    v_work = take(f16v ? 0 : paro_v_fp8_partial_floats(B, Hkv, Nk, D) * 4);
    k_partial = take(smooth_k ? BK * ceil_div(Nk, v_chunk(Nk)) * D * 4 : 0);
    k_mean = take(smooth_k ? BK * D * 2 : 0);
    const bool s = op_short(BK, Nk, D, per_thread) && !f16v;
    resid = take(s ? BK * nbk * 2 * D * 4 : 0);   // (the chunks in v_work are read until the last tile)
  }
};

// Whether op_head does it all, and how it divides K (op_prep_short is what it stands against).  A compute unit holds one of its
// workgroups (16 waves of 92 to 101 registers), so what counts is how many rounds of 256 they come to.  K by 256 tokens is
// taken where all fit into one round.  Otherwise a workgroup takes the K of a whole head (with smooth_k all of those that share
// a head would read it all for the mean): in one round up to 768 tokens, beyond that not where such a workgroup has the
// longest time of its own (D = 128 with the mean) nor with float16 tiles; in two rounds up to 512 tokens, beyond that at D = 64
// where the second is more than half full.  Without the mean two rounds of 256 tokens are the better ones up to 768 tokens.
// Operator, us, op_prep_short / op_head:
//   smooth_k       D = 64   N = 512   60 heads 21.1 / 16.2   85 heads 23.1 / 18.5   100 heads 24.4 / 24.5   170 heads 30.9 / 29.6
//                           N = 1024  32 heads 23.5 / 22.9   85 heads 33.3 / 30.9   100 heads 38.3 / 40.0   170 heads 54.6 / 53.0
//                  D = 128  N = 320   43 heads 25.7 / 21.2   85 heads 30.3 / 29.4   100 heads 31.3 / 31.8
//                           N = 1024  16 heads 29.4 / 25.8   43 heads 37.1 / 39.2    60 heads 44.4 / 50.2   100 heads 67.1 / 72.7
//   without (and with K by 256 tokens in two or three rounds)
//                  D = 64   N = 1024  60 heads 27.6 / 26.0 (27.5)   100 heads 36.4 / 37.0 (37.7)
//                  D = 128  N = 512   70 heads 31.7 / 31.5 (30.5)   N = 1024 51 heads 37.5 / 36.8 (44.0)
//   float16 tiles  D = 64   N = 700   64 heads 26.0 / 24.6   90 heads 28.8 / 34.3
//                  D = 128  N = 384   90 heads 34.7 / 29.8   N = 1024 43 heads 39.1 / 43.3
static void op_head_plan(OpParams& p, int64_t BK, int D, bool per_thread, bool f16v) {
  const int64_t k_parts = ceil_div(p.nbk, 4), v_parts = f16v ? k_parts : D / 32, by_tokens = BK * (k_parts + v_parts),
                by_heads = BK * (1 + v_parts);
  bool fits = by_tokens <= 256 || (by_tokens <= 512 && by_heads > 256 && !p.stats_k && p.Nk <= 768);
  p.k_rounds = fits ? 1 : (int)k_parts;
  if (!fits && by_heads <= 256) fits = p.Nk <= 768 || (!f16v && (D == 64 || !p.stats_k));
  else if (!fits && by_heads <= 512) fits = p.Nk <= 512 || (!f16v && D == 64 && by_heads > 400);
  p.k_parts = ceil_div(p.nbk, 4 * p.k_rounds);
  p.one_launch = fits && !per_thread && p.Nk <= OP_HEAD_TOKENS && p.stats_k + p.stats_v > 0;
}

template <int DT, int D, bool F16V>
static int launch_op_head(const OpParams& p, hipStream_t st) {
  const int parts = p.k_parts + (F16V ? ceil_div(p.nbk, 4) : D / 32);
  hipLaunchKernelGGL((op_head_kernel<DT, D, F16V>), dim3(p.B * p.Hkv * parts), dim3(1024), 0, st, p);
  PARO_HIP(hipGetLastError());
  return PARO_OK;
}

template <int DT, int D>
static int launch_op_prep(const OpParams& p, bool per_thread, bool f16v, hipStream_t st) {
  if (p.one_launch) return f16v ? launch_op_head<DT, D, true>(p, st) : launch_op_head<DT, D, false>(p, st);
  if (p.stats_k + p.stats_v > 0) {
    hipLaunchKernelGGL((op_stats_kernel<DT, D>), dim3(p.chunks * (p.stats_k + p.stats_v), p.Hkv, p.B), dim3(256), 0, st, p);
    if (p.short_prep) {
      const dim3 all(p.kv_blocks);
      if (f16v) hipLaunchKernelGGL((op_prep_short_kernel<DT, D, true>), all, dim3(256), 0, st, p);
      else hipLaunchKernelGGL((op_prep_short_kernel<DT, D, false>), all, dim3(256), 0, st, p);
      PARO_HIP(hipGetLastError());
      return PARO_OK;
    }
    hipLaunchKernelGGL((op_finalize_kernel<DT, D>), dim3(p.B * p.Hkv * (p.stats_k + p.stats_v)), dim3(1024), 0, st, p);
  }
  const int q_blocks = p.q_pass ? p.B * p.H * ceil_div(per_thread ? p.nbq : 2 * p.nbq, 4) : 0;
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
  p.q_pass = op_q_pass((int64_t)B * H * p.nbq, (int64_t)B * Hkv, Nk, D, smooth_k != 0, per_thread, f16v);
  p.lse_add = p.q_pass && smooth_k ? lse : nullptr;   // (the attention kernel adds to what the row holds)
  p.chunks = ceil_div(Nk, v_chunk(Nk));
  p.stats_k = smooth_k != 0; p.stats_v = !f16v;
  p.kv_blocks = B * Hkv * (p.nbk + ceil_div(p.nbk, 4));
  p.sm_scale = sm_scale;
  op_head_plan(p, (int64_t)B * Hkv, D, per_thread, f16v);
  p.short_prep = op_short((int64_t)B * Hkv, Nk, D, per_thread);
  if (p.short_prep && p.v_resid) p.v_resid = (float*)(ws + at.resid);
  hipStream_t st = (hipStream_t)stream;
  int rc;
  if (dtype == PARO_DTYPE_F16)
    rc = D == 64 ? launch_op_prep<PARO_DTYPE_F16, 64>(p, per_thread, f16v, st) : launch_op_prep<PARO_DTYPE_F16, 128>(p, per_thread, f16v, st);
  else
    rc = D == 64 ? launch_op_prep<PARO_DTYPE_BF16, 64>(p, per_thread, f16v, st) : launch_op_prep<PARO_DTYPE_BF16, 128>(p, per_thread, f16v, st);
  if (rc) return rc;
  AttnExtra extra;
  // (of v_work, what lies in front of the residual sums is nobody's any more)
  if (v_resid_offset((int64_t)B * Hkv, Nk, D) >= (int64_t)B * H &&
      attn_wants_share(B, H, Nq, Nk, D, is_causal != 0, flags | (per_thread ? PARO_ATTN_QK_PER_THREAD : 0)))
    extra.share = (int*)p.v_work;
  if (p.v_resid && !p.one_launch && !per_thread && attn_takes_residual(B, H, Nq, Nk, D, is_causal != 0, lse != nullptr, flags)) {
    extra.v_resid = p.v_resid;
    extra.resid_rows = 2 * p.nbk;
  } else if (p.v_resid && !p.one_launch) {
    const ShareLook look = {sparse, sparse_batch_stride, H, sparse_batch_stride != 0 ? B * H : H, p.nbq, p.nbk, is_causal, extra.share};
    if ((rc = v_fp8_add_residual(p.v_resid, p.v_scale, p.v_mean, B, Hkv, Nk, D, st, extra.share ? &look : nullptr))) return rc;
    extra.share_ready = extra.share != nullptr;
  }
  extra.lse_scale = 0.6931471805599453f;
  extra.lse_add = p.lse_add != nullptr;
  if (!p.q_pass) {
    extra.q16 = p.q;
    extra.k_mean = p.k_mean;
    extra.lse_dot_scale = sm_scale;
  }
  const int64_t qs_b = p.q_pass ? (int64_t)H * Nq * D : q_stride_b, qs_h = p.q_pass ? (int64_t)Nq * D : q_stride_h;
  return attn_sparse_impl(p.q8, p.k8, p.v_tiles, p.q_scale, p.k_scale, p.v_scale, smooth_v ? p.v_mean : nullptr, sparse,
                          sparse_batch_stride, out, dtype, lse, extra, nullptr, B, H, Hkv, Nq, Nk, D, qs_b, qs_h,
                          p.q_pass ? D : q_stride_n, (int64_t)Hkv * Nk * D, (int64_t)Nk * D, D, o_stride_b, o_stride_h,
                          o_stride_n, sm_scale, is_causal, flags | (per_thread ? PARO_ATTN_QK_PER_THREAD : 0), nullptr, 0, 0, 0,
                          0, stream);
}
