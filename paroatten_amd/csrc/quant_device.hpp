// Bodies of the INT8 quantisation of Q and K as device functions, so that one launch can run several of them side by
// side.  The launches that use them: quant_int8.hip (one tensor), attn_operator.hip (K and the V conversion; with few
// q-blocks or per-thread scales Q too, which otherwise the attention kernels quantise).
//
// One 64-lane wave owns one group of G tokens x D channels: every lane holds G*D/64 values in
// registers (16-byte loads, consecutive lanes on consecutive addresses), the group maximum is a
// wave reduction, and the int8 result leaves as 8-byte stores.  Nothing goes through LDS.
// Arithmetic follows QuantInt8Kernel of the reference (csrc/fused/fused.cu:64-198) in IEEE fp32:
// compiled without fast-math and with fp contraction off.
#pragma once
#include "paro_device.hpp"

namespace paro {

// eight consecutive 16-bit values as fp32
template <int DT>
__device__ __forceinline__ void load8_f32(const unsigned short* p, float (&f)[8]) {
  const v4i m = *reinterpret_cast<const v4i*>(p);
#pragma unroll
  for (int j = 0; j < 8; j++) f[j] = elem16_to_f32<DT>(m, j);
}

// Group g of one (batch, head): x, out and scale point at its first token, mean (MEAN) at its D channel means.
// SMS: the values are multiplied by sm_scale first.  dot (may be null): dot[token] = sm_scale * x[token] . dot_with, in
// fp32, for tokens below N (SMS and dot do not go together).
template <int DT, int D, int G, bool MEAN, bool SMS>
__device__ __forceinline__ void quant_group_body(const unsigned short* __restrict__ x,
                                                 const unsigned short* __restrict__ mean, int8_t* __restrict__ out,
                                                 float* __restrict__ scale, int N, int g, int64_t xs_n, int64_t os_n,
                                                 float sm_scale, float* __restrict__ dot = nullptr,
                                                 const unsigned short* __restrict__ dot_with = nullptr) {
  constexpr int LPR = D / 8;          // lanes per token row (16-byte chunks)
  constexpr int CH = G * D / 512;     // 16-byte chunks per lane
  constexpr int ROWS_PER_IT = 64 / LPR;
  const int lane = threadIdx.x & 63;
  const int col = (lane % LPR) * 8;
  const int row0 = lane / LPR;

  float mv[8];
  if constexpr (MEAN) load8_f32<DT>(mean + col, mv);

  const unsigned short* xb = x + col;
  v4i raw[CH];
#pragma unroll
  for (int i = 0; i < CH; i++) {
    const int tok = g * G + i * ROWS_PER_IT + row0;
    raw[i] = (tok < N) ? __builtin_nontemporal_load(reinterpret_cast<const v4i*>(xb + (int64_t)tok * xs_n))
                       : v4i{0, 0, 0, 0};
  }

  // value of element (chunk i, slot j) after mean subtraction / scaling; recomputed in the
  // second pass instead of being kept, so that only the packed input stays in registers
  auto value = [&](int i, int j) -> float {
    float f = elem16_to_f32<DT>(raw[i], j);
    if constexpr (MEAN) f -= mv[j];
    if constexpr (SMS) f *= sm_scale;
    return f;
  };

  float amax = 0.0000001f;
#pragma unroll
  for (int i = 0; i < CH; i++) {
    const int tok = g * G + i * ROWS_PER_IT + row0;
    if (tok < N) {  // rows past the end read as zero, whatever the mean
#pragma unroll
      for (int j = 0; j < 8; j++) amax = fmaxf(amax, fabsf(value(i, j)));
    }
  }
  amax = wave_max(amax);
  // (opaque: the converted values of the first pass would otherwise be kept, four registers a word instead of one, which
  // at D = 128 leaves two waves per SIMD)
#pragma unroll
  for (int i = 0; i < CH; i++) asm volatile("" : "+v"(raw[i]));
  if (lane == 0) scale[g] = amax / 127.0f;
  const float inv = 127.0f / amax;

  if (dot != nullptr) {   // (uniform)
    float w[8];
    load8_f32<DT>(dot_with + col, w);
#pragma unroll
    for (int i = 0; i < CH; i++) {
      float d = 0.f;
#pragma unroll
      for (int j = 0; j < 8; j++) d = fmaf(elem16_to_f32<DT>(raw[i], j), w[j], d);
      // the LPR lanes of a row: lane ^ 1, ^ 2, then the other quad of eight, then the other eight of sixteen (mirrors)
      d += row_dpp<0xB1>(d);
      d += row_dpp<0x4E>(d);
      d += row_dpp<0x141>(d);
      if constexpr (LPR == 16) d += row_dpp<0x140>(d);
      const int tok = g * G + i * ROWS_PER_IT + row0;
      if (lane % LPR == 0 && tok < N) dot[tok] = d * sm_scale;
    }
  }

  int8_t* ob = out + col;
#pragma unroll
  for (int i = 0; i < CH; i++) {
    const int tok = g * G + i * ROWS_PER_IT + row0;
    // |value * (127/amax)| <= 127 up to rounding: the reference's clamp to [-128,127] never acts
    float y[8];
#pragma unroll
    for (int j = 0; j < 8; j++) y[j] = value(i, j) * inv;
    if (tok < N)
      __builtin_nontemporal_store(
          v2i{(int)pack4_rint_i8(y[0], y[1], y[2], y[3]), (int)pack4_rint_i8(y[4], y[5], y[6], y[7])},
          reinterpret_cast<v2i*>(ob + (int64_t)tok * os_n));
  }
}

// The same arithmetic on the per-thread groups of qk_quant_gran 3: a wave owns 64 tokens (number w) and their 16 (Q: two
// 32-token groups of 8) or 4 (K) scales.  Token row r of the 64 belongs to group
//   Q: (r / 32) * 8 + r % 8        K: (r % 8) / 2
// A lane's chunks sit in rows row0 + i * ROWS_PER_IT; every group maximum is a full wave reduction of the
// lanes' contributions to that group (the kernel is bound by HBM, not by these).
template <int DT, int D, bool KEY, bool MEAN>
__device__ __forceinline__ void quant_per_thread_body(const unsigned short* __restrict__ x,
                                                      const unsigned short* __restrict__ mean,
                                                      int8_t* __restrict__ out, float* __restrict__ scale, int N, int w,
                                                      int64_t xs_n, int64_t os_n, float sm_scale = 0.f,
                                                      float* __restrict__ dot = nullptr,
                                                      const unsigned short* __restrict__ dot_with = nullptr) {
  constexpr int LPR = D / 8;
  constexpr int CH = 64 * D / 512;
  constexpr int ROWS_PER_IT = 64 / LPR;
  constexpr int NG = KEY ? 4 : 16;
  const int lane = threadIdx.x & 63;
  const int col = (lane % LPR) * 8;
  const int row0 = lane / LPR;
  auto group_of = [](int r) { return KEY ? (r % 8) / 2 : (r / 32) * 8 + r % 8; };

  float mv[8];
  if constexpr (MEAN) load8_f32<DT>(mean + col, mv);
  const unsigned short* xb = x + col;
  v4i raw[CH];
#pragma unroll
  for (int i = 0; i < CH; i++) {
    const int tok = w * 64 + i * ROWS_PER_IT + row0;
    raw[i] = (tok < N) ? __builtin_nontemporal_load(reinterpret_cast<const v4i*>(xb + (int64_t)tok * xs_n))
                       : v4i{0, 0, 0, 0};
  }
  auto value = [&](int i, int j) -> float {
    float f = elem16_to_f32<DT>(raw[i], j);
    if constexpr (MEAN) f -= mv[j];
    return f;
  };
  // this lane's maximum per chunk, then per group over the wave
  float cmax[CH];
#pragma unroll
  for (int i = 0; i < CH; i++) {
    const int tok = w * 64 + i * ROWS_PER_IT + row0;
    cmax[i] = 0.f;
    if (tok < N) {
#pragma unroll
      for (int j = 0; j < 8; j++) cmax[i] = fmaxf(cmax[i], fabsf(value(i, j)));
    }
  }
#pragma unroll
  for (int i = 0; i < CH; i++) asm volatile("" : "+v"(raw[i]));   // (as in quant_group_body)
  float inv[CH];
#pragma unroll
  for (int g = 0; g < NG; g++) {
    float a = 0.0000001f;
#pragma unroll
    for (int i = 0; i < CH; i++)
      if (group_of(i * ROWS_PER_IT + row0) == g) a = fmaxf(a, cmax[i]);
    a = wave_max(a);
    if (lane == 0) scale[(int64_t)w * NG + g] = a / 127.0f;
#pragma unroll
    for (int i = 0; i < CH; i++)
      if (group_of(i * ROWS_PER_IT + row0) == g) inv[i] = 127.0f / a;
  }
  if (dot != nullptr) {   // (uniform; as in quant_group_body)
    float wv[8];
    load8_f32<DT>(dot_with + col, wv);
#pragma unroll
    for (int i = 0; i < CH; i++) {
      float d = 0.f;
#pragma unroll
      for (int j = 0; j < 8; j++) d = fmaf(elem16_to_f32<DT>(raw[i], j), wv[j], d);
      d += row_dpp<0xB1>(d);
      d += row_dpp<0x4E>(d);
      d += row_dpp<0x141>(d);
      if constexpr (LPR == 16) d += row_dpp<0x140>(d);
      const int tok = w * 64 + i * ROWS_PER_IT + row0;
      if (lane % LPR == 0 && tok < N) dot[tok] = d * sm_scale;
    }
  }
  int8_t* ob = out + col;
#pragma unroll
  for (int i = 0; i < CH; i++) {
    const int tok = w * 64 + i * ROWS_PER_IT + row0;
    float y[8];
#pragma unroll
    for (int j = 0; j < 8; j++) y[j] = value(i, j) * inv[i];
    if (tok < N)
      __builtin_nontemporal_store(
          v2i{(int)pack4_rint_i8(y[0], y[1], y[2], y[3]), (int)pack4_rint_i8(y[4], y[5], y[6], y[7])},
          reinterpret_cast<v2i*>(ob + (int64_t)tok * os_n));
  }
}

}  // namespace paro
