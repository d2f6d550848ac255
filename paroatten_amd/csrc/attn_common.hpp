// Shared by the attention kernels of this library (attn_sparse.hip: two waves per 64-row q-block, any head
// size and variant; attn_sparse_w64.hip: one wave per q-block, D = 64; attn_sparse_split.hip: several kept blocks of a
// q-block at a time; attn_sparse_pv16.hip: float16 P.V product): launch parameters, the constants of the
// softmax-weight arithmetic and small device helpers.  gfx950 only.
#pragma once
#include "paro_device.hpp"
#include "share_device.hpp"
#include <type_traits>

namespace paro {

struct AttnParams {
  const int8_t* q8;
  const int8_t* k8;
  const uint8_t* v8;
  const float* q_scale;
  const float* k_scale;
  const float* v_scale;
  const float* v_mean;
  const uint8_t* sparse;
  void* out;
  float* lse;            // what is stored: base-2 log-sum-exp * lse_scale (+ what the row holds before, with lse_add)
  float lse_scale;
  int lse_add;
  int32_t* s_dump;
  int64_t sparse_bs;
  int64_t qs_b, qs_h, qs_n;
  int64_t ks_b, ks_h, ks_n;
  int64_t os_b, os_h, os_n;
  int B, H, Hkv, Nq, Nk, nbq, nbk;
  int total;  // B*H*nbq workgroups that have work
  float sm_scale_log2e;
  // optional inverse permutation on the way out: q-row r of head h is stored at token
  // n_text + unpermute(r - n_text, orders[h]) (rows below n_text stay); orders == nullptr: row r
  const int* orders;
  int n_text, F, Hh, W;
  int pacing;  // +1: paced launch asked for, -1: plain launch asked for, 0: the library chooses
  // Q as the 16-bit tensor (of the output's type; qs_* are its strides, q8 and q_scale are not read): the kernels quantise
  // the rows of their q-block themselves (QRows).  k_mean [B,Hkv,D] (may be null; with lse): the mean that has been taken
  // off K, the row's log-sum-exp gets lse_dot_scale * q . k_mean.
  // (Which of the two a kernel reads is a template parameter, Q16.  As a branch at run time it cost calls on INT8 Q 0.1 to 0.5 us
  // in front of the loop, 1 to 2 % of those below 50 us: 48 heads, N = 1024, D = 64 9.07 / 8.92 us, 40 heads, N = 2048,
  // D = 128 38.2 / 37.45, two heads, N = 4096 12.40 / 12.28 and 18.58 / 18.21; calls on 16-bit Q are the same.)
  const unsigned short* q16;
  const unsigned short* k_mean;
  float lse_dot_scale;
  // Scratch of the call (null: none given), one word per head of the mask: whether the pair kernel takes it (attn_share_kernel)
  int* share;
  int share_ready;   // it holds that already
  // The residual sums of the V tiles, [B,Hkv][resid_rows][D], that v_mean still lacks (null: it is complete).  attn_sparse_split.hip
  // alone takes them (attn_takes_residual).
  const float* v_resid;
  int resid_rows;
};

__device__ __forceinline__ bool tiles_shared(const AttnParams& p, int bh) { return p.share[p.sparse_bs != 0 ? bh : bh % p.H] != 0; }

// P~ = 2^(S*c - m + P_EXP_OFFSET).  m is the running row maximum, refreshed lazily: only when a
// weight leaves the range of e4m3 are m, O and the row sums rescaled.  Fast exponentials: a weight that would round to
// more than 448, the largest e4m3 value (a score about 3.8 octaves above m).  True exponentials: a block maximum more than
// P_HEADROOM above m.  (The weight of a fresh maximum is 2^5, which e4m3 holds exactly: letting it grow to the last code
// cost up to 0.2 % in the error against 64 bits.)
constexpr float P_EXP_OFFSET = 5.0f;
constexpr float P_HEADROOM = 3.75f;
constexpr int S_MAGIC_BITS = 0x4B400000;  // float 1.5 * 2^23
constexpr float S_MAGIC_F = 12582912.0f;
constexpr int FP8_ONES = 0x38383838;  // four e4m3 1.0
constexpr float FAST_EXP_SHIFT = -0.35f;  // centres the linear-mantissa error of the fast exponential
// fast path: the real-valued byte b becomes the 16-bit field round((b + 0.5) * 256), whose HIGH byte is
// round(b); the field is bounded by 0x7FFF, so the byte is bounded by 0x7F
constexpr float FAST_FIELD_SCALE = 256.0f / 32767.0f;

// The q-block (numbered over batch, head, q-block) that is the slot-th of XCD xcd, per = ceil(total / 8) to each;
// p.total or more: none.  Each XCD walks a contiguous range of them, so that the K8 / V8 of the head it is working on
// stay in its own L2.  Causal: a q-block's work grows with its index.  The longest of a head go first, so that short ones
// fill the card at the end, and heads that do not come out even are dealt out q-block by q-block, since the two halves of
// a head are 1 : 3 in work.  B = 2, H = 32, N = 8192, D = 128, every block below the diagonal, kernel alone: 609 -> 592 us;
// B = 1, H = 48, D = 64: 273 -> 257 us.
// PAIR: the same over pairs of neighbouring q-blocks of a head, qblock_units of them.
template <bool PAIR> __device__ __forceinline__ int qblock_units(const AttnParams& p) {
  return PAIR ? p.B * p.H * ((p.nbq + 1) >> 1) : p.total;
}
template <bool CAUSAL, bool PAIR = false>
__device__ __forceinline__ int qblock_of(const AttnParams& p, int xcd, int slot, int per) {
  if constexpr (!CAUSAL) return xcd * per + slot;
  const int n = PAIR ? (p.nbq + 1) >> 1 : p.nbq, total = qblock_units<PAIR>(p);
  const int heads = total / n, own = (heads >> 3) * n;   // q-blocks of the heads that an XCD has to itself
  const int i = slot < own ? xcd * own + slot : 8 * own + (slot - own) * 8 + xcd;
  const int head = i / n;
  return head < heads ? head * n + (n - 1 - (i - head * n)) : total;
}

__device__ __forceinline__ void store_lse(const AttnParams& p, int64_t row, float lse2) {
  p.lse[row] = p.lse_add ? fmaf(lse2, p.lse_scale, p.lse[row]) : lse2 * p.lse_scale;
}

__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

__device__ __forceinline__ float max3_abs(float a, float b, float c) {   // max(|a|, |b|, c)
  float r;
  asm("v_max3_f32 %0, |%1|, |%2|, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// The 32 q-rows of one wave (or half of one), from 16 bits: INT8 codes in the B operand's order, and their scale.  Lane: row
// lane % 32, channels 32 ks + 16 (lane / 32) .. + 15 of k-step ks.  Codes and scale are those of quant_group_body, to the
// bit (rows past the end repeat the last one, which leaves the maximum as it is; their results are never stored).
// A pass of its own for Q (3 bytes per element, and a fourth to read the codes back) is bound by HBM, the attention
// kernel is not.
template <int DT, int D>
struct QRows {
  v4i raw[D / 16];
  // p: the row's first channel, plus 16 (lane / 32).  (Ordinary loads: a line of memory is fetched in pieces by two to four
  // of them; with non-temporal ones the operator lost 1 to 2 %)
  __device__ __forceinline__ void load(const unsigned short* p) {
#pragma unroll
    for (int ks = 0; ks < D / 32; ks++)
#pragma unroll
      for (int i = 0; i < 2; i++)
        raw[2 * ks + i] = *reinterpret_cast<const v4i*>(p + 32 * ks + 8 * i);
  }
  // the codes; returns the scale (the same in every lane)
  __device__ __forceinline__ float quantise(v4i (&qf)[D / 32]) const {
    float amax = 0.0000001f;
#pragma unroll
    for (int c = 0; c < D / 16; c++)
#pragma unroll
      for (int j = 0; j < 8; j += 2) amax = max3_abs(elem16_to_f32<DT>(raw[c], j), elem16_to_f32<DT>(raw[c], j + 1), amax);
    amax = wave_max(amax);
    const float inv = 127.0f / amax;
#pragma unroll
    for (int c = 0; c < D / 16; c++) {
      float y[8];
#pragma unroll
      for (int j = 0; j < 8; j++) y[j] = elem16_to_f32<DT>(raw[c], j) * inv;
      qf[c >> 1][2 * (c & 1)] = (int)pack4_rint_i8(y[0], y[1], y[2], y[3]);
      qf[c >> 1][2 * (c & 1) + 1] = (int)pack4_rint_i8(y[4], y[5], y[6], y[7]);
    }
    return amax / 127.0f;
  }
  // the row's product with w[0..D) (w: plus 16 (lane / 32)), in the order of quant_group_body
  __device__ __forceinline__ float dot(const unsigned short* w) const {
    float t[D / 32];
#pragma unroll
    for (int ks = 0; ks < D / 32; ks++) {
      float d[2];
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const v4i wr = *reinterpret_cast<const v4i*>(w + 32 * ks + 8 * i);
        d[i] = 0.f;
#pragma unroll
        for (int j = 0; j < 8; j++) d[i] = fmaf(elem16_to_f32<DT>(raw[2 * ks + i], j), elem16_to_f32<DT>(wr, j), d[i]);
      }
      float a, b;
      with_lane_xor32(d[0] + d[1], a, b);
      t[ks] = a + b;
    }
    if constexpr (D == 64) return t[0] + t[1];
    else return (t[0] + t[1]) + (t[2] + t[3]);
  }
};

// two floats -> two e4m3 bytes in the low (HI = false) or high half of a word; the other half of the
// destination is left as it is, so a full word takes one call of each kind
template <bool HI>
__device__ __forceinline__ void cvt_pk_fp8(int& w, float a, float b) {
  if constexpr (HI) asm("v_cvt_pk_fp8_f32 %0, %1, %2 op_sel:[0,0,1]" : "+v"(w) : "v"(a), "v"(b));
  else asm("v_cvt_pk_fp8_f32 %0, %1, %2" : "=v"(w) : "v"(a), "v"(b));  // upper half: don't care, overwritten next
}

// Whether one of a block's weights (true exponentials, 64 columns of 32 q-rows as e4m3 bytes) can be above
// 2^(P_EXP_OFFSET + P_HEADROOM) = 420.4, without a search: as e5m2 the bytes from 0x7C on (384 and up, e4m3's NaN among
// them) are infinite or NaN and all others finite, so that a product against the selector operand of the row sums tells,
// on the matrix pipe, of which a kernel with true exponentials leaves most idle (it is bound by its 117 vector instructions
// a block).  B = 2, H = 48, N = 17776, D = 64, density 0.3, with the V conversion: 1.89 ms with a search of the block maximum,
// 17 v_max3, on every block, 1.82 ms this way, 1.81 ms when only a weight beyond the last code moved the maximum; with the
// log-sum-exp, two waves per q-block, 2.14, 2.12 and 2.07 ms.
__device__ __forceinline__ v4f headroom_probe(const v8i& selector, const v8i& weights) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(selector, weights, v4f{0.f, 0.f, 0.f, 0.f}, 0, 1, 0, 0, 0, 0);
}
__device__ __forceinline__ bool headroom_suspect(const v4f& probe) {   // wave-uniform
  return __ballot(!(probe[0] + probe[1] < INFINITY)) != 0ull;
}

// a*b + c clamped to [0,1] (the clamp is an output modifier: no extra instruction)
__device__ __forceinline__ float fma_clamp01(float a, float b, float c) {
  float r;
  asm("v_fma_f32 %0, %1, %2, %3 clamp" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// two floats in [0,1] -> round(x * 32767) as two 16-bit fields (never negative, at most 0x7FFF)
__device__ __forceinline__ int cvt_pknorm_i16(float a, float b) {
  // (the builtin, not inline assembly: between two assembly statements the compiler assumes the worst
  // hazard and pads with s_nop)
  return __builtin_bit_cast(int, __builtin_amdgcn_cvt_pknorm_i16(a, b));
}

__device__ __forceinline__ float partner_max(float x) {
  // max of own value and that of lane ^ 32: v_permlane32_swap exchanges the upper half of its
  // first operand with the lower half of its second
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return max3(__uint_as_float(r[0]), __uint_as_float(r[1]), __uint_as_float(r[1]));
}

__device__ __forceinline__ v4i buffer_load16(__amdgpu_buffer_rsrc_t rsrc, int voffset, int soffset) {
  // out-of-range bytes read as 0 (raw buffer, bounds-checked by the hardware)
  return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voffset, soffset, 0));
}

// LDS-DMA: 16 bytes per lane from a buffer straight into LDS at lds_base + lane*16; no registers, no
// ds_write; completion is counted by vmcnt
// IMM (a compile-time constant below 4096) is added to BOTH the memory offset and the LDS address: the
// pieces of one tile share one LDS base register (M0) and differ in IMM only
template <int IMM>
__device__ __forceinline__ void buffer_load16_lds(__amdgpu_buffer_rsrc_t rsrc, uint8_t* lds_base, int voffset,
                                                  int soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)lds_base, 16, voffset,
                                           soffset, IMM, 0);
}

// The one-wave-per-q-block kernel (D = 64, no score dump, plain launch).  out_dtype: PARO_DTYPE_*.
int launch_attn_w64(const AttnParams& p, int out_dtype, bool causal, bool exact, hipStream_t st);

// The kernel with a float16 P.V product (attn_sparse_pv16.hip): p.v8 points at paro_v_f16_pack's tiles, p.v_scale
// and p.v_mean may be null.  Either head size, with or without lse, plain launch.
int launch_attn_pv16(const AttnParams& p, int D, int out_dtype, bool causal, hipStream_t st);

// The kernel that takes several kept blocks of a q-block at a time (attn_sparse_split.hip): either head size, with or
// without lse, plain launch.  split_width: how many, or 0 where another kernel is the faster one.
int split_width(const AttnParams& p, int D);
bool split_takes_residual(int64_t q_blocks, int nbk, int D);   // AttnParams::v_resid
int launch_attn_split(const AttnParams& p, int D, int out_dtype, bool causal, bool exact, hipStream_t st);

// Q from 16 bits, and what goes into a stored log-sum-exp (AttnParams says what they are)
struct AttnExtra {
  float lse_scale = 1.0f;
  bool lse_add = false;
  const unsigned short* q16 = nullptr;
  const unsigned short* k_mean = nullptr;
  float lse_dot_scale = 0.f;
  int* share = nullptr;   // B * H words, or null
  bool share_ready = false;
  const float* v_resid = nullptr;
  int resid_rows = 0;
};

// Whether a call of these sizes and flags, on FP8 tiles, adds the residual sums up by itself
bool attn_takes_residual(int B, int H, int Nq, int Nk, int D, bool causal, bool with_lse, int flags);

// Whether a call of these sizes and flags has a use for AttnExtra::share
bool attn_wants_share(int B, int H, int Nq, int Nk, int D, bool causal, int flags);

// paro_attn_sparse_fwd / _unpermute_fwd (attn_sparse.hip).  extra.q16: q8 and q_scale are not read, the q strides are those of
// the 16-bit tensor, which is of the type out_dtype.
int attn_sparse_impl(const int8_t* q8, const int8_t* k8, const uint8_t* v8, const float* q_scale, const float* k_scale,
                     const float* v_scale, const float* v_mean, const uint8_t* sparse, int64_t sparse_batch_stride,
                     void* out, int out_dtype, float* lse, const AttnExtra& extra, int32_t* s_dump, int B,
                     int H, int Hkv, int Nq, int Nk, int D, int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_n,
                     int64_t k_stride_b, int64_t k_stride_h, int64_t k_stride_n, int64_t o_stride_b, int64_t o_stride_h,
                     int64_t o_stride_n, float sm_scale, int is_causal, int flags, const int32_t* orders, int n_text, int F,
                     int Hh, int W, void* stream);

}  // namespace paro
