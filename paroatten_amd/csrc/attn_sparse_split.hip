// Block-sparse quantised attention for gfx950 where there are too few q-blocks to fill the card: W kept blocks of a q-block
// at a time.
//
// Same arithmetic as attn_sparse.hip and the same weights, code for code: S^T = K8.Q8^T on v_mfma_i32_32x32x32_i8, base-2
// online softmax with weights rounded to e4m3, O^T += V8^T.P~^T on v_mfma_f32_32x32x64_f8f6f4, row sums of the rounded
// weights from v_mfma_f32_16x16x128_f8f6f4.  There, one or two waves walk the kept blocks of a q-block one after the other,
// and with fewer q-blocks than compute units most SIMDs have nothing to do.  Here a workgroup of W waves takes 32 q-rows
// (half a q-block) and W blocks of the list per round, one per wave, each with its own operands and accumulators; the first
// wave adds the shares up at the end.
//
// The weights of a block are rounded against the running maximum, so all waves keep the maximum that the walk in list
// order would have: it changes only when a weight leaves its range (rarely, and in the first block), each wave says so in LDS
// before the round's barrier, and the waves of such a round settle it in list order.  A wave before the block that
// moved the maximum keeps its weights and is rescaled after its product, one behind it computes its own again.
//
// What bounds it, by the clock inside the kernel at N = 4096, two heads, D = 64, W = 4, 11 us: 3.4 us until the first scores (a
// microsecond of it before the first load), 0.7 us a round, in which four waves fetch 32 KB through one compute unit's 64 bytes
// a clock, 1 us from the last round to the last store.  Each wave taking the first maximum for itself (instead of the first
// wave for all of them, 0.6 us), the next round's products in front of the look at the row sums and all waves adding up
// (instead of the first): 12.6 -> 11.8 us.  With the registers of two waves per SIMD at D = 64: 256 q-blocks 17.4 -> 14.3 us,
// 384 21.9 -> 18.4.  (Tried: eight blocks a round, no faster at 64 q-blocks; K through LDS at D = 64, 12.3; D = 128 in the
// registers of two waves per SIMD spills 70 of them, three times the time.)  The log-sum-exp at D = 64 spills two to four there, and
// is 12 to 24 % ahead of two waves per q-block all the same (split_width).
#include "attn_common.hpp"

namespace paro {

template <int D, int W> struct SplitLds {
  // D = 128: K goes through LDS, two tiles a wave.  (A row of K is a cache line there, of which one load instruction
  // of fragments takes 32 bytes: straight into registers it measured 22.8 instead of 18.0 us at N = 4096, two heads.)
  static constexpr int RING = D == 128 ? 2 * 64 * D : 0;
  static constexpr int PIECES = D / 32 * 4 + 1;                  // a wave's share of the result: O, and (d[0], d[1], d_exact, -)
  static constexpr int SHARES = W * PIECES * 1024;
  static constexpr int EPI_OFF = W * RING > SHARES ? W * RING : SHARES;   // v_scale and v_mean of the head
  static constexpr int M_OFF = EPI_OFF + 2 * D * 4;              // the settled maximum of the 32 rows
  static constexpr int FLAG_OFF = M_OFF + 32 * 4;                // [round parity][8] bytes, one per wave
  // Partial sums of the residual sums, 1024 x 16 bytes: at D = 64 where the shares come at the end.
  static constexpr bool RESID = D == 64 || W == 4;
  static constexpr int RED_OFF = D == 64 ? 0 : FLAG_OFF + 16;
  static_assert(D == 128 || SHARES >= 1024 * 16, "the partial sums fit where the shares go");
  static constexpr int LIST_OFF = FLAG_OFF + 16 + (D == 128 && RESID ? 1024 * 16 : 0);
  static constexpr int LIST_PAD = 4 * W;                         // a wave looks up to 4 rounds ahead
};

template <int D, int OUT_DT, bool LSE, bool EXACT, int W, bool Q16>
__global__ void __launch_bounds__(64 * W, D == 64 ? 2 : 1) attn_sparse_split_kernel(const AttnParams p, const int causal) {
  using Lds = SplitLds<D, W>;
  constexpr int KS = D / 32;      // k-steps of the QK product
  constexpr int DT = D / 32;      // 32-channel tiles of O^T
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  float* clist = reinterpret_cast<float*>(smem + Lds::LIST_OFF);
  unsigned short* klist = reinterpret_cast<unsigned short*>(clist + p.nbk + Lds::LIST_PAD + 1);
  float* m_sh = reinterpret_cast<float*>(smem + Lds::M_OFF);
  uint8_t* flags = smem + Lds::FLAG_OFF;

  const int per = gridDim.x >> 3;   // each XCD walks a contiguous range of (batch, head, q-block, half)
  const int block = with_args(p, blockIdx.x);
  const int vid = (block & 7) * per + (block >> 3);
  if (vid >= 2 * p.total) return;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int l32 = lane & 31, lh = lane >> 5;
  const int half = vid & 1, qb = (vid >> 1) % p.nbq, bh = (vid >> 1) / p.nbq;
  const int h = bh % p.H, b = bh / p.H;
  const int64_t bhk = (int64_t)b * p.Hkv + h / (p.H / p.Hkv);
  const int order_h = p.orders != nullptr ? p.orders[h] : 0;

  // ---- mask row, scales and Q, requested together; every wave builds the same list (attn_sparse.hip says why) ----
  const float* ksc_base = p.k_scale + bhk * p.nbk;
  const int kmax = causal ? min(p.nbk, qb + 1) : p.nbk;
  const uint8_t* mrow = p.sparse + b * p.sparse_bs + ((int64_t)h * p.nbq + qb) * p.nbk;
  constexpr int MU = 8;
  uint8_t m[MU];
  float msc[MU];
  auto list_load = [&](int base) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < MU; u++) {
      const int j = min(base + u * 64 + lane, kmax - 1);
      m[u] = mrow[j];
      msc[u] = ksc_base[j];
    }
  };
  const int trash = p.nbk + Lds::LIST_PAD;
  int cnt = 0;
  auto list_take = [&](int base) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < MU; u++) {
      const int j = base + u * 64 + lane;
      const bool keep = m[u] != 0 && j < kmax;
      const unsigned long long bal = __ballot(keep);
      const int pos = keep ? cnt + __popcll(bal & ((1ull << lane) - 1ull)) : trash;
      klist[pos] = (unsigned short)j;
      clist[pos] = msc[u];
      cnt += __popcll(bal);
    }
  };
  list_load(0);
  const int qrow = qb * 64 + half * 32 + l32;
  v4i qf[KS];
  float qsc = 0.f;
  [[maybe_unused]] QRows<OUT_DT, D> q16;
  {
    const int64_t qoff = b * p.qs_b + h * p.qs_h + (int64_t)min(qrow, p.Nq - 1) * p.qs_n + 16 * lh;
    if constexpr (Q16) {
      q16.load(p.q16 + qoff);
    } else {
#pragma unroll
      for (int ks = 0; ks < KS; ks++) qf[ks] = *reinterpret_cast<const v4i*>(p.q8 + qoff + 32 * ks);
      qsc = p.q_scale[((int64_t)b * p.H + h) * (p.nbq * 2) + qb * 2 + half];
    }
  }
  float* epi = reinterpret_cast<float*>(smem + Lds::EPI_OFF);
  float epi_sc = 0.f, epi_mn = 0.f;
  const int epi_ch = t % D;   // (W * 64 >= D; every wave writes the same values)
  epi_sc = p.v_scale[bhk * D + epi_ch];
  if (p.v_mean) epi_mn = p.v_mean[bhk * D + epi_ch];
  // What v_mean still lacks, in the order of v_residual_kernel, to the bit: SL partial sums per channel, added up below
  constexpr int C4 = D / 4, SL = 1024 / C4, SIDE = 64 * W / C4, PASSES = SL / SIDE;
  v4f* red = reinterpret_cast<v4f*>(smem + Lds::RED_OFF);
  if (Lds::RESID && p.v_resid != nullptr) {
    const v4f* src = reinterpret_cast<const v4f*>(p.v_resid + bhk * p.resid_rows * D) + t % C4;
    v4f x[PASSES];
#pragma unroll
    for (int u = 0; u < PASSES; u++) x[u] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int r = t / C4; r < p.resid_rows; r += SL)
#pragma unroll
      for (int u = 0; u < PASSES; u++) {
        const v4f y = src[(int64_t)min(r + u * SIDE, p.resid_rows - 1) * C4];
#pragma unroll
        for (int q = 0; q < 4; q++) x[u][q] += r + u * SIDE < p.resid_rows ? y[q] : 0.f;
      }
#pragma unroll
    for (int u = 0; u < PASSES; u++) red[(t / C4 + u * SIDE) * C4 + t % C4] = x[u];
  }
  list_take(0);
  for (int base = 64 * MU; base < kmax; base += 64 * MU) {
    list_load(base);
    list_take(base);
  }
  if (cnt > 0 && lane < Lds::LIST_PAD) {   // pad with the last kept block
    klist[cnt + lane] = klist[cnt - 1];
    clist[cnt + lane] = clist[cnt - 1];
  }
  epi[epi_ch] = epi_sc;
  epi[D + epi_ch] = epi_mn;
  __syncthreads();

  using OutT = F16x<OUT_DT>;
  auto out_row_ptr = [&]() __attribute__((always_inline)) {
    int drow = qrow;
    if (p.orders != nullptr && qrow >= p.n_text && qrow < p.Nq)
      drow = p.n_text + unpermute_index(qrow - p.n_text, order_h, p.F, p.Hh, p.W);
    return reinterpret_cast<unsigned short*>(p.out) + b * p.os_b + h * p.os_h + (int64_t)drow * p.os_n;
  };
  const int64_t lse_row = ((int64_t)b * p.H + h) * p.Nq + qrow;
  if (cnt == 0) {  // no kept block: the row outputs 0
    if (wave == 0 && qrow < p.Nq) {
      unsigned short* outp = out_row_ptr();
#pragma unroll
      for (int c = 0; c < D / 16; c++) *reinterpret_cast<v4i*>(outp + (lh * (D / 16) + c) * 8) = v4i{0, 0, 0, 0};
      if (LSE && lh == 0) p.lse[lse_row] = -INFINITY;
    }
    return;
  }

  // ---- operands: a wave is the only one to use its tiles, so they come straight into registers in fragment order, two
  //      sets of each; K (ks, mt): row 32*mt + l32, channels 32*ks + 16*lh; V (dt, mt): 16 bytes a lane, as packed ----
  const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      uniform_ptr(p.k8 + b * p.ks_b + (h / (p.H / p.Hkv)) * p.ks_h), 0, (int)((int64_t)(p.Nk - 1) * p.ks_n + D), 0x00020000);
  const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      uniform_ptr(p.v8 + bhk * p.nbk * (int64_t)(64 * D)), 0, p.nbk * 64 * D, 0x00020000);
  constexpr bool K_LDS = Lds::RING != 0;
  v4i kfrag[K_LDS ? 1 : 2][2 * KS], vfrag[2][DT][2];
  const int k_off = l32 * (int)p.ks_n + 16 * lh, k_off2 = k_off + 32 * (int)p.ks_n;
  auto load_k = [&](int kb, v4i (&f)[2 * KS]) __attribute__((always_inline)) {   // rows >= Nk read as 0
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      f[ks * 2] = buffer_load16(k_rsrc, k_off + 32 * ks, kb * 64 * (int)p.ks_n);
      f[ks * 2 + 1] = buffer_load16(k_rsrc, k_off2 + 32 * ks, kb * 64 * (int)p.ks_n);
    }
  };
  uint8_t* ring = smem + wave * Lds::RING;
  auto dma_k = [&](int kb, int st) __attribute__((always_inline)) {   // chunk c of a row is at chunk position c ^ (row ^ row / 8) % 8
#pragma unroll
    for (int i = 0; i < D / 16; i++) {
      const int row = i * (1024 / D) + lane / (D / 16);
      buffer_load16_lds<0>(k_rsrc, ring + st * 64 * D + i * 1024,
                           row * (int)p.ks_n + (((lane % (D / 16)) ^ ((row ^ (row >> 3)) & 7)) * 16), kb * 64 * (int)p.ks_n);
    }
  };
  auto read_k = [&](int st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2 * KS; i++) {
      const int row = 32 * (i & 1) + l32;
      kfrag[0][i] = *reinterpret_cast<const v4i*>(ring + st * 64 * D + row * D + (((i & ~1) + lh) ^ ((row ^ (row >> 3)) & 7)) * 16);
    }
  };
  auto load_v = [&](int kb, v4i (&f)[DT][2]) __attribute__((always_inline)) {
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int mt = 0; mt < 2; mt++) f[dt][mt] = buffer_load16(v_rsrc, lane * 16 + (dt * 2 + mt) * 1024, kb * 64 * D);
  };
  v16i magic;
#pragma unroll
  for (int i = 0; i < 16; i++) magic[i] = S_MAGIC_BITS;
  auto qk = [&](v16i (&acc)[2], const v4i (&f)[2 * KS]) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
#pragma unroll
      for (int mt = 0; mt < 2; mt++)
        acc[mt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f[ks * 2 + mt], qf[ks], ks == 0 ? magic : acc[mt], 0, 0, 0);
  };

  // ---- state of this wave: its share of O and of the row sums, relative to the common running maximum ----
  v16f o_acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int i = 0; i < 16; i++) o_acc[dt][i] = 0.f;
  v4f d_acc = {0.f, 0.f, 0.f, 0.f};   // lanes 0..15: rows lane and lane + 16 in [0], [1]
  v4f d_new = {0.f, 0.f, 0.f, 0.f};   // with the newest block, not yet accepted; EXACT: its headroom_probe
  const int sel_word = ((lane & 15) == ((lane >> 4) & 1)) ? FP8_ONES : 0;
  const v8i ones = {sel_word, sel_word, sel_word, sel_word, sel_word, sel_word, sel_word, sel_word};
  float m_i = -1e30f, m_off = 0.f, m_off8 = 0.f, d_exact = 0.f, rs = 0.f;
  v8i pf;
  auto set_max = [&](float m_new) __attribute__((always_inline)) {
    m_i = m_new;
    m_off = P_EXP_OFFSET - m_new;
    m_off8 = (8.0f * (P_EXP_OFFSET + 7.0f - m_new) + FAST_EXP_SHIFT + 0.5f) * FAST_FIELD_SCALE;
  };
  auto rescale = [&](float alpha) __attribute__((always_inline)) {
    d_acc[0] *= alpha;
    d_acc[1] *= __shfl(alpha, (lane & 15) + 16, 64);
    if constexpr (LSE) d_exact *= alpha;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int i = 0; i < 16; i++) o_acc[dt][i] *= alpha;
  };
  // the weights of the scores in acc against the maximum as it is, and their row sums, NaN where a weight left e4m3;
  // EXACT: the probe for a weight beyond the headroom (attn_sparse.hip describes the two forms)
  auto block_max = [&](const v16i (&acc)[2], float c) __attribute__((always_inline)) {
    float mx = max3(__int_as_float(acc[0][0]), __int_as_float(acc[0][1]), __int_as_float(acc[1][0]));
    mx = max3(mx, __int_as_float(acc[1][1]), __int_as_float(acc[1][1]));
    float my = max3(__int_as_float(acc[0][2]), __int_as_float(acc[0][3]), __int_as_float(acc[1][2]));
    my = max3(my, __int_as_float(acc[1][3]), __int_as_float(acc[1][3]));
#pragma unroll
    for (int i = 4; i < 16; i += 2) {
      mx = max3(mx, __int_as_float(acc[0][i]), __int_as_float(acc[0][i + 1]));
      my = max3(my, __int_as_float(acc[1][i]), __int_as_float(acc[1][i + 1]));
    }
    return fmaf(partner_max(max3(mx, my, my)), c, -S_MAGIC_F * c);
  };
  auto words = [&](const v16i (&acc)[2], float c) __attribute__((always_inline)) {
    if constexpr (EXACT) {
      const float bias = fmaf(-S_MAGIC_F, c, m_off);
      rs = 0.f;
#pragma unroll
      for (int r = 0; r < 8; r++) {
        float u[4];
#pragma unroll
        for (int q = 0; q < 4; q++) u[q] = __builtin_amdgcn_exp2f(fmaf(__int_as_float(acc[r >> 2][4 * (r & 3) + q]), c, bias));
        if constexpr (LSE) {
          rs += (u[0] + u[1]) + (u[2] + u[3]);
          asm volatile("" : "+v"(rs));   // (taken here: deferred, the sum would keep all the weights)
        }
        int w;
        cvt_pk_fp8<false>(w, u[0], u[1]);
        cvt_pk_fp8<true>(w, u[2], u[3]);
        pf[r] = w;
      }
    } else {
      const float c8 = (8.0f * FAST_FIELD_SCALE) * c;
      const float bias8 = fmaf(-S_MAGIC_F, c8, m_off8);
#pragma unroll
      for (int r = 0; r < 8; r++) {
        float u[4];
#pragma unroll
        for (int q = 0; q < 4; q++) u[q] = fma_clamp01(__int_as_float(acc[r >> 2][4 * (r & 3) + q]), c8, bias8);
        pf[r] = (int)__builtin_amdgcn_perm((unsigned)cvt_pknorm_i16(u[1], u[3]), (unsigned)cvt_pknorm_i16(u[0], u[2]), 0x07030501u);
      }
    }
    if constexpr (EXACT) d_new = headroom_probe(ones, pf);
    else d_new = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(ones, pf, d_acc, 0, 0, 0, 0, 0, 0);
  };
  auto left_range = [&](const v16i (&acc)[2], float c) __attribute__((always_inline)) {   // wave-uniform
    if constexpr (EXACT) return headroom_suspect(d_new) && __ballot(block_max(acc, c) > m_i + P_HEADROOM) != 0ull;
    else return __ballot(__builtin_isunordered(d_new[0], d_new[1])) != 0ull;
  };
  // A round in which a weight left its range (and the first): the waves settle the maximum in list order.  i: the first wave
  // that said so, flag: the round's flags.  Returns by what this wave's accumulators have to be multiplied after its product.
  using Flags = std::conditional_t<W == 4, unsigned, unsigned short>;   // a byte per wave
  auto settle = [&](const v16i (&acc)[2], float c, bool active, int i, uint8_t* flag) __attribute__((always_inline)) {
    float post = 1.0f;
    for (;;) {
      if (wave == i) {
        const float m_new = fmaxf(m_i, block_max(acc, c));
        const float alpha = __builtin_amdgcn_exp2f(m_i - m_new);
        set_max(m_new);
        rescale(alpha);
        words(acc, c);
        if (lh == 0) m_sh[l32] = m_new;
      }
      __syncthreads();
      bool left = false;
      if (wave != i) {
        const float m_new = m_sh[l32];
        const float alpha = __builtin_amdgcn_exp2f(m_i - m_new);
        set_max(m_new);
        if (wave < i) {
          post *= alpha;   // (this round's weights stand, against the maximum before)
        } else {
          rescale(alpha);
          if (active) {
            words(acc, c);
            left = left_range(acc, c);
          }
        }
      }
      if (lane == 0) flag[wave] = left;
      __syncthreads();
      const unsigned f = __builtin_amdgcn_readfirstlane((unsigned)*reinterpret_cast<const Flags*>(flag));
      if (f == 0) return post;
      i = __builtin_ctz(f) >> 3;
    }
  };

  // ---- prologue: round 0's scores ----
  auto quantise_q = [&]() __attribute__((always_inline)) {   // (Q from 16 bits: while the tiles are on their way)
    if constexpr (Q16) {
      qsc = q16.quantise(qf);
      if constexpr (LSE) {
        if (wave == 0 && p.k_mean != nullptr) {
          const float d = q16.dot(p.k_mean + bhk * D + 16 * lh) * p.lse_dot_scale;
          if (lh == 0 && qrow < p.Nq) p.lse[((int64_t)b * p.H + h) * p.Nq + qrow] = d;
        }
      }
    }
    qsc *= p.sm_scale_log2e;
  };
  const int rounds = (cnt + W - 1) / W;
  auto block_of = [&](int r) __attribute__((always_inline)) { return __builtin_amdgcn_readfirstlane((int)klist[r * W + wave]); };
  int kb_c = block_of(0), kb_1 = block_of(1), kb_2 = block_of(2);
  const int kb_first = __builtin_amdgcn_readfirstlane((int)klist[0]);
  v4i k_first[2 * KS];
  if constexpr (K_LDS) {
    // (issued in this order: the count below leaves in flight what comes after the first tile, and that of round 0 what comes
    // after the second: V alone.  0x78F: requests stay on their side, what computes may cross; a barrier for everything took
    // N = 12000, one head, log-sum-exp from 90.7 to 91.7 us)
    load_k(kb_first, k_first);
    dma_k(kb_c, 0);
    __builtin_amdgcn_sched_barrier(0);
    dma_k(kb_1, 1);
    __builtin_amdgcn_sched_barrier(0x78F);
    load_v(kb_c, vfrag[0]);
    __builtin_amdgcn_sched_barrier(0);
    quantise_q();
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(D / 16 + 2 * DT) : "memory");
    read_k(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  } else {
    load_k(kb_c, kfrag[0]);
    load_k(kb_first, k_first);
    load_k(kb_1, kfrag[1]);
    load_v(kb_c, vfrag[0]);
    quantise_q();
  }
  if (Lds::RESID && p.v_resid != nullptr && t < D) {   // (while the tiles are on their way; read behind the barriers of the rounds)
    float s = 0.f;
    for (int i = 0; i < SL; i++) s += red[i * C4 + (t >> 2)][t & 3];
    epi[D + t] = epi_mn + epi_sc * (s / (float)p.Nk);
  }
  v16i acc[2][2];   // [round parity][row tile of the 64 keys]: the next round's products are issued before the barrier
  qk(acc[0], kfrag[0]);
  // columns past the end of K or above the diagonal leave the softmax
  auto mask_edge = [&](v16i (&s)[2], int kb) __attribute__((always_inline)) {
    if ((kb == p.nbk - 1 && (p.Nk & 63) != 0) || (causal && kb == qb)) {
      int thr = p.Nk - kb * 64 - 4 * lh;
      if (causal) thr = min(thr, qrow + 1 - kb * 64 - 4 * lh);
#pragma unroll
      for (int mt = 0; mt < 2; mt++)
#pragma unroll
        for (int i = 0; i < 16; i++)
          if (32 * mt + 8 * (i >> 2) + (i & 3) >= thr) s[mt][i] = (int)0xFF800000u;
    }
  };
  {   // the maximum of the first block of the list: every wave takes it for itself
    v16i s0[2];
    qk(s0, k_first);
    mask_edge(s0, kb_first);
    set_max(fmaxf(m_i, block_max(s0, qsc * clist[0])));
  }

  float c_cur = qsc * clist[wave];
  // One round.  cur holds the scores of this round's block, nxt receives those of the next.
  auto round = [&](int r, auto parc) __attribute__((always_inline)) {
    constexpr int par = decltype(parc)::value;
    v16i(&cur)[2] = acc[par];
    v16i(&nxt)[2] = acc[par ^ 1];
    const int j = r * W + wave;
    const bool active = j < cnt;
    const float c = c_cur, c_next = qsc * clist[j + W];
    const int kidx = (int)klist[j + 3 * W];
    if constexpr (K_LDS) {   // K(r + 1) has landed: everything older than V(r), whose requests are the last ones
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * DT) : "memory");
      read_k(par ^ 1);
    }
    if (active) {
      mask_edge(cur, kb_c);
      words(cur, c);
    }
    // (the next round's products run on while the row sums are looked at and the waves meet)
    __builtin_amdgcn_sched_barrier(0);
    qk(nxt, kfrag[K_LDS ? 0 : par ^ 1]);
    __builtin_amdgcn_sched_barrier(0);
    uint8_t* flag = flags + par * 8;
    const bool left = active && left_range(cur, c);
    if (lane == 0) flag[wave] = left;
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (K_LDS) {
      dma_k(kb_2, par);                          // K(r + 2): K(r) has been used
      __builtin_amdgcn_sched_barrier(0x78F);     // (in front of V: the next round's count leaves in flight the last 2 * DT)
    } else {
      load_k(kb_2, kfrag[par]);
    }
    load_v(kb_1, vfrag[par ^ 1]);                // V(r + 1)
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();   // (a bare one: the loads stay in flight)
    const unsigned f = __builtin_amdgcn_readfirstlane((unsigned)*reinterpret_cast<const Flags*>(flag));
    float post = 1.0f;
    if (f != 0) post = settle(cur, c, active, __builtin_ctz(f) >> 3, flag);
    if (active) {
#pragma unroll
      for (int dt = 0; dt < DT; dt++) {
        const v8i a = {vfrag[par][dt][0][0], vfrag[par][dt][0][1], vfrag[par][dt][0][2], vfrag[par][dt][0][3],
                       vfrag[par][dt][1][0], vfrag[par][dt][1][1], vfrag[par][dt][1][2], vfrag[par][dt][1][3]};
        o_acc[dt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, pf, o_acc[dt], 0, 0, 0, 0, 0, 0);
      }
      if constexpr (EXACT) d_acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(ones, pf, d_acc, 0, 0, 0, 0, 0, 0);
      else d_acc = d_new;
      if constexpr (LSE) d_exact += rs;
    }
    if (f != 0) rescale(post);
    c_cur = c_next;
    kb_c = kb_1; kb_1 = kb_2; kb_2 = __builtin_amdgcn_readfirstlane(kidx);
  };
  for (int r = 0; r < rounds; r += 2) {
    round(r, std::integral_constant<int, 0>{});
    if (r + 1 >= rounds) break;
    round(r + 1, std::integral_constant<int, 1>{});
  }

  if constexpr (K_LDS) {   // the DMA of padded blocks: nobody reads it
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }
  // ---- every wave adds up its part of the channels, in the order of the waves, and stores it: 16-byte pieces
  //      [wave][piece][lane], piece (dt, g) channels 32 dt + 8 g + 4 lh .. + 3 of row l32 ----
  constexpr int PIECES = Lds::PIECES, OWN = DT * 4 / W;
  v4f* parts = reinterpret_cast<v4f*>(smem);
  {
    v4f* dst = parts + wave * PIECES * 64 + lane;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int g = 0; g < 4; g++)
        dst[(dt * 4 + g) * 64] = v4f{o_acc[dt][4 * g], o_acc[dt][4 * g + 1], o_acc[dt][4 * g + 2], o_acc[dt][4 * g + 3]};
    dst[DT * 4 * 64] = v4f{d_acc[0], d_acc[1], d_exact, 0.f};
  }
  __syncthreads();
  v4f o_sum[OWN], d_sum = parts[DT * 4 * 64 + lane];
  const v4f* own = parts + wave * OWN * 64 + lane;
#pragma unroll
  for (int i = 0; i < OWN; i++) o_sum[i] = own[i * 64];
#pragma unroll
  for (int o = 1; o < W; o++) {
#pragma unroll
    for (int i = 0; i < OWN; i++) {
      const v4f x = own[(o * PIECES + i) * 64];
#pragma unroll
      for (int q = 0; q < 4; q++) o_sum[i][q] += x[q];
    }
    const v4f x = parts[(o * PIECES + DT * 4) * 64 + lane];
#pragma unroll
    for (int q = 0; q < 3; q++) d_sum[q] += x[q];
  }

  // ---- epilogue: O = O~/d * v_scale + v_mean ----
  const float d_lo = __shfl(d_sum[0], l32 & 15, 64), d_hi = __shfl(d_sum[1], l32 & 15, 64);
  const float inv = 1.0f / (l32 < 16 ? d_lo : d_hi);
  if (qrow < p.Nq) {
    unsigned short* outp = out_row_ptr();
#pragma unroll
    for (int i = 0; i < OWN; i++) {
      const int ch = 8 * (wave * OWN + i) + 4 * lh;
      const v4f sc = *reinterpret_cast<const v4f*>(epi + ch), mn = *reinterpret_cast<const v4f*>(epi + D + ch);
      unsigned short r[4];
#pragma unroll
      for (int q = 0; q < 4; q++) r[q] = OutT::from_f32(fmaf(o_sum[i][q] * inv, sc[q], mn[q]));
      *reinterpret_cast<v2i*>(outp + ch) =
          v2i{(int)((unsigned)r[0] | ((unsigned)r[1] << 16)), (int)((unsigned)r[2] | ((unsigned)r[3] << 16))};
    }
  }
  if constexpr (LSE) {
    const float d_full = d_sum[2] + __shfl_xor(d_sum[2], 32, 64);
    if (wave == 0 && qrow < p.Nq && lh == 0) store_lse(p, lse_row, m_i + __builtin_amdgcn_logf(d_full) - P_EXP_OFFSET);
  }
}

template <int D>
static size_t split_lds(int nbk, int W) {
  const int list = W == 4 ? SplitLds<D, 4>::LIST_OFF : SplitLds<D, 2>::LIST_OFF;
  return list + (((size_t)(nbk + 4 * W + 1) * 6 + 15) & ~(size_t)15);
}

template <int D, int OUT_DT, int W, bool Q16>
static int launch_split(const AttnParams& p, bool causal, bool exact, hipStream_t st) {
  const size_t smem = split_lds<D>(p.nbk, W);
  auto kern = p.lse != nullptr ? attn_sparse_split_kernel<D, OUT_DT, true, true, W, Q16>
              : exact          ? attn_sparse_split_kernel<D, OUT_DT, false, true, W, Q16>
                               : attn_sparse_split_kernel<D, OUT_DT, false, false, W, Q16>;
  if (smem > 48 * 1024)
    PARO_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
  hipLaunchKernelGGL(kern, dim3(((2 * p.total + 7) / 8) * 8), dim3(64 * W), smem, st, p, causal ? 1 : 0);
  PARO_HIP(hipGetLastError());
  return PARO_OK;
}

// Measured against two waves per q-block (attn_sparse.hip), us, lists of 0.3 of the key blocks; q-blocks:
//                              64            128            192            256            384            512
//   D = 64   64 key blocks   W = 4 is 1.52, 1.49, 1.55, 1.50, 1.00 and 0.87 times as fast, W = 2 1.25, 1.22, 1.27, 1.27, 1.16, 1.15:
//            two waves     14.40          14.93          17.93          18.04          18.10          19.03
//            32 (W = 4)       1.24           1.24           1.22           1.17           0.81           0.76
//               (W = 2)       1.14           1.16           1.11           1.14           1.09           1.04
//            20 (W = 4)       1.17           1.15           0.98           0.81           0.71           0.61
//               (W = 2)       1.13           1.11           1.02           1.07           1.02           0.82 (520)
//            12 (W = 4)       1.03           1.02           0.92           0.94           0.68           0.56
//             8 (W = 2, with the operator's other launches)  1.02  1.03
//   D = 128  64 (W = 4)       1.53           1.52           1.10           0.93
//               (W = 2)       1.24           1.24           1.12           1.12
//            12 (W = 4)       1.25           0.78           0.73           0.73
//               (W = 2)       1.22           1.21           1.11           1.13
//             4 (W = 2, with the operator's other launches)  1.12  1.12  1.04  1.03
// A SIMD holds two of these waves at D = 64 and one at D = 128, so W is what fills the card with one round of workgroups.
// (Beyond: D = 64, 520 q-blocks, W = 2 0.82; D = 128, 260 q-blocks, W = 2 0.87.)  Longer lists gain more, up to 1.9 times at 77
// blocks of 128; of the lists the host knows only the bound, the number of key blocks.  With less than one block in eight
// kept (lists of one to four) the lines below lose up to 6 %, at 12 to 20 key blocks.
// (Those are of the attention alone, on operands that it has just read.  Behind the launches that write them, which is how it is
// called, each workgroup's first tiles come from further away, the waves of this kernel wait for them all together, and it gains
// less.  Replayed graphs, faster than two waves by, in per cent, runs of 0.25 / scattered blocks of 0.3 / every block:
//   D = 64   q-blocks                 110 to 120         180 to 256               320             400            500
//   operator       7 key blocks   1 / 2 / 3
//                 27              16 / 25 / 35   (W = 4) 6 / 16 / 21   (W = 2) 4 / 4 / 9      2 / 3 / 4
//                 64                             (W = 4) 16 / 29 / 34          8 / 11 / 13    8 / 15 / 10    4 / 10 / 5
//   layer          7             -0 / -1 / -3
//                 12 (W = 4)     -2 / -2 / 3
//                 27              -2 / 2 / 8     (W = 2) -5 / -5 / -4  (W = 2) -2 / -3 / -0   -5 / -4 / -2
//                 36               1 / 11 / 19   (W = 4) -3 / 3 / 6            -1 / -3 / 2    -4 / -2 / -0   -5 / -3 / -1
//                 64                             (W = 4) 2 / 8 / 21            -1 / 0 / 4     0 / 2 / 5      -3 / 0 / 1
//                100                             (W = 4) 4 / 19 / 34           1 / 5 / 8      0 / 1 / 7      -2 / 1 / 4
//   D = 128: 3 to 25 ahead in both.
// An operator call saves the launch of the residual sums besides, a layer, which stores through the inverse permutation, does
// not: there two waves keep the calls of more than 256 q-blocks below 76 key blocks and those of fewer than 12.  Around that line,
// on the mean of runs of 0.15 and 0.3, scattered blocks of 0.2 and 0.4 and every block: 48 key blocks -2.6 to 0.1, 56 -2.3 to 0.2, 64
// -0.9 to 0.4, 72 (288, 360, 432 and 504 q-blocks) 0.4, 1.0, 0.0 and -1.4, 80 (320, 400, 480) 2.0, 0.5 and 0.4, 91 0.6 to 3.4.)
// The lines of the log-sum-exp, 20 key blocks and 448 q-blocks, are not where this kernel stops paying (operator, D = 64, 400
// q-blocks, W = 2: 12 to 20 % ahead): the answers of paro_attn_kernel_form for calls of 512 q-blocks, and the bits of short calls,
// which are the per-thread kernel's, are older than it and kept.
int split_width(const AttnParams& p, int D) {
  int W = 0;
  if (p.lse != nullptr && (p.nbk < 20 || p.total > 448)) return 0;
  if (p.orders != nullptr && D == 64 && (p.nbk < 12 || (p.total > 256 && p.nbk < 76))) return 0;
  if (D == 64) {
    if (p.total <= 128) W = p.nbk >= 12 ? 4 : p.nbk >= 7 ? 2 : 0;
    else if (p.total <= 512 && p.nbk >= 20) W = p.total <= 256 && p.nbk >= 32 ? 4 : 2;
  } else if (p.total <= 256) {
    W = p.total <= 128 && p.nbk >= 16 ? 4 : 2;
  }
  const size_t smem = D == 64 ? split_lds<64>(p.nbk, W) : split_lds<128>(p.nbk, W);
  return smem <= 160 * 1024 ? W : 0;
}

// A launch of their own for the residual sums of V is worth 1 to 1.4 us; here every workgroup reads all of its head's, beside its
// mask row.  Operator, device time, us, a launch of their own / here: D = 64, two heads N = 1200 16.9 / 15.8, N = 2048 17.6 / 16.5,
// N = 4096 20.9 / 19.7 (four heads 23.6 / 22.2, eight 29.5 / 28.4), N = 8192 one head 25.3 / 25.4, two 29.1 / 28.7; one head, N = 30000
// 81.8 / 85.9.  D = 128, W = 4, N = 1200 23.4 / 22.3, N = 2048 25.2 / 23.8, N = 4096 30.7 / 30.0, N = 8192 38.9 / 38.9; W = 2, where
// the partial sums take the LDS of another workgroup, N = 2048, eight heads 30.9 / 32.8, N = 4096, four heads 37.5 / 43.0.
bool split_takes_residual(int64_t q_blocks, int nbk, int D) {
  return nbk <= 64 && (D == 64 || (q_blocks <= 128 && nbk >= 16));   // (D = 128: W = 4)
}

int launch_attn_split(const AttnParams& p, int D, int out_dtype, bool causal, bool exact, hipStream_t st) {
  const int W = split_width(p, D);
#define PARO_SPLIT_Q(DV, OV, QV) \
  (W == 4 ? launch_split<DV, OV, 4, QV>(p, causal, exact, st) : launch_split<DV, OV, 2, QV>(p, causal, exact, st))
#define PARO_SPLIT(DV, OV) (p.q16 != nullptr ? PARO_SPLIT_Q(DV, OV, true) : PARO_SPLIT_Q(DV, OV, false))
  if (D == 64) return out_dtype == PARO_DTYPE_F16 ? PARO_SPLIT(64, PARO_DTYPE_F16) : PARO_SPLIT(64, PARO_DTYPE_BF16);
  return out_dtype == PARO_DTYPE_F16 ? PARO_SPLIT(128, PARO_DTYPE_F16) : PARO_SPLIT(128, PARO_DTYPE_BF16);
#undef PARO_SPLIT
#undef PARO_SPLIT_Q
}

}  // namespace paro
