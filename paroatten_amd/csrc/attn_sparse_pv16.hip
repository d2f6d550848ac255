// Block-sparse quantised attention with a 16-bit P.V product (PARO_ATTN_PV_F16), gfx950.
//
//   S^T = K8 . Q8^T      v_mfma_i32_32x32x32_i8      exact int32 (as in attn_sparse.hip)
//   P~  = 2^(S*c - m + 5) true exponentials, rounded to float16 (round to nearest even)
//   O^T += V16^T . P~^T  v_mfma_f32_32x32x16_f16     fp32 accumulation, V in float16 as given (no scale, no mean)
//   d   = sum_j P~       v_mfma_f32_16x16x32_f16 against a selector operand; with lse also in fp32 on the vector pipe
//
// This is the accuracy mode: what the reference's kernel of the same name computes, a float16 P.V product
// (csrc/qattn/qk_int_sv_f16_cuda_sm80.cu:263-391, attn_utils.cuh:383-488), where the default kernels of this
// library round P and V to FP8 e4m3.  An e4m3 code is up to 2^-4 off its value, and a q-row that one to three
// keys dominate carries that error undiluted; float16 is 2^-11.  Mask semantics, scale indexing, edge columns,
// causal masking, the unpermuting store and the log-sum-exp are those of attn_sparse.hip.
//
// Two waves per 64-row q-block (32 q-rows each).  One iteration per kept block in two phases: the weights of
// S(i) on the vector pipe, then the products S(i+1) = K(i+1).Q and O += V(i).P(i) back to back, which run on
// under the weights of block i+1; K8 and V16 tiles come in by LDS-DMA through two stages each, one barrier per
// block.  There is no row maximum per block and no sum on the vector pipe: the weights are computed with the
// running maximum as it is, and the row sums, from the matrix pipe, tell when one left float16.
//
// The row sums are fp32 sums of the weights as rounded to float16, those of the product, where they used to be of the
// weights before rounding.  That is the nearer normaliser: what the rounding adds to a row's weights on average leaves numerator
// and denominator alike.  Error against 64 bits of the two, relative, on the same scores, without the output's rounding:
// scores N(0, s), V ~ N(mean, 1), s = 1 and 512 keys 1.90e-4 before and 1.89e-4 now (mean 0), 1.92e-5 and 1.35e-5 (mean 1);
// s = 3 and 4096 keys 9.7e-5 and 9.4e-5, 3.7e-5 and 2.5e-5; never more than before for s = 0.3 to 6 and 64 to 4096 keys.
// The kernel's own outputs (float16, whose rounding alone is 2.07e-4): N = 2048, D = 64, 2.91e-4 and 2.92e-4; scores three
// times as wide 2.53e-4 and 2.67e-4.
//
// B = 2, H = 48, N = 17776, D = 64, density 0.3: 2.43-2.58 -> 2.13-2.23 ms on the same card; B = 1, H = 40, N = 16384,
// D = 128: 1.71 -> 1.56 ms (before: products and weights of a block in sequence, maximum and sums on the vector pipe).
// The cycles fell by 21 % and the shader clock from 1.67 to 1.49 GHz: it is bound by what the card lets it draw.
// Left out (results invalid), these save: half the P.V products 16 %, the tile DMA 14 %, the exponentials 12 %, half
// the Q.K products 7 %, the V fragment reads 4 %, the K fragment reads 3 %, three of four row-sum products 3 %.
//
// V16 tiles (paro_v_f16_pack): per (batch, kv-head, 64-token block) D/32 x 4 pieces of 1 KB; halfword e (0..7)
// of lane l of piece (dt, s) is token 64*kb + 32*(s/2) + 16*(s%2) + 8*(e/4) + 4*(l/32) + e%4, channel
// 32*dt + l%32: the A-operand fragment of v_mfma_f32_32x32x16_f16 under the kv-order that the S^T accumulator
// fragment imposes on the B operand (a lane's weights 8*(s%2) .. 8*(s%2)+7 of row tile s/2 are its B fragment of
// step s), so that no data moves between lanes from one product to the next.  Tokens past the end are 0.
#include "attn_common.hpp"
#include "v_pack_device.hpp"

namespace paro {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));

template <int D> struct Pv16Lds {
  static constexpr int NST = 2;
  static constexpr int KTILE = 64 * D;        // int8, 16-byte chunks XOR-swizzled as in attn_sparse.hip
  static constexpr int VTILE = 64 * D * 2;    // float16, fragment order as in memory
  static constexpr int V_OFF = NST * KTILE;
  static constexpr int LIST_OFF = NST * (KTILE + VTILE);
  static constexpr int LIST_PAD = 8;
  static __device__ __forceinline__ int swz(int row) {
    if constexpr (D == 64) return (row >> 2) & 3;
    else return (row ^ (row >> 3)) & 7;
  }
};

// The S^T accumulators start at the bit pattern of the float 1/(2 pi), which is an inline constant of the matrix
// instruction (no registers): 0x3E22F983 = 10680707 * 2^-26.  The int32 result then reads as the float
// (10680707 + S) * 2^-26 exactly, as long as it stays in that binade: |S| < 2292099, and 128*128*128 is less.
constexpr float S_INV2PI_F = 10680707.0f / 67108864.0f;
constexpr float S_INV2PI_SCALE = 67108864.0f;

// The first product of both score tiles of a block, with that constant as its accumulator operand.  (Inline assembly: the
// compiler puts a constant that two products use into a block of 16 registers, and the matrix unit then reads them in one
// product of every two (D = 64) or four.  The kernel runs at the clock that the power limit leaves: B = 2, H = 48, N = 17776,
// D = 64, density 0.3, the whole operator 2327 us with the block, 2263 us this way.)
// The compiler does not know these for matrix instructions and keeps no distance to them by itself.  Behind: the result goes
// to another product as its accumulator and nowhere else, one on the same registers from first to last, which needs no
// distance.  In front: should an operand come from a vector instruction it needs two wait states, the s_nop.
__device__ __forceinline__ void qk_first(v16i (&acc)[2], const v4i& k0, const v4i& k1, const v4i& q) {
  asm("s_nop 1\n\tv_mfma_i32_32x32x32_i8 %0, %2, %4, 0.15915494\n\tv_mfma_i32_32x32x32_i8 %1, %3, %4, 0.15915494"
      : "=&v"(acc[0]), "=&v"(acc[1]) : "v"(k0), "v"(k1), "v"(q));
}

template <int D, int OUT_DT, bool LSE, bool Q16>
__global__ void __launch_bounds__(128, (D == 64 ? 3 : 2)) attn_sparse_pv16_kernel(const AttnParams p, const int causal) {
  using Lds = Pv16Lds<D>;
  constexpr int KS = D / 32;         // k-steps of the QK MFMA
  constexpr int DT_TILES = D / 32;   // 32-channel tiles of O^T
  constexpr int KPW = D / 32;        // 1 KB pieces of a K tile per wave (half a tile)
  constexpr int VPW = D / 16;        // 1 KB pieces of a V tile per wave

  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  float* clist = reinterpret_cast<float*>(smem + Lds::LIST_OFF);
  unsigned short* klist = reinterpret_cast<unsigned short*>(clist + p.nbk + Lds::LIST_PAD + 1);

  // (arguments as they come to be needed: all of them asked for at once, 8 heads of 4000 tokens, D = 64 took 40.1 us instead of 38.2)
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, per = gridDim.x >> 3;
  const int vid = causal ? qblock_of<true>(p, xcd, slot, per) : qblock_of<false>(p, xcd, slot, per);
  if (vid >= p.total) return;

  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int l32 = lane & 31, lh = lane >> 5;
  const int qb = vid % p.nbq, bh = vid / p.nbq;
  const int h = bh % p.H, b = bh / p.H;
  const int hk = h / (p.H / p.Hkv);
  const int64_t bhk = (int64_t)b * p.Hkv + hk;
  const int order_h = p.orders != nullptr ? p.orders[h] : 0;

  // ---- compact list of the kept key blocks and their scales, requested together with Q and without a branch
  //      (attn_sparse.hip says why); both waves build the same lists ----
  const float* ksc_base = p.k_scale + bhk * p.nbk;
  const int kmax = causal ? min(p.nbk, qb + 1) : p.nbk;
  const uint8_t* mrow = p.sparse + b * p.sparse_bs + ((int64_t)h * p.nbq + qb) * p.nbk;
  constexpr int MU = 8;
  uint8_t m[MU];
  float msc[MU];
  auto list_load = [&](int base) {
#pragma unroll
    for (int u = 0; u < MU; u++) {
      const int j = min(base + u * 64 + lane, kmax - 1);
      m[u] = mrow[j];
      msc[u] = ksc_base[j];
    }
  };
  const int trash = p.nbk + Lds::LIST_PAD;   // entries that are not kept go to this spare slot
  int cnt = 0;
  auto list_take = [&](int base) {
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

  // ---- Q fragments and scale of this wave's 32 rows ----
  const int qrow = qb * 64 + wave * 32 + l32;
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
      qsc = p.q_scale[((int64_t)b * p.H + h) * (p.nbq * 2) + qb * 2 + wave];
    }
  }

  list_take(0);
  for (int base = 64 * MU; base < kmax; base += 64 * MU) {
    list_load(base);
    list_take(base);
  }
  if (cnt > 0 && lane < Lds::LIST_PAD) {   // the loop looks three blocks ahead without a branch
    klist[cnt + lane] = klist[cnt - 1];
    clist[cnt + lane] = clist[cnt - 1];
  }
  __syncthreads();

  using OutT = F16x<OUT_DT>;
  auto out_row_ptr = [&]() {
    int drow = qrow;
    if (p.orders != nullptr && qrow >= p.n_text && qrow < p.Nq)
      drow = p.n_text + unpermute_index(qrow - p.n_text, order_h, p.F, p.Hh, p.W);
    return reinterpret_cast<unsigned short*>(p.out) + b * p.os_b + h * p.os_h + (int64_t)drow * p.os_n;
  };
  if (cnt == 0) {  // no kept block: the row outputs 0 (reference: m = -5e6, d = 1, O = 0)
    if (qrow < p.Nq) {
      unsigned short* outp = out_row_ptr();
#pragma unroll
      for (int c = 0; c < D / 16; c++) *reinterpret_cast<v4i*>(outp + (lh * (D / 16) + c) * 8) = v4i{0, 0, 0, 0};
      if (LSE && lh == 0) p.lse[((int64_t)b * p.H + h) * p.Nq + qrow] = -INFINITY;
    }
    return;
  }

  // ---- tile movers: each wave moves half of every tile, 1 KB per instruction ----
  const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      uniform_ptr(p.k8 + b * p.ks_b + hk * p.ks_h), 0, (int)((int64_t)(p.Nk - 1) * p.ks_n + D), 0x00020000);
  const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      uniform_ptr(p.v8 + bhk * p.nbk * (int64_t)Lds::VTILE), 0, p.nbk * Lds::VTILE, 0x00020000);
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  int k_goff[KPW];
#pragma unroll
  for (int i = 0; i < KPW; i++) {
    const int pos = (wave_u * KPW + i) * 1024 + lane * 16;   // byte position inside the LDS tile
    const int row = pos / D, cpos = (pos % D) / 16;
    // (less the immediate offset that the instruction adds on both sides; row * ks_n >= i * 1024)
    k_goff[i] = row * (int)p.ks_n + ((cpos ^ Lds::swz(row)) * 16) - i * 1024;
  }
  const int k_blk_stride = 64 * (int)p.ks_n;
  auto load_k = [&](int kb, int st) {   // rows >= Nk read as 0
    uint8_t* base = smem + st * Lds::KTILE + wave_u * KPW * 1024;
    buffer_load16_lds<0>(k_rsrc, base, k_goff[0], kb * k_blk_stride);
    buffer_load16_lds<1024>(k_rsrc, base, k_goff[1], kb * k_blk_stride);
    if constexpr (KPW == 4) {
      buffer_load16_lds<2048>(k_rsrc, base, k_goff[2], kb * k_blk_stride);
      buffer_load16_lds<3072>(k_rsrc, base, k_goff[3], kb * k_blk_stride);
    }
  };
  const int v_goff = lane * 16;
  auto load_v = [&](int kb, int st) {
#pragma unroll
    for (int q = 0; q < VPW / 4; q++) {
      uint8_t* base = smem + Lds::V_OFF + st * Lds::VTILE + (wave_u * VPW + 4 * q) * 1024;
      const int off = kb * Lds::VTILE + (wave_u * VPW + 4 * q) * 1024;
      buffer_load16_lds<0>(v_rsrc, base, v_goff, off);
      buffer_load16_lds<1024>(v_rsrc, base, v_goff, off);
      buffer_load16_lds<2048>(v_rsrc, base, v_goff, off);
      buffer_load16_lds<3072>(v_rsrc, base, v_goff, off);
    }
  };

  // ---- fragments and products ----
  v4i kfrag[2 * KS];   // (ks, mt): row 32*mt + l32, chunk 2*ks + lh at its swizzled position
  int kr_off[2 * KS];
#pragma unroll
  for (int ks = 0; ks < KS; ks++)
#pragma unroll
    for (int mt = 0; mt < 2; mt++) {
      const int row = 32 * mt + l32;
      kr_off[ks * 2 + mt] = row * D + (((2 * ks + lh) ^ Lds::swz(row)) * 16);
    }
  auto read_k_frags = [&](int st) {
#pragma unroll
    for (int i = 0; i < 2 * KS; i++) kfrag[i] = *reinterpret_cast<const v4i*>(smem + st * Lds::KTILE + kr_off[i]);
  };
  v16i acc[2];
  auto qk_step = [&](int ks) {
    if (ks == 0) {
      qk_first(acc, kfrag[0], kfrag[1], qf[0]);
    } else {
#pragma unroll
      for (int mt = 0; mt < 2; mt++)
        acc[mt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kfrag[ks * 2 + mt], qf[ks], acc[mt], 0, 0, 0);
    }
  };
  v8h vfrag[DT_TILES];
  const int vr_base = Lds::V_OFF + lane * 16;
  auto read_v_frags = [&](int st, int s) {   // the pieces of k-step s
#pragma unroll
    for (int dt = 0; dt < DT_TILES; dt++)
      vfrag[dt] = *reinterpret_cast<const v8h*>(smem + vr_base + st * Lds::VTILE + (dt * 4 + s) * 1024);
  };

  // ---- state ----
  v16f o_acc[DT_TILES];
#pragma unroll
  for (int dt = 0; dt < DT_TILES; dt++)
#pragma unroll
    for (int i = 0; i < 16; i++) o_acc[dt][i] = 0.f;
  // Row sums of the rounded weights: in a 16x16x32 product B lane l supplies k-range 8*(l/16) .. +7 of column l%16;
  // the weights' fragment has q-row l%32 there, so k-ranges 0 and 2 belong to q-rows 0..15, 1 and 3 to q-rows 16..31.
  // With A row 0 = ones on {0, 2} and A row 1 = ones on {1, 3}, lanes 0..15 get the sums of q-rows lane and lane + 16.
  v4f d_acc = {0.f, 0.f, 0.f, 0.f};
  v8h ones;
#pragma unroll
  for (int i = 0; i < 8; i++) ones[i] = ((lane & 15) == ((lane >> 4) & 1)) ? (_Float16)1.0f : (_Float16)0.0f;
  float m_i = -1e30f, m_off = 0.f;
  float d_exact = 0.f;   // LSE: sum of the unrounded weights of this lane's 32 columns per block
  v8h pf[4];

  int kb_c = __builtin_amdgcn_readfirstlane((int)klist[0]);
  int kb_1 = __builtin_amdgcn_readfirstlane((int)klist[1]);
  int kb_2 = __builtin_amdgcn_readfirstlane((int)klist[2]);
  load_k(kb_c, 0);
  load_k(kb_1, 1);
  load_v(kb_c, 0);
  // (Q from 16 bits: quantised while the tiles are on their way)
  if constexpr (Q16) {
    qsc = q16.quantise(qf);
    if constexpr (LSE) {
      if (p.k_mean != nullptr) {
        const float d = q16.dot(p.k_mean + bhk * D + 16 * lh) * p.lse_dot_scale;
        if (lh == 0 && qrow < p.Nq) p.lse[((int64_t)b * p.H + h) * p.Nq + qrow] = d;
      }
    }
  }
  qsc *= p.sm_scale_log2e * S_INV2PI_SCALE;
  float c_cur = qsc * clist[0];
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  read_k_frags(0);
#pragma unroll
  for (int ks = 0; ks < KS; ks++) qk_step(ks);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // K(0) is in registers: its stage may be refilled
  __builtin_amdgcn_s_barrier();

  // One block; `acc` holds its S^T on entry and that of the next block on exit.  st = it % 2.
  auto step = [&](int it, int st) {
    load_k(kb_2, st);        // K(it+2) into the stage K(it) has left
    load_v(kb_1, st ^ 1);    // V(it+1) into the stage V(it-1) has left
    const int kidx_v = (int)klist[it + 3];
    const float c_next = qsc * clist[it + 1];
    const float c = c_cur;
    float bias = fmaf(-S_INV2PI_F, c, m_off);   // t = S*c - m + OFFSET from the biased score

    float s[2][16];
#pragma unroll
    for (int mt = 0; mt < 2; mt++)
#pragma unroll
      for (int i = 0; i < 16; i++) s[mt][i] = __int_as_float(acc[mt][i]);

    // -- columns past the end of K (last block) or above the diagonal (causal) leave the softmax
    const bool edge = (kb_c == p.nbk - 1 && (p.Nk & 63) != 0) || (causal && kb_c == qb);
    if (edge) {
      int kb_e = kb_c;
      asm volatile("" : "+s"(kb_e));   // opaque: otherwise 32 lane masks are hoisted into scalar registers
      int thr = p.Nk - kb_e * 64 - 4 * lh;
      if (causal) thr = min(thr, qrow + 1 - kb_e * 64 - 4 * lh);
#pragma unroll
      for (int mt = 0; mt < 2; mt++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
          const int cidx = 32 * mt + 8 * (i >> 2) + (i & 3);
          if (cidx >= thr) s[mt][i] = -INFINITY;
        }
    }

    // -- weights: float16, in the order the B fragments of the four steps take them.  Optimistic about the maximum:
    //    a weight beyond float16 (a score more than eleven octaves above the running maximum) becomes infinite and
    //    shows in the row sums, which are taken before anything else uses the weights; only then, and in the first
    //    block, is the block's maximum searched, O and the sums rescaled, and the weights computed again.
    float rs;
    v4f d_new;
    auto weights = [&]() {
      rs = 0.f;
#pragma unroll
      for (int k = 0; k < 4; k++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const int mt = k >> 1, i = 8 * (k & 1) + 2 * j;
          v2f w;
          w[0] = __builtin_amdgcn_exp2f(fmaf(s[mt][i], c, bias));
          w[1] = __builtin_amdgcn_exp2f(fmaf(s[mt][i + 1], c, bias));
          if constexpr (LSE) {
            rs += w[0] + w[1];
            asm volatile("" : "+v"(rs));   // (taken here: deferred to the weights' acceptance, the sum would keep all of them)
          }
          const v2h hw = __builtin_convertvector(w, v2h);
          pf[k][2 * j] = hw[0];
          pf[k][2 * j + 1] = hw[1];
        }
      d_new = d_acc;
#pragma unroll
      for (int k = 0; k < 4; k++) d_new = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, pf[k], d_new, 0, 0, 0);
    };
    weights();
    __builtin_amdgcn_sched_barrier(0);
    read_k_frags(st ^ 1);   // issued here: they cover the latency of the row sums
    __builtin_amdgcn_sched_barrier(0);
    if (it == 0 || __ballot(!(d_new[0] + d_new[1] < INFINITY)) != 0ull) {
      float mx0 = max3(s[0][0], s[0][1], s[0][2]), mx1 = max3(s[0][8], s[0][9], s[0][10]);
      float mx2 = max3(s[1][0], s[1][1], s[1][2]), mx3 = max3(s[1][8], s[1][9], s[1][10]);
#pragma unroll
      for (int i = 3; i < 7; i += 2) {
        mx0 = max3(mx0, s[0][i], s[0][i + 1]);
        mx1 = max3(mx1, s[0][i + 8], s[0][i + 9]);
        mx2 = max3(mx2, s[1][i], s[1][i + 1]);
        mx3 = max3(mx3, s[1][i + 8], s[1][i + 9]);
      }
      mx0 = max3(mx0, s[0][7], s[0][15]);
      mx2 = max3(mx2, s[1][7], s[1][15]);
      const float smax = max3(max3(mx0, mx1, mx2), mx3, mx3);
      const float m_new = fmaxf(m_i, fmaf(partner_max(smax), c, -S_INV2PI_F * c));
      const float alpha = __builtin_amdgcn_exp2f(m_i - m_new);
      m_i = m_new;
      m_off = P_EXP_OFFSET - m_new;
      bias = fmaf(-S_INV2PI_F, c, m_off);
      if constexpr (LSE) d_exact *= alpha;
      d_acc[0] *= alpha;                                   // lanes 0..15: q-row lane
      d_acc[1] *= __shfl(alpha, (lane & 15) + 16, 64);     // and q-row lane + 16
#pragma unroll
      for (int dt = 0; dt < DT_TILES; dt++)
#pragma unroll
        for (int i = 0; i < 16; i++) o_acc[dt][i] *= alpha;
      weights();
    }
    d_acc = d_new;
    if constexpr (LSE) d_exact += rs;
    __builtin_amdgcn_sched_barrier(0);

    // -- matrix phase: S^T of the next block, then O^T += V^T . P~^T
    read_v_frags(st, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < KS; ks++) qk_step(ks);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < 4; k++) {
#pragma unroll
      for (int dt = 0; dt < DT_TILES; dt++) o_acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vfrag[dt], pf[k], o_acc[dt], 0, 0, 0);
      if (k < 3) read_v_frags(st, k + 1);
    }
    __builtin_amdgcn_sched_barrier(0);

    // -- the next block's tiles have to have landed before the barrier publishes them; the barrier also says
    //    that every wave is done reading this stage
    const int kb_3 = __builtin_amdgcn_readfirstlane(kidx_v);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    kb_c = kb_1; kb_1 = kb_2; kb_2 = kb_3;
    c_cur = c_next;
  };
  for (int it = 0; it < cnt; it += 2) {
    step(it, 0);
    if (it + 1 >= cnt) break;
    step(it + 1, 1);
  }

  // ---- epilogue: O = O~ / d (times v_scale plus v_mean when the caller gives them) ----
  const float d_lo = __shfl(d_acc[0], l32 & 15, 64), d_hi = __shfl(d_acc[1], l32 & 15, 64);
  const float inv = 1.0f / (l32 < 16 ? d_lo : d_hi);
  if (qrow < p.Nq) {
    unsigned short* outp = out_row_ptr();
    const float* vsc = p.v_scale ? p.v_scale + bhk * D : nullptr;
    const float* vmn = p.v_mean ? p.v_mean + bhk * D : nullptr;
#pragma unroll
    for (int dt = 0; dt < DT_TILES; dt++) {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int ch = 32 * dt + 8 * g + 4 * lh;
        v4f sc = {1.f, 1.f, 1.f, 1.f}, mn = {0.f, 0.f, 0.f, 0.f};
        if (vsc) sc = *reinterpret_cast<const v4f*>(vsc + ch);
        if (vmn) mn = *reinterpret_cast<const v4f*>(vmn + ch);
        unsigned short r[4];
#pragma unroll
        for (int q = 0; q < 4; q++) r[q] = OutT::from_f32(fmaf(o_acc[dt][4 * g + q] * inv, sc[q], mn[q]));
        *reinterpret_cast<v2i*>(outp + ch) =
            v2i{(int)((unsigned)r[0] | ((unsigned)r[1] << 16)), (int)((unsigned)r[2] | ((unsigned)r[3] << 16))};
      }
    }
  }
  if constexpr (LSE) {   // (the exact sum of the weights before their rounding)
    const float d_full = d_exact + __shfl_xor(d_exact, 32, 64);
    if (qrow < p.Nq && lh == 0)
      store_lse(p, ((int64_t)b * p.H + h) * p.Nq + qrow, m_i + __builtin_amdgcn_logf(d_full) - P_EXP_OFFSET);
  }
}

template <int D, int OUT_DT, bool LSE, bool Q16>
static int launch_pv16(const AttnParams& p, bool causal, hipStream_t st) {
  const size_t smem = Pv16Lds<D>::LIST_OFF + (((size_t)(p.nbk + Pv16Lds<D>::LIST_PAD + 1) * 6 + 15) & ~(size_t)15);
  PARO_CHECK(smem <= 160 * 1024, PARO_ERR_RUNTIME, "kv_len %d: the list of %d key blocks does not fit the local data share",
             p.Nk, p.nbk);
  const int grid = ((p.total + 7) / 8) * 8;
  auto kern = attn_sparse_pv16_kernel<D, OUT_DT, LSE, Q16>;
  if (smem > 48 * 1024)
    PARO_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
  hipLaunchKernelGGL(kern, dim3(grid), dim3(128), smem, st, p, causal ? 1 : 0);
  PARO_HIP(hipGetLastError());
  return PARO_OK;
}

template <int D, int OUT_DT>
static int dispatch_pv16(const AttnParams& p, bool causal, hipStream_t st) {
  if (p.q16 != nullptr)
    return p.lse != nullptr ? launch_pv16<D, OUT_DT, true, true>(p, causal, st) : launch_pv16<D, OUT_DT, false, true>(p, causal, st);
  return p.lse != nullptr ? launch_pv16<D, OUT_DT, true, false>(p, causal, st) : launch_pv16<D, OUT_DT, false, false>(p, causal, st);
}

int launch_attn_pv16(const AttnParams& p, int D, int out_dtype, bool causal, hipStream_t st) {
  if (D == 64)
    return out_dtype == PARO_DTYPE_F16 ? dispatch_pv16<64, PARO_DTYPE_F16>(p, causal, st) : dispatch_pv16<64, PARO_DTYPE_BF16>(p, causal, st);
  return out_dtype == PARO_DTYPE_F16 ? dispatch_pv16<128, PARO_DTYPE_F16>(p, causal, st) : dispatch_pv16<128, PARO_DTYPE_BF16>(p, causal, st);
}

// ---- V -> float16 tiles in fragment order: one workgroup per (batch, kv-head, 64-token block) ----
template <int DT, int D>
__global__ void __launch_bounds__(256) v_f16_pack_kernel(const unsigned short* __restrict__ v, unsigned short* __restrict__ out,
                                                         int Hkv, int N, int nb, int64_t sb, int64_t sh, int64_t sn) {
  const int kb = blockIdx.x % nb, bh = blockIdx.x / nb;
  v_f16_pack_body<DT, D>(v + bh / Hkv * sb + bh % Hkv * sh, out, N, nb, sn, kb, bh);
}

}  // namespace paro

extern "C" int64_t paro_v_f16_bytes(int B, int Hkv, int N, int D) {
  return (int64_t)B * Hkv * ((N + 63) / 64) * 64 * D * 2;
}

extern "C" int paro_v_f16_pack(const void* v, int dtype, void* v16, int B, int Hkv, int N, int D, int64_t v_stride_b,
                               int64_t v_stride_h, int64_t v_stride_n, void* stream) {
  using namespace paro;
  PARO_CHECK(v && v16, PARO_ERR_RUNTIME, "paro_v_f16_pack: null tensor pointer");
  PARO_CHECK(B > 0 && Hkv > 0 && N > 0, PARO_ERR_RUNTIME, "paro_v_f16_pack: empty shape");
  PARO_CHECK(D == 64 || D == 128, PARO_ERR_INVALID_VALUE, "Unsupported head dim: %d", D);
  PARO_CHECK(dtype == PARO_DTYPE_F16 || dtype == PARO_DTYPE_BF16, PARO_ERR_RUNTIME,
             "Unsupported input dtype (expect float16 or bfloat16)");
  PARO_CHECK(((uintptr_t)v % 16) == 0 && ((uintptr_t)v16 % 16) == 0 && v_stride_b % 8 == 0 && v_stride_h % 8 == 0 &&
                 v_stride_n % 8 == 0,
             PARO_ERR_RUNTIME, "Tensor value must be 16-byte aligned with strides that are multiples of 8");
  const int nb = (N + 63) / 64;
  PARO_CHECK((int64_t)B * Hkv * nb < (int64_t)1 << 31, PARO_ERR_RUNTIME, "paro_v_f16_pack: too many blocks");
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)(B * Hkv * nb));
#define PARO_V16(DTC, DD)                                                                                          \
  hipLaunchKernelGGL((v_f16_pack_kernel<DTC, DD>), grid, dim3(256), 0, st, (const unsigned short*)v,                \
                     (unsigned short*)v16, Hkv, N, nb, v_stride_b, v_stride_h, v_stride_n)
  if (dtype == PARO_DTYPE_F16) {
    if (D == 64) PARO_V16(PARO_DTYPE_F16, 64); else PARO_V16(PARO_DTYPE_F16, 128);
  } else {
    if (D == 64) PARO_V16(PARO_DTYPE_BF16, 64); else PARO_V16(PARO_DTYPE_BF16, 128);
  }
#undef PARO_V16
  PARO_HIP(hipGetLastError());
  return PARO_OK;
}
