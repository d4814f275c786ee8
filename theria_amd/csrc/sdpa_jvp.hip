// Frozen-stats SDPA JVP for gfx950.
//
// Replaces the eager sdpa_jvp of the reference (theria/attention/triton_sdpa_backward.py:465-503),
// which materialises several (B,H,T,M) float32 tensors. Contract (docs/phase9.md:30-39): P is rebuilt
// from the saved row statistics and held fixed, and with tangents (tq, tk, tv)
//   G = scale (tq K^T + Q tk^T),  c_i = sum_j P_ij G_ij,
//   tO = P o (G - c) V + P tv = (P o G) V - c o O + P tv,
// where O = P V (the saved forward output, or rebuilt in the same pass when it is not supplied).
// The same kernel yields the G_dO output of the double backward (tangents = cotangents of dQ, dK, dV).
//
// 16-bit inputs: the two large terms (P o G) V and c o O of tO cancel, so operand rounding in them is
// amplified (a bfloat16-rounded P o G gave 0.03 absolute error on a row with four visible keys). Both
// products are therefore formed from two-term 16-bit splits (hi + lo) of P o G and of P, and O is always
// rebuilt in the pass from the same P (the saved O, rounded to 16 bits, is not used). The key-split kernel
// (jvp_ksplit_kernel, below) takes the split at head dims up to 64 only in waves holding a row flagged peaked in lse:
// elsewhere the rounding of P o G and P spreads over many keys and one 16-bit term each keeps the 16-bit bar.
// p.normalize divides P by its own row sum (every dtype): the JVP of the exact softmax for an lse this
// library's forward wrote (a 16-bit forward's lse comes from rounded probabilities, so P rebuilt from it
// sums to 1 only within ~2^-9). Without it P = exp(S - lse) is held exactly as given, which is the
// reference's frozen-stats contract for caller-supplied (m, l).
//
// Work decomposition as in the forward: one workgroup = 4 waves = 128 query rows, lane per query in
// the transposed score tiles S^T = K Q^T and G^T = K tq^T + tk Q^T (Q and tq stay in registers as B
// operands); per 64-key tile, K, tk, V, tv are staged in LDS and the three output products
// (P o G) V, P tv and (if needed) P V accumulate lane-per-query as V^T (.)^T, with V^T / tv^T
// fragments from the LDS transpose read. A single pass: c_i is folded in at the end.
#include <initializer_list>
#include <type_traits>

#include "dispatch.hpp"
#include "sdpa_common.hpp"
#include "sdpa_lds.hpp"

namespace theria {

// Tiles pass through registers into padded LDS rows. NW: waves per workgroup, four or two (at most 64 queries).
template <typename T, int DP, bool CAUSAL, bool HAS_O, int NW = 4>
__global__ __launch_bounds__(64 * NW, sizeof(T) == 4 && DP == 32 ? 2 : 1) void jvp_kernel(const JvpParams p) {
  // float32 forms its scores as the forward does, from split operands: lse was rounded with those scores, and scores of
  // another order of rounding don't cancel its error (T20 M90 D80 std 2, 2-norm against float64: 1.20e-6 -> 7.3e-7).
  // Above head dim 64 this also beats the float32 MFMA, ~40 spilled registers included (us: B4 H8 T700 D128 276 -> 188,
  // B16 H16 T300 D128 causal 381 -> 282, B300 H8 T20 M90 D80 438 -> 394).
  using OP = Ops<T, DP>;
  using F = typename OP::F;
  constexpr int KC = OP::KC;
  constexpr int BM = 32 * NW, NT = 64 * NW;
  constexpr int BN = (DP == 128 || sizeof(T) == 4) ? 32 : 64;  // keys per tile (register budget)
  constexpr int PITCH = OP::PITCH;
  constexpr int NDT = DP / 32, NKC = DP / KC, NPC = 32 / KC, NST = BN / 32;
  __shared__ __attribute__((aligned(16))) T sK0[BN * PITCH], sV0[BN * PITCH], stK0[BN * PITCH], stV0[BN * PITCH];

  const Shape& s = p.s;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 31, g = lane >> 5;
  const int nqb = (s.T + BM - 1) / BM;
  const int bid = xcd_remap(blockIdx.x, gridDim.x);
  const int bh = bid / nqb;
  int qb = bid - bh * nqb;
  if (CAUSAL) qb = nqb - 1 - qb;
  const int b = bh / s.H, h = bh - b * s.H;
  const T* Q = (const T*)p.q.p + b * p.q.sb + h * p.q.sh;
  const T* K = (const T*)p.k.p + b * p.k.sb + h * p.k.sh;
  const T* V = (const T*)p.v.p + b * p.v.sb + h * p.v.sh;
  const bool has_tq = p.tq.p != nullptr, has_tk = p.tk.p != nullptr, has_tv = p.tv.p != nullptr;
  const T* TQ = has_tq ? (const T*)p.tq.p + b * p.tq.sb + h * p.tq.sh : nullptr;
  const T* TK = has_tk ? (const T*)p.tk.p + b * p.tk.sb + h * p.tk.sh : nullptr;
  const T* TV = has_tv ? (const T*)p.tv.p + b * p.tv.sb + h * p.tv.sh : nullptr;
  const int q0w = qb * BM + wave * 32;
  const int myq = q0w + li;
  const bool qvalid = myq < s.T;
  const int64_t row_id = (int64_t)bh * s.T + myq;

  F qf[NKC], tqf[NKC];
  {
    typename OP::Raw qraw[NKC], tqraw[NKC];
#pragma unroll
    for (int c = 0; c < NKC; ++c) {
      qraw[c] = OP::raw(Q, p.q.sr, myq, s.T, c, s.D, s.vec);
      tqraw[c] = has_tq ? OP::raw(TQ, p.tq.sr, myq, s.T, c, s.D, s.vec) : typename OP::Raw{};
    }
#pragma unroll
    for (int c = 0; c < NKC; ++c) {
      qf[c] = OP::frag(qraw[c]);
      tqf[c] = OP::frag(tqraw[c]);
    }
  }
  f32x16_t accA[NDT], accC[NDT], accO[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) {
    accA[dt] = zero16();
    accC[dt] = zero16();
    accO[dt] = zero16();
  }
  const float c2 = s.scale * kLog2e;
  const float lse2 = qvalid ? p.lse[row_id] * kLog2e : THERIA_INF;
  const float moff = lse2 == -THERIA_INF ? THERIA_INF : lse2;  // a row without visible keys has P = 0
  constexpr bool SPLIT = sizeof(T) == 2;     // hi/lo operands, renormalised P (see the header)
  constexpr bool REBUILD = SPLIT || !HAS_O;  // O = P V formed in this pass
  float cpart = 0.f, lpart = 0.f;

  int kend = s.M;
  if (CAUSAL) kend = min(s.M, qb * BM + BM);
  const int nkt = (kend + BN - 1) / BN;
  // The key tile kt held in (tK, tV, ttK, ttV).
  auto compute = [&](auto mask_tag, int kt, const T* tK, const T* tV, const T* ttK, const T* ttV) __attribute__((always_inline)) {
    constexpr bool MASK = decltype(mask_tag)::value;
    const int k0 = kt * BN;
    if (CAUSAL && k0 > q0w + 31) return;

    f32x16_t sc[NST], gm[NST];
#pragma unroll
    for (int t = 0; t < NST; ++t) {
      sc[t] = zero16();
      gm[t] = zero16();
#pragma unroll
      for (int c = 0; c < NKC; ++c) {
        const F kfr = OP::cols(tK, t * 32 + li, c);
        sc[t] = OP::mma(kfr, qf[c], sc[t]);
        if (has_tq) gm[t] = OP::mma(kfr, tqf[c], gm[t]);
        if (has_tk) gm[t] = OP::mma(OP::cols(ttK, t * 32 + li, c), qf[c], gm[t]);
      }
    }
#pragma unroll
    for (int t = 0; t < NST; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float pv = fast_exp2(fmaf(sc[t][r], c2, -moff));
        if constexpr (MASK) {
          const int key = k0 + t * 32 + acc_row(r, g);
          if (key >= s.M || (CAUSAL && key > myq)) pv = 0.f;
        }
        sc[t][r] = pv;
        lpart += pv;
        const float pg = pv * gm[t][r];
        gm[t][r] = pg;
        cpart += pg;
      }
#pragma unroll
    for (int t = 0; t < NST; ++t)
#pragma unroll
      for (int cc = 0; cc < NPC; ++cc) {
        F pf, pgf, pf_lo{}, pgf_lo{};
        if constexpr (SPLIT) {
          split_frag<T>(sc[t], cc, pf, pf_lo);
          split_frag<T>(gm[t], cc, pgf, pgf_lo);
        } else {
          pf = OP::acc(sc[t], cc);
          pgf = OP::acc(gm[t], cc);
        }
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
          const F vfr = OP::rows(tV, t * 32, cc, dt * 32);
          accA[dt] = OP::mma(vfr, pgf, accA[dt]);
          if (SPLIT) accA[dt] = OP::mma(vfr, pgf_lo, accA[dt]);
          if (REBUILD) accO[dt] = OP::mma(vfr, pf, accO[dt]);
          if (REBUILD && SPLIT) accO[dt] = OP::mma(vfr, pf_lo, accO[dt]);
          if (has_tv) accC[dt] = OP::mma(OP::rows(ttV, t * 32, cc, dt * 32), pf, accC[dt]);
        }
      }
  };

  {
    TileStage<T, BN, DP, NT> gK, gV, gtK, gtV;
    auto prefetch = [&](int k0) {
      gK.load(K, p.k.sr, k0, s.M, s.D, s.vec);
      gV.load(V, p.v.sr, k0, s.M, s.D, s.vec);
      if (has_tk) gtK.load(TK, p.tk.sr, k0, s.M, s.D, s.vec);
      if (has_tv) gtV.load(TV, p.tv.sr, k0, s.M, s.D, s.vec);
    };
    if (nkt > 0) prefetch(0);
    auto step = [&](auto mask_tag, int kt) __attribute__((always_inline)) {
      __syncthreads();
      OP::store(gK, sK0, true, gV, sV0, true, gtK, stK0, has_tk, gtV, stV0, has_tv);
      __syncthreads();
      if (kt + 1 < nkt) prefetch((kt + 1) * BN);
      compute(mask_tag, kt, sK0, sV0, stK0, stV0);
    };
    // the tiles with every key in range and visible to the block, then the others with the mask
    const int nfull = min(nkt, CAUSAL ? min(s.M / BN, qb * BM / BN) : s.M / BN);
    int kt = 0;
    for (; kt < nfull; ++kt) step(std::false_type{}, kt);
    for (; kt < nkt; ++kt) step(std::true_type{}, kt);
  }

  // normalize: P / L with L = sum_j P_j, i.e. every term below is divided by L (and a rebuilt O as well)
  float inv = 1.f;
  if (p.normalize) {
    const float L = pair_sum(lpart);
    inv = L > 0.f ? 1.f / L : 0.f;
  }
  const float cval = pair_sum(cpart) * s.scale * inv;
  if (qvalid) {
    const T* O = (HAS_O && !REBUILD) ? (const T*)p.o.p + b * p.o.sb + h * p.o.sh : nullptr;
    T* TO = (T*)p.tout.p + b * p.tout.sb + h * p.tout.sh;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const int d0 = dt * 32 + 8 * qd + 4 * g;
        if (d0 < s.D) {
          f32x4_t ov;
          if (!REBUILD) {
            ov = load4<T>(O, p.o.sr, myq, d0, s.D, s.vec);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) ov[e] = accO[dt][4 * qd + e] * inv;
          }
          float r4[4];
#pragma unroll
          for (int e = 0; e < 4; ++e)
            r4[e] = inv * (s.scale * accA[dt][4 * qd + e] + accC[dt][4 * qd + e]) - cval * ov[e];
          store4<T>(TO, p.tout.sr, myq, d0, s.D, r4[0], r4[1], r4[2], r4[3], s.vec);
        }
      }
  }
}

// 16-bit inputs with LDS-DMA tiles (a head dim that is a multiple of 8, computed at DP = 64 or 128 with the tile columns
// past D zero): the same JVP with the keys of a query block split between two groups. DP = 64: groups of four waves
// (eight-wave workgroups), so that a SIMD holds two waves at 256 registers each
// where jvp_kernel holds one at ~380 (config 4: B H T / 32 = 1024 query waves for 1024 SIMDs; 27.1 -> 23.0 us
// there, same box). Each group streams its own half of the key tiles (64 keys per tile, 128 KB of LDS in
// all) through its own double-buffered tiles; both groups meet at the same barrier every step (a group
// whose half is shorter idles through the last step). The float32 partial sums of group 1 (accumulators,
// row sums) are exchanged through LDS at the end. DP = 128, whose accumulators take a whole SIMD per wave: G = 2 groups of
// two waves (64 queries, 32-key tiles) where 128-query workgroups would leave CUs idle, else G = 1 group of four waves
// (128 queries, no exchange), which reads each tile for twice the queries (us, the one-group kernel it replaced -> G = 2 /
// G = 1, bfloat16 D128: B2 H8 T1024 84 -> 46 / 62, B2 H16 T1024 90 -> 84 / 74, B1 H4 T8192 601 -> 511 / 457, B64 H8 T1000
// M96 250 -> 320 / 217, B2 H8 T1024 causal 84 -> 36 / 56; with one 16-bit term instead of two the better of each took 39, 59,
// 354, 217 and 30 us, at 1.4 times the error). ALL: every tangent is given (the presence tests are then
// constants, and the loop body has no branches between its products).
template <typename T, bool CAUSAL, bool ALL, bool FD, int DP, int G>
__global__ __launch_bounds__(DP == 64 ? 512 : 256, DP == 64 ? 2 : 1) void jvp_ksplit_kernel(const JvpParams p) {
  using MM = Mfma<T>;
  using F = typename MM::frag_t;
  static_assert(sizeof(T) == 2, "16-bit inputs only");
  static_assert(G == 2 || DP == 128, "one group only at DP = 128");
  constexpr int NW = DP == 64 ? 4 : 4 / G, GT = 64 * NW, BM = 32 * NW, BN = DP == 64 ? 64 : 32, NST = BN / 32;
  constexpr int NDT = DP / 32, NKC = DP / MM::KC, NPC = 32 / MM::KC;
  constexpr int TB = BN * DP * 2;  // bytes per tile
  // DP = 64: each group fills its own tiles; 128: all four waves fill both groups' (a slab is then 16 rows)
  constexpr bool JOINT = DP == 128 && G == 2;
  using Dma = SwzDma<4, DP>;
  constexpr int NSLAB = BN / Dma::SLAB_ROWS;
  static_assert(NSLAB * Dma::SLAB_ROWS == BN, "key tiles must be whole DMA slabs");
  // [group][set][K, V, tK, tV]; reused for the partial sums after the key loop
  __shared__ __attribute__((aligned(1024))) char smem[G * 2 * 4 * TB];
  static_assert(G == 1 || sizeof(smem) >= (NDT * 3 * 16 + 4) * GT * 4, "the partial sums fit in the tile memory");

  const Shape& s = p.s;
  const int lane = threadIdx.x & 63, li = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = (unsigned)wave / NW, wig = (unsigned)wave % NW;  // key group, wave in group
  const int nqb = (s.T + BM - 1) / BM;
  const int bid = xcd_remap(blockIdx.x, gridDim.x);
  const int bh = bid / nqb;
  int qb = bid - bh * nqb;
  if (CAUSAL) qb = nqb - 1 - qb;
  const int b = bh / s.H, h = bh - b * s.H;
  const T* Q = (const T*)p.q.p + b * p.q.sb + h * p.q.sh;
  const T* K = (const T*)p.k.p + b * p.k.sb + h * p.k.sh;
  const T* V = (const T*)p.v.p + b * p.v.sb + h * p.v.sh;
  const bool has_tq = ALL || p.tq.p != nullptr, has_tk = ALL || p.tk.p != nullptr, has_tv = ALL || p.tv.p != nullptr;
  const T* TQ = has_tq ? (const T*)p.tq.p + b * p.tq.sb + h * p.tq.sh : nullptr;
  const T* TK = has_tk ? (const T*)p.tk.p + b * p.tk.sb + h * p.tk.sh : nullptr;
  const T* TV = has_tv ? (const T*)p.tv.p + b * p.tv.sb + h * p.tv.sh : nullptr;
  const int q0w = qb * BM + wig * 32;
  const int myq = q0w + li;
  const bool qvalid = myq < s.T;
  const int64_t row_id = (int64_t)bh * s.T + myq;

  F qf[NKC], tqf[NKC];
#pragma unroll
  for (int c = 0; c < NKC; ++c) {
    qf[c] = gload_frag<T>(Q, p.q.sr, myq, s.T, c, s.D, s.vec);
    tqf[c] = has_tq ? gload_frag<T>(TQ, p.tq.sr, myq, s.T, c, s.D, s.vec) : F{};
  }
  f32x16_t accA[NDT], accC[NDT], accO[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) {
    accA[dt] = zero16();
    accC[dt] = zero16();
    accO[dt] = zero16();
  }
  const float c2 = s.scale * kLog2e;
  const float lse_raw = qvalid ? p.lse[row_id] : THERIA_INF;
  const float lse2 = lse_raw * kLog2e;
  const float moff = lse2 == -THERIA_INF ? THERIA_INF : lse2;  // a row without visible keys has P = 0
  float cpart = 0.f, lpart = 0.f;
  // DP = 64: the two-term products only in waves holding a row flagged peaked in lse (a dominant probability, which
  // rows with few visible keys have): there (P o G) V and c o O cancel. Elsewhere the rounding of P o G and
  // P spreads over many keys and one 16-bit term each keeps the bar (uniform per wave). DP = 128: every wave, so that
  // nothing but the rounding of the output shows (and a caller's lse, which carries no flags, decides nothing).
  const bool split = DP == 128 || __any(lse_peaked(lse_raw));

  int kend = s.M;
  if (CAUSAL) kend = min(s.M, qb * BM + BM);
  const int nkt = (kend + BN - 1) / BN;
  const int half = (nkt + G - 1) / G;
  const int kt0 = grp * half, kt1 = min(nkt, kt0 + half);  // this group's tiles [kt0, kt1)

  // The key tile kt held in (tK, tV, ttK, ttV): as jvp_kernel, 32-key subtiles one after the other. MASK: the
  // tile reaches past the last key or (causal) past this wave's first query.
  auto compute = [&](auto split_tag, auto mask_tag, int kt, const char* tK, const char* tV, const char* ttK,
                     const char* ttV) __attribute__((always_inline)) {
    constexpr bool SPLIT = decltype(split_tag)::value;
    constexpr bool MASK = decltype(mask_tag)::value;
#pragma unroll
    for (int st = 0; st < NST; ++st) {
      const int k0 = kt * BN + 32 * st;
      if (CAUSAL && k0 > q0w + 31) continue;
      f32x16_t sc = zero16(), gm = zero16();
#pragma unroll
      for (int c = 0; c < NKC; ++c) {
        const F kfr = swz_cols<T, DP>(tK, 32 * st + li, c);
        sc = MM::mma(kfr, qf[c], sc);
        if (has_tq) gm = MM::mma(kfr, tqf[c], gm);
        if (has_tk) gm = MM::mma(swz_cols<T, DP>(ttK, 32 * st + li, c), qf[c], gm);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float pv = fast_exp2(fmaf(sc[r], c2, -moff));
        if constexpr (MASK) {
          const int key = k0 + acc_row(r, g);
          if (key >= s.M || (CAUSAL && key > myq)) pv = 0.f;
        }
        sc[r] = pv;
        lpart += pv;
        const float pg = pv * gm[r];
        gm[r] = pg;
        cpart += pg;
      }
      if constexpr (SPLIT) {
#pragma unroll
        for (int cc = 0; cc < NPC; ++cc) {
          F pf, pf_lo, pgf, pgf_lo;
          split_frag<T>(sc, cc, pf, pf_lo);
          split_frag<T>(gm, cc, pgf, pgf_lo);
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) {
            const F vfr = swz_rows<T, DP>(tV, 32 * st, cc, dt * 32);
            accA[dt] = MM::mma(vfr, pgf, accA[dt]);
            accA[dt] = MM::mma(vfr, pgf_lo, accA[dt]);
            accO[dt] = MM::mma(vfr, pf, accO[dt]);
            accO[dt] = MM::mma(vfr, pf_lo, accO[dt]);
            if (has_tv) accC[dt] = MM::mma(swz_rows<T, DP>(ttV, 32 * st, cc, dt * 32), pf, accC[dt]);
          }
        }
      } else {
#pragma unroll
        for (int cc = 0; cc < NPC; ++cc) {
          const F pf = acc_frag<T>(sc, cc), pgf = acc_frag<T>(gm, cc);
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) {
            const F vfr = swz_rows<T, DP>(tV, 32 * st, cc, dt * 32);
            accA[dt] = MM::mma(vfr, pgf, accA[dt]);
            accO[dt] = MM::mma(vfr, pf, accO[dt]);
            if (has_tv) accC[dt] = MM::mma(swz_rows<T, DP>(ttV, 32 * st, cc, dt * 32), pf, accC[dt]);
          }
        }
      }
    }
  };

  // Head dims below DP (a multiple of 8): the tiles' columns past D are filled with zeros by the DMA.
  const Dma dma(JOINT ? wave : wig, lane, FD ? DP / 8 : s.D / 8);  // FD: head dim DP
  // Byte offsets fit in 32 bits: the host only selects this path when each (batch, head) slab of K, V, tK
  // and tV spans less than 2^31 bytes.
  const uint32_t krs = (uint32_t)p.k.sr * 2, vrs = (uint32_t)p.v.sr * 2;
  const uint32_t tkrs = has_tk ? (uint32_t)p.tk.sr * 2 : 0u, tvrs = has_tv ? (uint32_t)p.tv.sr * 2 : 0u;
  const int64_t rb = 2 * (FD ? DP : s.D);  // bytes of a row the DMA reads
  const rsrc_t krsrc = make_rsrc(K, (uint32_t)slab_span(s.M, krs, rb)),
               vrsrc = make_rsrc(V, (uint32_t)slab_span(s.M, vrs, rb));
  const rsrc_t tkrsrc = make_rsrc(has_tk ? (const void*)TK : (const void*)K, (uint32_t)slab_span(s.M, tkrs, rb));
  const rsrc_t tvrsrc = make_rsrc(has_tv ? (const void*)TV : (const void*)V, (uint32_t)slab_span(s.M, tvrs, rb));
  auto tile_of = [&](int gg, int set, int a) { return smem + ((gg * 2 + set) * 4 + a) * TB; };  // a: K, V, tK, tV
  auto tile = [&](int set, int a) { return tile_of(grp, set, a); };
  auto issue_one = [&](int gg, int kt, int set) __attribute__((always_inline)) {
    const int k0 = kt * BN;
    dma.template issue_clamped<NSLAB>(krsrc, krs, k0, s.M, tile_of(gg, set, 0));
    dma.template issue_clamped<NSLAB>(vrsrc, vrs, k0, s.M, tile_of(gg, set, 1));
    if (has_tk) dma.template issue_clamped<NSLAB>(tkrsrc, tkrs, k0, s.M, tile_of(gg, set, 2));
    if (has_tv) dma.template issue_clamped<NSLAB>(tvrsrc, tvrs, k0, s.M, tile_of(gg, set, 3));
  };
  auto issue_joint = [&](int i) __attribute__((always_inline)) {  // step i's tiles of both groups
    if (i < half) issue_one(0, i, i & 1);
    if (i < half && half + i < nkt) issue_one(1, half + i, i & 1);
  };
  // Step i: tile kt0 + i of this group (if it has one) from set i & 1; the next one's copies go to the other
  // set, read in step i - 1, which every wave has finished at the barrier. The tiles from mask_from on may
  // reach past the last key or (causal) past the block's first query and take the masked copy of the loop;
  // the groups may be in different copies at a step, but both meet the same barriers.
  const int mask_from = min(kend % BN ? nkt - 1 : nkt, CAUSAL ? qb * BM / BN : nkt);
  auto sweep = [&](auto split_tag) __attribute__((always_inline)) {
    auto step = [&](auto mask_tag, int i) __attribute__((always_inline)) {
      const int kt = kt0 + i;
      wait_vm_all();
      __syncthreads();
      if constexpr (JOINT)
        issue_joint(i + 1);
      else if (kt + 1 < kt1)
        issue_one(grp, kt + 1, (i + 1) & 1);
      if (kt < kt1) compute(split_tag, mask_tag, kt, tile(i & 1, 0), tile(i & 1, 1), tile(i & 1, 2), tile(i & 1, 3));
    };
    const int isplit = min(half, max(0, mask_from - kt0));
    int i = 0;
    for (; i < isplit; ++i) step(std::false_type{}, i);
    for (; i < half; ++i) step(std::true_type{}, i);
  };
  if constexpr (JOINT)
    issue_joint(0);
  else if (kt0 < kt1)
    issue_one(grp, kt0, 0);
  // The waves of a workgroup may take different copies of the loop: both meet the same barriers.
  if (DP == 128 || split) {
    sweep(std::integral_constant<bool, true>{});
  } else {
    if constexpr (DP == 64) sweep(std::integral_constant<bool, false>{});
  }

  // Epilogue as jvp_kernel's (O rebuilt from the same P; normalize: P divided by its own row sum), for the N column tiles
  // from DT0 on.
  auto store = [&](auto dt0_tag, auto n_tag) __attribute__((always_inline)) {
    constexpr int DT0 = decltype(dt0_tag)::value, N = decltype(n_tag)::value;
    float inv = 1.f;
    if (p.normalize) {
      const float L = pair_sum(lpart);
      inv = L > 0.f ? 1.f / L : 0.f;
    }
    const float cval = pair_sum(cpart) * s.scale * inv;
    if (qvalid) {
      T* TO = (T*)p.tout.p + b * p.tout.sb + h * p.tout.sh;
#pragma unroll
      for (int j = 0; j < N; ++j)
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
          const int dt = DT0 + j, d0 = dt * 32 + 8 * qd + 4 * g;
          float r4[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float ov = accO[dt][4 * qd + e] * inv;
            r4[e] = inv * (s.scale * accA[dt][4 * qd + e] + accC[dt][4 * qd + e]) - cval * ov;
          }
          store4<T>(TO, p.tout.sr, myq, d0, s.D, r4[0], r4[1], r4[2], r4[3], s.vec);
        }
    }
  };
  if constexpr (G == 1) {
    store(std::integral_constant<int, 0>{}, std::integral_constant<int, NDT>{});
    return;
  }
  // The groups finish NH column tiles each (group g the tiles g NH ..): each hands the other's partial sums and its row
  // sums to the other group in one round, 16 bytes per lane per store (elements 4c .. 4c + 3 of accumulator a of tile j
  // of lane l of wave w of group g at words ((((g * NH + j) * 3 + a) * 4 + c) * GT + w * 64 + l) * 4, so one store
  // instruction covers 1 KiB of consecutive words), then stores its part of the output.
  constexpr int NH = NDT / 2;
  float* buf = reinterpret_cast<float*>(smem);
  f32x4_t* buf4 = reinterpret_cast<f32x4_t*>(smem);
  constexpr int RS = NDT * 3 * 4 * GT * 4;  // the row sums, [group][l, c]
  __syncthreads();  // every wave is done with the last tile
  auto finish = [&](auto keep_tag) __attribute__((always_inline)) {
    constexpr int KEEP = decltype(keep_tag)::value, GIVE = 1 - KEEP;
    const int me = wig * 64 + lane;
#pragma unroll
    for (int j = 0; j < NH; ++j)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int i = ((KEEP * NH + j) * 3 * 4 + c) * GT + me, dt = GIVE * NH + j;
        auto q4 = [&](const f32x16_t& a) { return f32x4_t{a[4 * c], a[4 * c + 1], a[4 * c + 2], a[4 * c + 3]}; };
        buf4[i] = q4(accA[dt]);
        buf4[i + 4 * GT] = q4(accO[dt]);
        if (has_tv) buf4[i + 8 * GT] = q4(accC[dt]);
      }
    buf[RS + KEEP * 2 * GT + me] = lpart;
    buf[RS + KEEP * 2 * GT + GT + me] = cpart;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NH; ++j)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int i = ((GIVE * NH + j) * 3 * 4 + c) * GT + me, dt = KEEP * NH + j;
        const f32x4_t a = buf4[i], o4 = buf4[i + 4 * GT];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          accA[dt][4 * c + e] += a[e];
          accO[dt][4 * c + e] += o4[e];
        }
        if (has_tv) {
          const f32x4_t c4 = buf4[i + 8 * GT];
#pragma unroll
          for (int e = 0; e < 4; ++e) accC[dt][4 * c + e] += c4[e];
        }
      }
    lpart += buf[RS + GIVE * 2 * GT + me];
    cpart += buf[RS + GIVE * 2 * GT + GT + me];

    store(std::integral_constant<int, KEEP * NH>{}, std::integral_constant<int, NH>{});
  };
  // both branches meet the one barrier inside finish
  if (grp == 0)
    finish(std::integral_constant<int, 0>{});
  else
    finish(std::integral_constant<int, 1>{});
}

template <bool HAS_O>
struct JvpLauncher {
  template <typename T, int DP, bool CAUSAL>
  static hipError_t run(const JvpParams& p, hipStream_t st) {
    const int nqb = (p.s.T + 127) / 128;
    const int64_t nblk = (int64_t)nqb * p.s.B * p.s.H;
    if (nblk == 0) return hipSuccess;
    if constexpr (sizeof(T) == 2) {
      // LDS-DMA tiles: 16-byte-aligned views, each streamed (batch, head) slab < 2^31 bytes, and a head dim that
      // is a multiple of 8 (columns past D zero-filled)
      bool ok = p.s.vec && p.s.D % 8 == 0;
      for (const View* v : {&p.k, &p.v, &p.tk, &p.tv})
        if (v->p && !slab_fits_dma(p.s.M, v->sr, p.s.D)) ok = false;
      if (ok) {
        const bool all = p.tq.p && p.tk.p && p.tv.p, fd = p.s.D == (DP <= 64 ? 64 : 128);
        auto go = [&](auto kp_tag, auto g_tag) {
          constexpr int KP = decltype(kp_tag)::value, G = decltype(g_tag)::value, BM = KP == 64 ? 128 : 128 / G;
          const dim3 grid((unsigned)((int64_t)((p.s.T + BM - 1) / BM) * p.s.B * p.s.H)), block(KP == 64 ? 512 : 256);
          if (all && fd)
            hipLaunchKernelGGL((jvp_ksplit_kernel<T, CAUSAL, true, true, KP, G>), grid, block, 0, st, p);
          else if (all)
            hipLaunchKernelGGL((jvp_ksplit_kernel<T, CAUSAL, true, false, KP, G>), grid, block, 0, st, p);
          else if (fd)
            hipLaunchKernelGGL((jvp_ksplit_kernel<T, CAUSAL, false, true, KP, G>), grid, block, 0, st, p);
          else
            hipLaunchKernelGGL((jvp_ksplit_kernel<T, CAUSAL, false, false, KP, G>), grid, block, 0, st, p);
        };
        using std::integral_constant;
        if constexpr (DP <= 64)
          go(integral_constant<int, 64>{}, integral_constant<int, 2>{});
        else if (p.s.T > 64 && nblk >= device_cu_count())
          go(integral_constant<int, 128>{}, integral_constant<int, 1>{});
        else
          go(integral_constant<int, 128>{}, integral_constant<int, 2>{});
        return hipGetLastError();
      }
    }
    // at most 64 queries, and more workgroups than CUs (one four-wave workgroup per CU is resident): float32 B400 H4
    // T64 D16 37.4 -> 26.9 us. Not in float32 above head dim 64, where staging a tile with half the threads spills.
    if constexpr (!(sizeof(T) == 4 && DP == 128)) {
      if (p.s.T <= 64 && nblk > device_cu_count()) {
        hipLaunchKernelGGL((jvp_kernel<T, DP, CAUSAL, HAS_O, 2>), dim3((unsigned)nblk), dim3(128), 0, st, p);
        return hipGetLastError();
      }
    }
    hipLaunchKernelGGL((jvp_kernel<T, DP, CAUSAL, HAS_O>), dim3((unsigned)nblk), dim3(256), 0, st, p);
    return hipGetLastError();
  }
};

hipError_t launch_jvp(const JvpParams& p, hipStream_t st) {
  return p.o.p ? dispatch_all<JvpLauncher<true>>(p, st) : dispatch_all<JvpLauncher<false>>(p, st);
}

}  // namespace theria
