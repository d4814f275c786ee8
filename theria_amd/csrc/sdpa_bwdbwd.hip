// SDPA double backward for gfx950: the vector-Jacobian product of the backward map
// (Q, K, V, dO) -> (dQ, dK, dV) with cotangents (gQ, gK, gV).
//
// The reference has no kernel for this (docs/STATUS.md:265-271; its HVP is finite differences of the
// VJP, theria/attention/hvp_utils.py:30-49, or autograd through eager PyTorch,
// theria/autograd/sdpa_custom_function.py:32-53). With s = scale, P from the saved lse,
// dP = dO V^T, z = delta (row term of the backward), dS = P o (dP - z):
//   Gam = s (gQ K^T + Q gK^T),  r_i = sum_j P_ij Gam_ij,   W = dO gV^T,
//   E1  = Gam o (dP - z) + W,   t_i = sum_j P_ij E1_ij,
//   Gbar_dP = P o (Gam - r),    Gbar_S = P o E1 - r o dS - t o P,
//   G_dO = Gbar_dP V + P gV     (the frozen-stats JVP with tangents (gQ, gK, gV): jvp kernel)
//   G_V  = Gbar_dP^T dO
//   G_Q  = s (Gbar_S K + dS gK) = s (sum_j (P o E1)_ij K_j - r_i (dS K)_i - t_i (P K)_i + (dS gK)_i)
//   G_K  = s (Gbar_S^T Q + dS^T gQ)
// (Gbar_S = P o (Gbar_P - s_row) with Gbar_P = E1 - r o dP and s_row = t - r z, rearranged so that a
// single pass over the keys suffices for G_Q.)
//
// rows kernel: lane per query (transposed score tiles, as in the forward). One pass over key tiles (64
//   keys as two 32-key subtiles for 16-bit inputs at head dim <= 64, else 32) accumulates the four D-wide
//   products of the G_Q expression plus r and t, writes G_Q, r, t.
//   16-bit workgroups holding a row flagged peaked in lse are redone after it (as extra workgroups of the
//   cols kernel's grid): with the exact r and t the first launch wrote, Gbar_S = P o ((Gam - r)(dP - z) + W - t)
//   is formed in float32 and, with dS, entered as two 16-bit terms (hi + lo), so that
//   G_Q = s (Gbar_S K + dS gK) is no longer a small difference of large products.
// cols kernel: lane per key (as in the backward). One pass over query tiles (64 queries as two 32-query
//   subtiles for 16-bit inputs at head dim <= 64, else 32) with r, t, z, lse per row staged in LDS
//   accumulates G_V and G_K in registers. 16-bit query tiles holding a row flagged peaked are skipped by
//   that pass and run after it with Gbar_dP, Gbar_S and dS entered as two 16-bit terms each (their sums over
//   many queries are small there).
// 16-bit inputs with a head dim that is a multiple of 8 and LDS-DMA tiles take two split kernels instead
// (sdpa_bwdbwd_split.hip).
#include <type_traits>

#include "dispatch.hpp"
#include "sdpa_common.hpp"
#include "sdpa_lds.hpp"

namespace theria {

// The K, V, gK, gV tiles pass through registers into padded LDS rows (two barriers per tile).
// EXACT: the second pass of 16-bit problems, which redoes only the workgroups holding a row flagged peaked in
// lse in the exact form (overwriting G_Q; r and t are the first launch's); apart, the first launch keeps its
// registers and schedule.
template <typename T, int DP, bool CAUSAL, bool EXACT>
__device__ __attribute__((always_inline)) inline void rows_block(const BwdBwdParams& p, const int blk, const int nblk) {
  using OP = Ops<T, DP>;
  using F = typename OP::F;
  constexpr int KC = OP::KC;
  constexpr int NW = 4, BM = 32 * NW, NT = 64 * NW;
  // keys per tile: two 32-key subtiles per tile where the registers allow (one wave per SIMD)
  constexpr int BN = (DP == 128 || sizeof(T) == 4) ? 32 : 64;
  constexpr int PITCH = OP::PITCH;
  constexpr int NDT = DP / 32, NKC = DP / KC, NPC = 32 / KC, NST = BN / 32;
  __shared__ __attribute__((aligned(16))) T sK0[BN * PITCH], sV0[BN * PITCH], sgK0[BN * PITCH], sgV0[BN * PITCH];

  const Shape& s = p.s;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 31, g = lane >> 5;
  const int nqb = (s.T + BM - 1) / BM;
  const int bid = xcd_remap(blk, nblk);
  const int bh = bid / nqb;
  int qb = bid - bh * nqb;
  if (CAUSAL && !EXACT) qb = nqb - 1 - qb;  // longest first (the exact pass: query order, see the cols grid)
  const int b = bh / s.H, h = bh - b * s.H;
  const T* Q = (const T*)p.q.p + b * p.q.sb + h * p.q.sh;
  const T* K = (const T*)p.k.p + b * p.k.sb + h * p.k.sh;
  const T* V = (const T*)p.v.p + b * p.v.sb + h * p.v.sh;
  const T* dO = (const T*)p.dout.p + b * p.dout.sb + h * p.dout.sh;
  const bool has_gq = p.gq.p != nullptr, has_gk = p.gk.p != nullptr, has_gv = p.gv.p != nullptr;
  const T* GQ = has_gq ? (const T*)p.gq.p + b * p.gq.sb + h * p.gq.sh : nullptr;
  const T* GK = has_gk ? (const T*)p.gk.p + b * p.gk.sb + h * p.gk.sh : nullptr;
  const T* GV = has_gv ? (const T*)p.gv.p + b * p.gv.sb + h * p.gv.sh : nullptr;
  const int q0w = qb * BM + wave * 32;
  const int myq = q0w + li;
  const bool qvalid = myq < s.T;
  const int64_t row_id = (int64_t)bh * s.T + myq;
  int kend = s.M;
  if (CAUSAL) kend = min(s.M, qb * BM + BM);
  const int nkt = (kend + BN - 1) / BN;
  // tiles that need no mask (their own copy of the loops)
  const int nfull = min(nkt, CAUSAL ? min(s.M / BN, qb * BM / BN) : s.M / BN);
  // 16-bit workgroups holding a row flagged peaked in lse take the exact form (uniform). Causal ones with at
  // most half the longest workgroup's key tiles run both of its passes in the first launch, inside that
  // launch's slack (every head's first query block holds such rows); the others are the second pass's.
  static_assert(!EXACT || sizeof(T) == 2, "the exact form is for 16-bit inputs");
  constexpr bool LIGHT_OK = CAUSAL && sizeof(T) == 2 && DP <= 64;  // at 128 the second sweep spills
  const bool light = LIGHT_OK && 2 * nkt <= (s.M + BN - 1) / BN;
  bool flagged = false;
  if (EXACT || (LIGHT_OK && light)) flagged = __syncthreads_or(qvalid && lse_peaked(p.lse[row_id]));
  const bool exact = EXACT && flagged && !light;
  // float32 at head dim 128 always takes the two passes: the one-pass form's four 128-wide accumulators and three operand
  // sets spilled ~700 registers, the exact form's passes hold two. The split products spill more than v_mfma_f32_32x32x2_f32
  // did (rows ~105 -> ~220 of 512 registers, columns ~200 -> ~330) and are faster all the same. HVP of <W, O>, us, the
  // one-pass form with v_mfma_f32_32x32x2_f32 -> two passes with it -> two passes with split products: B4 H8 T700 D128
  // 3724 -> 2593 -> 1666, B2 H16 T1000 D80 5333 -> 4027 -> 2447, causal 4586 -> 3099 -> 2193, B16 H16 T300 D128 causal
  // 4572 -> 3301 -> 2132.
  constexpr bool TWO = sizeof(T) == 4 && DP == 128;
  const bool two_pass = TWO || (!EXACT && LIGHT_OK && flagged && light);
  if (EXACT && !exact) return;

  F qf[NKC], dof[NKC], gqf[NKC];
  {
    typename OP::Raw r0[NKC], r1[NKC], r2[NKC];
#pragma unroll
    for (int c = 0; c < NKC; ++c) {
      r0[c] = OP::raw(Q, p.q.sr, myq, s.T, c, s.D, s.vec);
      r1[c] = OP::raw(dO, p.dout.sr, myq, s.T, c, s.D, s.vec);
      r2[c] = has_gq ? OP::raw(GQ, p.gq.sr, myq, s.T, c, s.D, s.vec) : typename OP::Raw{};
    }
#pragma unroll
    for (int c = 0; c < NKC; ++c) {
      qf[c] = OP::frag(r0[c]);
      dof[c] = OP::frag(r1[c]);
      gqf[c] = OP::frag(r2[c]);
    }
  }
  f32x16_t x13[NDT], x2[NDT], x4[NDT], yk[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) {
    x13[dt] = zero16();
    x2[dt] = zero16();
    x4[dt] = zero16();
    yk[dt] = zero16();
  }
  const float c2 = s.scale * kLog2e;
  const float lse2 = qvalid ? p.lse[row_id] * kLog2e : THERIA_INF;
  const float moff = lse2 == -THERIA_INF ? THERIA_INF : lse2;
  // float32: P = exp2((fl(S c2) - m2) - L2) from the row's own statistics, and dP formed from zero, both as in
  // the row-term pass that wrote m2, L2 and z (so the largest score gives exactly 2^-L2, and dP - z keeps only
  // z's own rounding)
  constexpr bool OWN = sizeof(T) == 4;
  const float m2 = OWN && qvalid ? p.lse[row_id] : THERIA_INF;
  const float l2 = OWN && qvalid ? p.row_l2[row_id] : 0.f;
  const float z = qvalid ? p.delta[row_id] : 0.f;
  float r_part = 0.f, t_part = 0.f;
  // 16-bit inputs: Gbar_S = P o ((Gam - r)(dP - z) + W - t), and for any row constants cr, ct
  //   Gbar_S = P o E1c - (r - cr) dS - (t - ct) P  with  E1c = (Gam - cr)(dP - z) + W - ct,
  // so x13 takes P o E1c and G_Q = s (x13 - (r - cr) x2 - t_c x4 + yk), t_c = sum_j of the rounded P o E1c
  // operands (= t - ct in exact arithmetic). The centres are r and t over the first key tile (a pre-pass),
  // used when that tile holds more than half of the row's probability (else cr = ct = 0):
  // on rows with few visible keys, where G_Q is a small difference of large terms, the products then carry
  // small centred values instead (one visible key gives G_Q = 0 exactly).
  float t_frag = 0.f, cr = 0.f, ct = 0.f;
  float rx = 0.f, tx = 0.f;  // exact row terms of the exact form
  float c_p = 0.f, c_pg = 0.f, c_pgd = 0.f, c_pd = 0.f, c_pw = 0.f;

  // The key tile kt held in (tK, tV, tgK, tgV), as 32-key subtiles.
  // PASS: 0 the pre-pass (sums only: for the centres over the first tile, or for r and t over every tile),
  // 1 the common pass, 3 the exact pass (Gbar_S from exact row terms r, t: 16-bit, and float32 at DP = 128).
  auto compute = [&](auto pass_tag, auto mask_tag, int kt, const T* tK, const T* tV, const T* tgK,
                     const T* tgV) __attribute__((always_inline)) {
    constexpr int PASS = decltype(pass_tag)::value;
    constexpr bool MASK = decltype(mask_tag)::value;  // the tile reaches past the last key or past the block's first query
    constexpr bool PRE = PASS == 0;
    const int k0 = kt * BN;
#pragma unroll
    for (int st = 0; st < NST; ++st) {
      const int k0s = k0 + 32 * st;  // this 32-key subtile
      if (CAUSAL && k0s > q0w + 31) continue;

      f32x16_t sc = zero16(), gm = zero16(), w = zero16(), dpz;
#pragma unroll
      for (int r = 0; r < 16; ++r) dpz[r] = OWN ? 0.f : -z;
#pragma unroll
      for (int c = 0; c < NKC; ++c) {
        const F kfr = OP::cols(tK, 32 * st + li, c);
        sc = OP::mma(kfr, qf[c], sc);
        dpz = OP::mma(OP::cols(tV, 32 * st + li, c), dof[c], dpz);
        if (has_gq) gm = OP::mma(kfr, gqf[c], gm);
        if (has_gk) gm = OP::mma(OP::cols(tgK, 32 * st + li, c), qf[c], gm);
        if (has_gv) w = OP::mma(OP::cols(tgV, 32 * st + li, c), dof[c], w);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        if constexpr (OWN) dpz[r] -= z;
        float pv = OWN ? own_prob(sc[r], c2, m2, l2) : fast_exp2(fmaf(sc[r], c2, -moff));
        if constexpr (MASK) {
          const int key = k0s + acc_row(r, g);
          if (key >= s.M || (CAUSAL && key > myq)) pv = 0.f;
        }
        const float gam = s.scale * gm[r];
        const float e1 = fmaf(gam, dpz[r], w[r]);
        const float pe1 = pv * e1;
        if constexpr (PRE) {
          c_p += pv;
          c_pg = fmaf(pv, gam, c_pg);
          c_pd = fmaf(pv, dpz[r], c_pd);
          c_pgd = fmaf(pv * gam, dpz[r], c_pgd);
          c_pw = fmaf(pv, w[r], c_pw);
        } else if constexpr (PASS == 3) {
          gm[r] = pv * (fmaf(gam - rx, dpz[r], w[r]) - tx);  // Gbar_S
          dpz[r] = pv * dpz[r];                              // dS
        } else {
          r_part = fmaf(pv, gam, r_part);
          t_part += pe1;
          sc[r] = pv;
          gm[r] = sizeof(T) == 2 ? pv * (fmaf(gam - cr, dpz[r], w[r]) - ct) : pe1;
          dpz[r] = pv * dpz[r];  // dS
        }
      }
      if constexpr (PRE) continue;
      if constexpr (PASS == 3 && sizeof(T) == 4) {
#pragma unroll
        for (int cc = 0; cc < NPC; ++cc) {
          const F gf = OP::acc(gm, cc), df = OP::acc(dpz, cc);
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) {
            x13[dt] = OP::mma(OP::rows(tK, 32 * st, cc, dt * 32), gf, x13[dt]);
            if (has_gk) yk[dt] = OP::mma(OP::rows(tgK, 32 * st, cc, dt * 32), df, yk[dt]);
          }
        }
        continue;
      }
      if constexpr (PASS == 3 && sizeof(T) == 2) {
#pragma unroll
        for (int cc = 0; cc < NPC; ++cc) {
          F gh, gl, dh, dl;
          split_frag<T>(gm, cc, gh, gl);
          split_frag<T>(dpz, cc, dh, dl);
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) {
            const F kr = OP::rows(tK, 32 * st, cc, dt * 32);
            x13[dt] = OP::mma(kr, gh, x13[dt]);
            x13[dt] = OP::mma(kr, gl, x13[dt]);
            if (has_gk) {
              const F gkr = OP::rows(tgK, 32 * st, cc, dt * 32);
              yk[dt] = OP::mma(gkr, dh, yk[dt]);
              yk[dt] = OP::mma(gkr, dl, yk[dt]);
            }
          }
        }
        continue;
      }
#pragma unroll
      for (int cc = 0; cc < NPC; ++cc) {
        const F pf = OP::acc(sc, cc);
        const F pe1f = OP::acc(gm, cc);
        const F dsf = OP::acc(dpz, cc);
        if constexpr (sizeof(T) == 2) t_frag = frag_sum<T>(pe1f, t_frag);
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
          const F kr = OP::rows(tK, 32 * st, cc, dt * 32);
          x13[dt] = OP::mma(kr, pe1f, x13[dt]);
          x2[dt] = OP::mma(kr, dsf, x2[dt]);
          x4[dt] = OP::mma(kr, pf, x4[dt]);
          if (has_gk) yk[dt] = OP::mma(OP::rows(tgK, 32 * st, cc, dt * 32), dsf, yk[dt]);
        }
      }
    }
  };

  const std::integral_constant<int, 0> pre_pass;
  const std::integral_constant<int, 1> full_pass;
  const std::integral_constant<int, 3> exact_pass;
  if (exact) {  // the first launch's exact float32 row terms (same stream, so already written)
    rx = qvalid ? p.r_row[row_id] : 0.f;
    tx = qvalid ? p.t_row[row_id] : 0.f;
  }
  // r = sum_j P Gam, t = sum_j P (Gam (dP - z) + W) from the pre-pass sums over all keys
  auto set_exact_terms = [&]() {
    rx = pair_sum(c_pg);
    tx = pair_sum(c_pgd) + pair_sum(c_pw);
  };
  auto set_centre = [&]() {
    const float sp = pair_sum(c_p), spg = pair_sum(c_pg), spd = pair_sum(c_pd), spgd = pair_sum(c_pgd),
                spw = pair_sum(c_pw);
    // only where the first tile holds most of the row's probability (its means then stand for the row)
    if (sp > 0.5f) {
      cr = spg / sp;
      ct = (spgd - cr * spd + spw) / sp;
    }
  };

  {
    TileStage<T, BN, DP, NT> gsK, gsV, gsgK, gsgV;
    auto prefetch = [&](int k0) {
      gsK.load(K, p.k.sr, k0, s.M, s.D, s.vec);
      gsV.load(V, p.v.sr, k0, s.M, s.D, s.vec);
      if (has_gk) gsgK.load(GK, p.gk.sr, k0, s.M, s.D, s.vec);
      if (has_gv) gsgV.load(GV, p.gv.sr, k0, s.M, s.D, s.vec);
    };
    // every key tile once, from tile 0 already prefetched
    auto sweep = [&](auto pass_tag) __attribute__((always_inline)) {
      auto step = [&](auto mask_tag, int kt) __attribute__((always_inline)) {
        __syncthreads();
        OP::store(gsK, sK0, true, gsV, sV0, true, gsgK, sgK0, has_gk, gsgV, sgV0, has_gv);
        __syncthreads();
        if (kt + 1 < nkt) prefetch((kt + 1) * BN);
        compute(pass_tag, mask_tag, kt, sK0, sV0, sgK0, sgV0);
      };
      int kt = 0;
      for (; kt < nfull; ++kt) step(std::false_type{}, kt);
      for (; kt < nkt; ++kt) step(std::true_type{}, kt);
    };
    if (nkt > 0) prefetch(0);
    if (exact) {
      if (nkt > 0) sweep(exact_pass);
    } else if (two_pass) {
      if (nkt > 0) {
        sweep(pre_pass);  // r and t of every row from all its keys
        set_exact_terms();
        prefetch(0);
        sweep(exact_pass);
      }
    } else {
      if (sizeof(T) == 2 && nkt > 0) {
        // centre pre-pass over tile 0 (the loop stages the same registers again)
        OP::store(gsK, sK0, true, gsV, sV0, true, gsgK, sgK0, has_gk, gsgV, sgV0, has_gv);
        __syncthreads();
        compute(pre_pass, std::true_type{}, 0, sK0, sV0, sgK0, sgV0);
        set_centre();
      }
      if constexpr (!TWO) sweep(full_pass);
    }
  }

  const float rr = two_pass ? rx : pair_sum(r_part), tt = two_pass ? tx : pair_sum(t_part);
  const float tg = sizeof(T) == 2 ? pair_sum(t_frag) : tt;  // t_c as G_Q uses it; the cols kernel takes tt
  const float rg = rr - cr;                                   // r - cr (cr = 0 for float32)
  if (qvalid) {
    T* OG = (T*)p.out_gq.p + b * p.out_gq.sb + h * p.out_gq.sh;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const int d0 = dt * 32 + 8 * qd + 4 * g;
        if (d0 < s.D) {
          float r4[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int i = 4 * qd + e;
            r4[e] = s.scale * (x13[dt][i] - rg * x2[dt][i] - tg * x4[dt][i] + yk[dt][i]);
          }
          store4<T>(OG, p.out_gq.sr, myq, d0, s.D, r4[0], r4[1], r4[2], r4[3], s.vec);
        }
      }
    if (g == 0 && !EXACT) {
      p.r_row[row_id] = rr;
      p.t_row[row_id] = tt;
    }
  }
}

template <typename T, int DP, bool CAUSAL, bool EXACT>
__global__ __launch_bounds__(256) void bwdbwd_rows_kernel(const BwdBwdParams p) {
  rows_block<T, DP, CAUSAL, EXACT>(p, blockIdx.x, gridDim.x);
}

// Q, dO, gQ tiles staged as in the rows kernel, the row terms beside them.
template <typename T, int DP, bool CAUSAL>
__device__ __attribute__((always_inline)) inline void cols_block(const BwdBwdParams& p, const int blk, const int nblk) {
  using OP = Ops<T, DP>;
  using F = typename OP::F;
  constexpr int KC = OP::KC;
  constexpr int NW = 4, BN = 32 * NW, NT = 64 * NW;
  // queries per tile: two 32-query subtiles per tile where the registers allow
  constexpr int BM = (DP == 128 || sizeof(T) == 4) ? 32 : 64;
  constexpr int PITCH = OP::PITCH;
  constexpr int NDT = DP / 32, NKC = DP / KC, NPC = 32 / KC, NSQ = BM / 32;
  // float32 (OWN): P = exp2((fl(S c2) - m2) - L2) with the rows' own m2 (in lse) and L2 (row_l2), and dP formed
  // from zero, as in the row-term pass that wrote them
  constexpr bool OWN = sizeof(T) == 4;
  constexpr int FLAG = OWN ? 5 * BM : 4 * BM;  // row terms, then whether the tile holds a row flagged peaked
  constexpr int RB = FLAG + 4;
  __shared__ __attribute__((aligned(16))) T sQ0[BM * PITCH], sdO0[BM * PITCH], sgQ0[BM * PITCH];
  // row terms [lse * log2(e) (float32: m2) | delta | r | t | (float32: L2) | peaked] of a tile
  __shared__ __attribute__((aligned(16))) float sRow0[RB];

  const Shape& s = p.s;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6, li = lane & 31, g = lane >> 5;
  const int nkb = (s.M + BN - 1) / BN;
  const int bid = xcd_remap(blk, nblk);
  const int bh = bid / nkb;
  const int kb = bid - bh * nkb;
  const int b = bh / s.H, h = bh - b * s.H;
  const T* Q = (const T*)p.q.p + b * p.q.sb + h * p.q.sh;
  const T* K = (const T*)p.k.p + b * p.k.sb + h * p.k.sh;
  const T* V = (const T*)p.v.p + b * p.v.sb + h * p.v.sh;
  const T* dO = (const T*)p.dout.p + b * p.dout.sb + h * p.dout.sh;
  const bool has_gq = p.gq.p != nullptr, has_gk = p.gk.p != nullptr, has_gv = p.gv.p != nullptr;
  const T* GQ = has_gq ? (const T*)p.gq.p + b * p.gq.sb + h * p.gq.sh : nullptr;
  const T* GK = has_gk ? (const T*)p.gk.p + b * p.gk.sb + h * p.gk.sh : nullptr;
  const T* GV = has_gv ? (const T*)p.gv.p + b * p.gv.sb + h * p.gv.sh : nullptr;
  const int key0 = kb * BN;
  const int kw0 = key0 + wave * 32;
  const int mykey = kw0 + li;

  F kf[NKC], vf[NKC], gkf[NKC], gvf[NKC];
  {
    typename OP::Raw r0[NKC], r1[NKC], r2[NKC], r3[NKC];
#pragma unroll
    for (int c = 0; c < NKC; ++c) {
      r0[c] = OP::raw(K, p.k.sr, mykey, s.M, c, s.D, s.vec);
      r1[c] = OP::raw(V, p.v.sr, mykey, s.M, c, s.D, s.vec);
      r2[c] = has_gk ? OP::raw(GK, p.gk.sr, mykey, s.M, c, s.D, s.vec) : typename OP::Raw{};
      r3[c] = has_gv ? OP::raw(GV, p.gv.sr, mykey, s.M, c, s.D, s.vec) : typename OP::Raw{};
    }
#pragma unroll
    for (int c = 0; c < NKC; ++c) {
      kf[c] = OP::frag(r0[c]);
      vf[c] = OP::frag(r1[c]);
      gkf[c] = OP::frag(r2[c]);
      gvf[c] = OP::frag(r3[c]);
    }
  }
  f32x16_t accV[NDT], accK[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) {
    accV[dt] = zero16();
    accK[dt] = zero16();
  }
  const float c2 = s.scale * kLog2e;
  const int qbeg = CAUSAL ? (key0 / BM) * BM : 0;
  const int nqt = s.T > qbeg ? (s.T - qbeg + BM - 1) / BM : 0;
  const int64_t rowbase = (int64_t)bh * s.T;

  // Row terms of a tile for thread tid < BM, held raw (rows past the end: lse = +inf) and converted when
  // stored: lse * log2(e) (+inf for rows past the end or without visible keys, so P = 0), delta, r, t.
  float r_lse = THERIA_INF, r_z = 0.f, r_r = 0.f, r_t = 0.f, r_l2 = 0.f;
  auto load_rows = [&](int it) {
    if (tid < BM && it < nqt) {
      const int qq = qbeg + it * BM + tid;
      const bool ok = qq < s.T;
      r_lse = ok ? p.lse[rowbase + qq] : THERIA_INF;
      r_z = ok ? p.delta[rowbase + qq] : 0.f;
      r_r = ok ? p.r_row[rowbase + qq] : 0.f;
      r_t = ok ? p.t_row[rowbase + qq] : 0.f;
      if constexpr (OWN) r_l2 = ok ? p.row_l2[rowbase + qq] : 0.f;
    }
  };
  auto store_rows = [&](float* sr) {
    if (tid < BM) {
      // float32: m2 as it is (+inf for a row without visible keys or past the end, so P = 0)
      sr[tid] = OWN ? r_lse : (__builtin_isinf(r_lse) ? THERIA_INF : r_lse * kLog2e);
      sr[BM + tid] = r_z;
      sr[2 * BM + tid] = r_r;
      sr[3 * BM + tid] = r_t;
      if constexpr (OWN) sr[4 * BM + tid] = r_l2;
      const bool pk = !OWN && __any(lse_peaked(r_lse));  // the tile's rows are the lanes of wave 0
      if (tid == 0) sr[FLAG] = pk ? 1.f : 0.f;
    }
  };

  // The query tile it held in (tQ, tO, tgQ) with its row terms in sr, as 32-query subtiles. SPLIT: Gbar_dP,
  // Gbar_S and dS enter the products as two 16-bit terms each.
  auto tile = [&](auto split_tag, auto diag_tag, int it, const T* tQ, const T* tO, const T* tgQ,
                  const float* sr) __attribute__((always_inline)) {
    constexpr bool SPLIT = decltype(split_tag)::value;
    constexpr bool DIAG = decltype(diag_tag)::value;  // causal: the tile starts before the block's last key
    const int q0 = qbeg + it * BM;
    if (CAUSAL && kw0 > q0 + BM - 1) return;
#pragma unroll
    for (int sq = 0; sq < NSQ; ++sq) {
      const int q0s = q0 + 32 * sq;  // this 32-query subtile
      if (CAUSAL && kw0 > q0s + 31) continue;

      f32x16_t sc = zero16(), gm = zero16(), w = zero16(), dpz;
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const f32x4_t z4 = *reinterpret_cast<const f32x4_t*>(sr + BM + 32 * sq + 8 * qd + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) dpz[4 * qd + e] = OWN ? 0.f : -z4[e];
      }
#pragma unroll
      for (int c = 0; c < NKC; ++c) {
        const F qfr = OP::cols(tQ, 32 * sq + li, c);
        const F ofr = OP::cols(tO, 32 * sq + li, c);
        sc = OP::template mma<true>(qfr, kf[c], sc);
        dpz = OP::template mma<true>(ofr, vf[c], dpz);
        if (has_gq) gm = OP::template mma<true>(OP::cols(tgQ, 32 * sq + li, c), kf[c], gm);
        if (has_gk) gm = OP::template mma<true>(qfr, gkf[c], gm);
        if (has_gv) w = OP::template mma<true>(ofr, gvf[c], w);
      }
      // the row terms are read here, four rows at a time, and the results take their operands' registers: gm <- Gbar_dP,
      // w <- Gbar_S, dpz <- dS
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const int o = 32 * sq + 8 * qd + 4 * g;
        const f32x4_t l4 = *reinterpret_cast<const f32x4_t*>(sr + o);
        const f32x4_t r4 = *reinterpret_cast<const f32x4_t*>(sr + 2 * BM + o);
        const f32x4_t t4 = *reinterpret_cast<const f32x4_t*>(sr + 3 * BM + o);
        f32x4_t z4{}, lo4{};
        if constexpr (OWN) {
          z4 = *reinterpret_cast<const f32x4_t*>(sr + BM + o);
          lo4 = *reinterpret_cast<const f32x4_t*>(sr + 4 * BM + o);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = 4 * qd + e;
          if constexpr (OWN) dpz[r] -= z4[e];
          float pv = OWN ? own_prob(sc[r], c2, l4[e], lo4[e]) : fast_exp2(fmaf(sc[r], c2, -l4[e]));
          if constexpr (DIAG)  // (a key past the end needs no mask: its lane's results are not stored)
            if (mykey > q0s + acc_row(r, g)) pv = 0.f;
          const float gam = s.scale * gm[r];
          const float ds = pv * dpz[r];
          const float e1 = fmaf(gam, dpz[r], w[r]);
          gm[r] = pv * (gam - r4[e]);
          w[r] = pv * e1 - r4[e] * ds - t4[e] * pv;
          dpz[r] = ds;
        }
      }
      if constexpr (SPLIT && sizeof(T) == 2) {
#pragma unroll
        for (int cc = 0; cc < NPC; ++cc) {
          F gdph, gdpl, gsh, gsl, dsh, dsl;
          split_frag<T>(gm, cc, gdph, gdpl);
          split_frag<T>(w, cc, gsh, gsl);
          split_frag<T>(dpz, cc, dsh, dsl);
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) {
            const F ro = OP::rows(tO, 32 * sq, cc, dt * 32);
            accV[dt] = OP::mma(gdph, ro, accV[dt]);
            accV[dt] = OP::mma(gdpl, ro, accV[dt]);
            const F rq = OP::rows(tQ, 32 * sq, cc, dt * 32);
            accK[dt] = OP::mma(gsh, rq, accK[dt]);
            accK[dt] = OP::mma(gsl, rq, accK[dt]);
            if (has_gq) {
              const F rg = OP::rows(tgQ, 32 * sq, cc, dt * 32);
              accK[dt] = OP::mma(dsh, rg, accK[dt]);
              accK[dt] = OP::mma(dsl, rg, accK[dt]);
            }
          }
        }
      } else {
#pragma unroll
        for (int cc = 0; cc < NPC; ++cc) {
          const F gdpf = OP::acc(gm, cc);
          const F gsf = OP::acc(w, cc);
          const F dsf = OP::acc(dpz, cc);
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) {
            accV[dt] = OP::mma(gdpf, OP::rows(tO, 32 * sq, cc, dt * 32), accV[dt]);
            accK[dt] = OP::mma(gsf, OP::rows(tQ, 32 * sq, cc, dt * 32), accK[dt]);
            if (has_gq) accK[dt] = OP::mma(dsf, OP::rows(tgQ, 32 * sq, cc, dt * 32), accK[dt]);
          }
        }
      }
    }
  };
  const std::integral_constant<bool, true> with_split;
  const std::integral_constant<bool, false> no_split;
  bool pk_any = false;  // uniform: a tile holding a peaked row was skipped (16-bit)
  auto compute = [&](auto diag_tag, int it, const T* tQ, const T* tO, const T* tgQ,
                     const float* sr) __attribute__((always_inline)) {
    // uniform: every thread reads the same flag
    const bool pk = sizeof(T) == 2 && __builtin_amdgcn_readfirstlane(__float_as_uint(sr[FLAG])) != 0u;
    pk_any |= pk;  // run after the loop, so the loop's schedule holds only the one-term products
    if (!pk) tile(no_split, diag_tag, it, tQ, tO, tgQ, sr);
  };
  // The tiles holding a peaked row, found 64 at a time from the lse flags and run one after the other with
  // the split products, from stage(it) (loads tile it into sQ0, sdO0, sgQ0 and its row terms into sRow0).
  auto peaked_tiles = [&](auto stage) __attribute__((always_inline)) {
    __shared__ int sPk[64];
    for (int t0 = 0; t0 < nqt; t0 += 64) {
      const int nt = min(64, nqt - t0);
      __syncthreads();  // every thread is done with the previous flags and tile buffers
      if (tid < 64) sPk[tid] = 0;
      __syncthreads();
      constexpr int RPT = (64 * BM + NT - 1) / NT;
      const int r0 = qbeg + t0 * BM, r1 = min(s.T, qbeg + (t0 + nt) * BM);
      float lv[RPT];
#pragma unroll
      for (int j = 0; j < RPT; ++j) {
        const int r = r0 + tid + NT * j;
        lv[j] = r < r1 ? p.lse[rowbase + r] : THERIA_INF;  // rows past the end: no flag
      }
#pragma unroll
      for (int j = 0; j < RPT; ++j)
        if (lse_peaked(lv[j])) sPk[(tid + NT * j) / BM] = 1;
      __syncthreads();
      for (int i = 0; i < nt; ++i) {
        if (!sPk[i]) continue;  // uniform: every thread reads the same flag
        stage(t0 + i);
        __syncthreads();
        tile(with_split, std::integral_constant<bool, CAUSAL>{}, t0 + i, sQ0, sdO0, sgQ0, sRow0);
        __syncthreads();  // the tile buffers are free again
      }
    }
  };

  {
    TileStage<T, BM, DP, NT> gsQ, gsO, gsgQ;
    auto prefetch = [&](int it) {
      const int q0 = qbeg + it * BM;
      gsQ.load(Q, p.q.sr, q0, s.T, s.D, s.vec);
      gsO.load(dO, p.dout.sr, q0, s.T, s.D, s.vec);
      if (has_gq) gsgQ.load(GQ, p.gq.sr, q0, s.T, s.D, s.vec);
      load_rows(it);
    };
    if (nqt > 0) prefetch(0);
    auto step = [&](auto diag_tag, int it) __attribute__((always_inline)) {
      __syncthreads();
      OP::store(gsQ, sQ0, true, gsO, sdO0, true, gsgQ, sgQ0, has_gq);
      store_rows(sRow0);
      __syncthreads();
      if (it + 1 < nqt) prefetch(it + 1);
      compute(diag_tag, it, sQ0, sdO0, sgQ0, sRow0);
    };
    const int ndiag = CAUSAL ? min(nqt, (key0 + BN - 1 - qbeg + BM - 1) / BM) : 0;
    int it = 0;
    for (; it < ndiag; ++it) step(std::integral_constant<bool, CAUSAL>{}, it);
    for (; it < nqt; ++it) step(std::false_type{}, it);
    if (pk_any)
      peaked_tiles([&](int it) __attribute__((always_inline)) {
        prefetch(it);
        OP::store(gsQ, sQ0, true, gsO, sdO0, true, gsgQ, sgQ0, has_gq);
        store_rows(sRow0);
      });
  }

  T* OV = (T*)p.out_gv.p + b * p.out_gv.sb + h * p.out_gv.sh;
  T* OK = (T*)p.out_gk.p + b * p.out_gk.sb + h * p.out_gk.sh;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) {
    const int d = dt * 32 + li;
    if (d < s.D) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = kw0 + acc_row(r, g);
        if (key < s.M) {
          OV[(int64_t)key * p.out_gv.sr + d] = (T)accV[dt][r];
          OK[(int64_t)key * p.out_gk.sr + d] = (T)(accK[dt][r] * s.scale);
        }
      }
    }
  }
}

template <typename T, int DP, bool CAUSAL>
__global__ __launch_bounds__(256) void bwdbwd_cols_kernel(const BwdBwdParams p) {
  cols_block<T, DP, CAUSAL>(p, blockIdx.x, gridDim.x);
}

// 16-bit: the rows kernel's second (exact) launch and the column blocks as one grid. The exact row blocks
// read only what the first rows launch wrote (r, t) and write only G_Q, so they are independent of the
// column blocks; in one grid they run beside them, instead of as a launch of their own whose few busy
// workgroups would leave the GPU idle.
template <typename T, int DP, bool CAUSAL>
__global__ __launch_bounds__(256) void bwdbwd_cols_exact_kernel(const BwdBwdParams p) {
  const int ncols = ((p.s.M + 127) / 128) * p.s.B * p.s.H;
  const int nrows = (int)gridDim.x - ncols;
  const int bid = blockIdx.x;  // uniform
  // Row blocks first: most exit at once (no flagged row), and the few heavy ones (a single peaked row makes
  // its block sweep every key) start at once. A workgroup waits for the CU of its own place in the grid,
  // so the column block placed like a heavy row block starts when that one ends; for causal problems the
  // row blocks run in query order (no heavy-first reversal), which pairs query block i with key block i,
  // whose lengths (i + 1 and n - i key tiles) add up to about the longest column block's.
  if (bid < nrows)
    rows_block<T, DP, CAUSAL, true>(p, bid, nrows);
  else
    cols_block<T, DP, CAUSAL>(p, bid - nrows, ncols);
}

// The split kernels (sdpa_bwdbwd_split.hip): whether they cover the problem, and their launches.
template <typename T>
bool rows_ks_ok(const BwdBwdParams& p);
template <typename T>
bool cols_qs_ok(const BwdBwdParams& p);
template <typename T, bool CAUSAL>
hipError_t launch_rows_ks(const BwdBwdParams& p, hipStream_t st);
template <typename T, bool CAUSAL>
hipError_t launch_cols_qs(const BwdBwdParams& p, hipStream_t st);

// 16-bit: the rows kernel's exact launch rides in the column grid when both are the general kernels.
template <typename T>
static bool exact_in_cols(const BwdBwdParams& p) {
  return sizeof(T) == 2 && !rows_ks_ok<T>(p) && !cols_qs_ok<T>(p);
}

struct RowsLauncher {
  template <typename T, int DP, bool CAUSAL>
  static hipError_t run(const BwdBwdParams& p, hipStream_t st) {
    const int nqb = (p.s.T + 127) / 128;
    const int64_t nblk = (int64_t)nqb * p.s.B * p.s.H;
    if (nblk == 0) return hipSuccess;
    if constexpr (sizeof(T) == 2) {
      // every row block exact in one launch (the column grid has no row blocks)
      if (rows_ks_ok<T>(p)) return launch_rows_ks<T, CAUSAL>(p, st);
    }
    hipLaunchKernelGGL((bwdbwd_rows_kernel<T, DP, CAUSAL, false>), dim3((unsigned)nblk), dim3(256), 0, st, p);
    if constexpr (sizeof(T) == 2)
      if (!exact_in_cols<T>(p))
        hipLaunchKernelGGL((bwdbwd_rows_kernel<T, DP, CAUSAL, true>), dim3((unsigned)nblk), dim3(256), 0, st, p);
    return hipGetLastError();
  }
};

// Runs after RowsLauncher on the same stream (the exact row blocks read the first rows launch's r and t).
struct ColsLauncher {
  template <typename T, int DP, bool CAUSAL>
  static hipError_t run(const BwdBwdParams& p, hipStream_t st) {
    const int64_t nblk = (int64_t)((p.s.M + 127) / 128) * p.s.B * p.s.H;
    const int64_t nrow = (int64_t)((p.s.T + 127) / 128) * p.s.B * p.s.H;
    if constexpr (sizeof(T) == 2) {
      if (cols_qs_ok<T>(p)) return launch_cols_qs<T, CAUSAL>(p, st);
      if (exact_in_cols<T>(p)) {
        if (nblk + nrow == 0) return hipSuccess;
        hipLaunchKernelGGL((bwdbwd_cols_exact_kernel<T, DP, CAUSAL>), dim3((unsigned)(nblk + nrow)), dim3(256), 0, st, p);
        return hipGetLastError();
      }
    }
    if (nblk == 0) return hipSuccess;
    hipLaunchKernelGGL((bwdbwd_cols_kernel<T, DP, CAUSAL>), dim3((unsigned)nblk), dim3(256), 0, st, p);
    return hipGetLastError();
  }
};

hipError_t launch_bwdbwd_rows(const BwdBwdParams& p, hipStream_t st) { return dispatch_all<RowsLauncher>(p, st); }

bool bwdbwd_rows_make_row_terms(const BwdBwdParams& p) {
  if (p.s.dtype == 1) return rows_ks_ok<_Float16>(p);
  if (p.s.dtype == 2) return rows_ks_ok<__bf16>(p);
  return false;
}
hipError_t launch_bwdbwd_cols(const BwdBwdParams& p, hipStream_t st) { return dispatch_all<ColsLauncher>(p, st); }

}  // namespace theria
