// Backward and double backward of small problems for gfx950: at most 64 queries and 64 keys per (batch, head), one
// two-wave workgroup for the whole problem and one launch for every output.
//
// Same contracts as the general kernels (sdpa_bwd.hip, sdpa_bwdbwd.hip; the formulas are there). At these sizes
// those run two (backward) to four (double backward) launches of 128-row blocks, half or more of whose waves have
// no rows, each launch reading every operand again and rebuilding the scores; few-hundred-token MAML batches
// (B400 H4 T64 D16 float32) then spend their time in launches and in one or two waves per SIMD.
//
// Two phases per workgroup, wave w owning queries 32w .. 32w + 31 and then keys 32w .. 32w + 31:
//  * rows: the key-side tensors in LDS, lane per query (S^T = K Q^T). Every score of the row is in registers (two
//    32-key subtiles), so the row statistics come first and each product is formed once, in its exact form:
//    G_Q = s (Gbar_S K + dS gK), G_dO = Gbar_dP V + P gV with Gbar_dP = P o (Gam - r),
//    Gbar_S = P o ((Gam - r)(dP - z) + W - t); the row terms go to LDS;
//  * columns: the query-side tensors in the same LDS, lane per key, scores formed again the other way round (their
//    products at these sizes cost less than transposing three matrices through LDS).
// float32 takes the three-term split products (MfmaX3); 16-bit inputs enter the accumulated products as two 16-bit
// terms (hi + lo), as the general kernels do on peaked rows. P = exp2(fl(S c) - max) / sum from the row's own scores
// in the double backward (the given lse is not needed there), exp(S - lse) in the backward.
// GPU time, general kernels (their float32 products still on v_mfma_f32_32x32x2_f32) -> here (us; backward / double
// backward): float32 B400 H4 T64 D16 94 / 279 -> 29 / 54, float32 B64 H8 T64 D64 65 / 188 -> 30 / 80, float32 B2 H2 T16 D8
// 13.5 / 31.0 -> 8.5 / 11.7, bfloat16 B64 H8 T64 D64 32 / 49 -> 21 / 27, bfloat16 B512 H8 T64 D128 causal 509 / 1268 ->
// 148 / 386, bfloat16 B1 H1 T64 D64 17.7 / 23.2 -> 11.2 / 18.3 (faster at every one of 20 shapes tried). What bounds it: one workgroup's chain of loads, products and
// exchanges (~12 us) times the rounds the registers and LDS leave (2 waves per SIMD; float32 D64, 104 KB, one workgroup
// per CU).
// DP = 16 exists only here: one k chunk, and half of the 32-wide output tile unused.
#include <type_traits>

#include "sdpa_common.hpp"
#include "sdpa_params.hpp"

namespace theria {

template <typename T, int DP>
struct Small {
  static constexpr int R = 64, NT = 128;  // rows per tile, threads
  using OP = Ops<T, DP>;
  using F = typename OP::F;
  using Stage = TileStage<T, R, DP, NT>;
  static constexpr int NKC = DP / OP::KC, NPC = 32 / OP::KC, NDT = DP < 32 ? 1 : DP / 32;
  // DP = 16: transpose reads take 32 columns, i.e. run 16 past the row's last plane (unused output columns)
  static constexpr int TILE = R * OP::PITCH + 32 / (int)sizeof(T);

  // acc += a x^T for chunk cc of the accumulator tile x (b operand), or x a (x as the a operand).
  struct Terms {
    F hi, lo;
  };
  __device__ __forceinline__ static Terms terms(const f32x16_t& x, int cc) {
    Terms t;
    if constexpr (sizeof(T) == 4)
      t.hi = OP::acc(x, cc);
    else
      split_frag<T>(x, cc, t.hi, t.lo);
    return t;
  }
  __device__ __forceinline__ static f32x16_t mma_b(const F& a, const Terms& x, f32x16_t acc) {
    acc = OP::mma(a, x.hi, acc);
    if constexpr (sizeof(T) == 2) acc = OP::mma(a, x.lo, acc);
    return acc;
  }
  __device__ __forceinline__ static f32x16_t mma_a(const Terms& x, const F& b, f32x16_t acc) {
    acc = OP::mma(x.hi, b, acc);
    if constexpr (sizeof(T) == 2) acc = OP::mma(x.lo, b, acc);
    return acc;
  }
  // out^T (lane per row): rows acc_row of the head dim, column = this lane's row `row`
  __device__ __forceinline__ static void store_t(const MutView& v, int b, int h, int row, const f32x16_t (&a)[NDT],
                                                 float mul, int D, bool vec) {
    const int g = (threadIdx.x >> 5) & 1;
    T* p = (T*)v.p + b * v.sb + h * v.sh;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const int d0 = dt * 32 + 8 * qd + 4 * g;
        if (d0 < D)
          store4<T>(p, v.sr, row, d0, D, a[dt][4 * qd] * mul, a[dt][4 * qd + 1] * mul, a[dt][4 * qd + 2] * mul,
                    a[dt][4 * qd + 3] * mul, vec);
      }
  }
  // out (lane per column d): row k0 + acc_row(r, g)
  __device__ __forceinline__ static void store_c(const MutView& v, int b, int h, int k0, int nrows,
                                                 const f32x16_t (&a)[NDT], float mul, int D) {
    const int lane = threadIdx.x & 63, li = lane & 31, g = lane >> 5;
    T* p = (T*)v.p + b * v.sb + h * v.sh;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
      const int d = dt * 32 + li;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = k0 + acc_row(r, g);
        if (d < D && row < nrows) p[(int64_t)row * v.sr + d] = (T)(a[dt][r] * mul);
      }
    }
  }
};

template <typename T>
__device__ __forceinline__ const T* slab(const View& v, int b, int h) {
  return v.p ? (const T*)v.p + b * v.sb + h * v.sh : nullptr;
}

template <typename T, int DP>
__global__ __launch_bounds__(128, (sizeof(T) == 4 ? DP <= 32 : DP <= 64) ? 2 : 1) void small_bwdbwd_kernel(
    const BwdBwdParams p) {
  using K_ = Small<T, DP>;
  using OP = typename K_::OP;
  using F = typename K_::F;
  constexpr int NKC = K_::NKC, NPC = K_::NPC, NDT = K_::NDT, R = K_::R;
  __shared__ __attribute__((aligned(16))) T tile[4][K_::TILE];
  __shared__ __attribute__((aligned(16))) float sRow[5][R];  // m2, 1 / l, z, r, t of each query

  const Shape& s = p.s;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 31, g = lane >> 5;
  const int b = blockIdx.x / s.H, h = blockIdx.x - b * s.H;
  const T *Q = slab<T>(p.q, b, h), *K = slab<T>(p.k, b, h), *V = slab<T>(p.v, b, h), *dO = slab<T>(p.dout, b, h);
  const T *GQ = slab<T>(p.gq, b, h), *GK = slab<T>(p.gk, b, h), *GV = slab<T>(p.gv, b, h);
  const bool has_gq = GQ != nullptr, has_gk = GK != nullptr, has_gv = GV != nullptr;
  const float c2 = s.scale * kLog2e;
  const int w0 = 32 * wave, my = w0 + li;  // this wave's first row (query or key) and this lane's

  // Every load of the row phase in flight together, and (PRE: where the registers allow) the column phase's tiles.
  constexpr bool PRE = DP <= 32;
  typename K_::Stage qs, os, gs_;
  typename OP::Raw r0[NKC], r1[NKC], r2[NKC];
  auto load_q_side = [&]() {
    qs.load(Q, p.q.sr, 0, s.T, s.D, s.vec);
    os.load(dO, p.dout.sr, 0, s.T, s.D, s.vec);
    if (has_gq) gs_.load(GQ, p.gq.sr, 0, s.T, s.D, s.vec);
  };
  {
    typename K_::Stage a, c, d, e;
    a.load(K, p.k.sr, 0, s.M, s.D, s.vec);
    c.load(V, p.v.sr, 0, s.M, s.D, s.vec);
    if (has_gk) d.load(GK, p.gk.sr, 0, s.M, s.D, s.vec);
    if (has_gv) e.load(GV, p.gv.sr, 0, s.M, s.D, s.vec);
#pragma unroll
    for (int c_ = 0; c_ < NKC; ++c_) {
      r0[c_] = OP::raw(Q, p.q.sr, my, s.T, c_, s.D, s.vec);
      r1[c_] = OP::raw(dO, p.dout.sr, my, s.T, c_, s.D, s.vec);
      r2[c_] = has_gq ? OP::raw(GQ, p.gq.sr, my, s.T, c_, s.D, s.vec) : typename OP::Raw{};
    }
    if (PRE) load_q_side();
    OP::store(a, tile[0], true, c, tile[1], true, d, tile[2], has_gk, e, tile[3], has_gv);
  }
  __syncthreads();

  if (w0 < s.T) {  // wave-uniform
    F qf[NKC], of[NKC], gf[NKC];
#pragma unroll
    for (int c = 0; c < NKC; ++c) {
      qf[c] = OP::frag(r0[c]);
      of[c] = OP::frag(r1[c]);
      gf[c] = OP::frag(r2[c]);
    }
    f32x16_t sc[2], dp[2], gm[2], w[2];
    const int lim = s.causal ? min(s.M, my + 1) : s.M;  // first key this query cannot see
    float m2 = -THERIA_INF;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      sc[t] = dp[t] = gm[t] = w[t] = zero16();
      if (32 * t < s.M) {
#pragma unroll
        for (int c = 0; c < NKC; ++c) {
          const F kf = OP::cols(tile[0], 32 * t + li, c);
          sc[t] = OP::mma(kf, qf[c], sc[t]);
          dp[t] = OP::mma(OP::cols(tile[1], 32 * t + li, c), of[c], dp[t]);
          if (has_gq) gm[t] = OP::mma(kf, gf[c], gm[t]);
          if (has_gk) gm[t] = OP::mma(OP::cols(tile[2], 32 * t + li, c), qf[c], gm[t]);
          if (has_gv) w[t] = OP::mma(OP::cols(tile[3], 32 * t + li, c), of[c], w[t]);
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        sc[t][r] = 32 * t + acc_row(r, g) < lim ? mul_rn(sc[t][r], c2) : -THERIA_INF;
        m2 = fmaxf(m2, sc[t][r]);
      }
    }
    m2 = pair_max(m2);  // -inf: every visible score is (or is NaN, which the sums below keep)
    float l = 0.f, a = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float pv = sc[t][r] == -THERIA_INF ? 0.f : fast_exp2(sc[t][r] - m2);
        sc[t][r] = pv;
        l += pv;
        a = fmaf(pv, dp[t][r], a);
      }
    l = pair_sum(l);
    const bool none = l == 0.f;  // no visible key: P = 0
    const float inv = none ? 0.f : 1.f / l, z = pair_sum(a) * inv;
    float rr = 0.f, tt = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        sc[t][r] *= inv;
        gm[t][r] *= s.scale;
        dp[t][r] -= z;
        rr = fmaf(sc[t][r], gm[t][r], rr);
        tt = fmaf(sc[t][r], fmaf(gm[t][r], dp[t][r], w[t][r]), tt);
      }
    rr = pair_sum(rr);
    tt = pair_sum(tt);
    if (g == 0) {
      const bool ok = my < s.T && !none;  // rows past the end or without a visible key: P = exp2(-inf) = 0
      sRow[0][my] = ok ? m2 : THERIA_INF;
      sRow[1][my] = ok ? inv : 0.f;
      sRow[2][my] = ok ? z : 0.f;
      sRow[3][my] = ok ? rr : 0.f;
      sRow[4][my] = ok ? tt : 0.f;
    }
    f32x16_t accQ[NDT], accO[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) accQ[dt] = accO[dt] = zero16();
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if (32 * t >= s.M) continue;  // uniform
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float pv = sc[t][r], gr = gm[t][r] - rr, dz = dp[t][r];
        gm[t][r] = pv * gr;                              // Gbar_dP
        w[t][r] = pv * (fmaf(gr, dz, w[t][r]) - tt);     // Gbar_S
        dp[t][r] = pv * dz;                              // dS
      }
#pragma unroll
      for (int cc = 0; cc < NPC; ++cc) {
        const auto gs = K_::terms(w[t], cc), ds = K_::terms(dp[t], cc), gd = K_::terms(gm[t], cc),
                   pf = K_::terms(sc[t], cc);
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
          accQ[dt] = K_::mma_b(OP::rows(tile[0], 32 * t, cc, dt * 32), gs, accQ[dt]);
          if (has_gk) accQ[dt] = K_::mma_b(OP::rows(tile[2], 32 * t, cc, dt * 32), ds, accQ[dt]);
          accO[dt] = K_::mma_b(OP::rows(tile[1], 32 * t, cc, dt * 32), gd, accO[dt]);
          if (has_gv) accO[dt] = K_::mma_b(OP::rows(tile[3], 32 * t, cc, dt * 32), pf, accO[dt]);
        }
      }
    }
    if (my < s.T) {
      K_::store_t(p.out_gq, b, h, my, accQ, s.scale, s.D, s.vec);
      K_::store_t(p.out_gdo, b, h, my, accO, 1.f, s.D, s.vec);
    }
  }

  if (!PRE) load_q_side();
  // this lane's key as the column phase's operands, from the tiles
  F kf[NKC], vf[NKC], gkf[NKC], gvf[NKC];
#pragma unroll
  for (int c_ = 0; c_ < NKC; ++c_) {
    kf[c_] = OP::cols(tile[0], my, c_);
    vf[c_] = OP::cols(tile[1], my, c_);
    gkf[c_] = has_gk ? OP::cols(tile[2], my, c_) : F{};
    gvf[c_] = has_gv ? OP::cols(tile[3], my, c_) : F{};
  }
  __syncthreads();  // both waves are done with the key-side tiles
  OP::store(qs, tile[0], true, os, tile[1], true, gs_, tile[2], has_gq);
  __syncthreads();
  if (w0 >= s.M) return;

  f32x16_t accK[NDT], accV[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) accK[dt] = accV[dt] = zero16();
  for (int t = 0; 32 * t < s.T; ++t) {
    f32x16_t sc = zero16(), dp = zero16(), gm = zero16(), w = zero16();
#pragma unroll
    for (int c_ = 0; c_ < NKC; ++c_) {
      const F q = OP::cols(tile[0], 32 * t + li, c_), o = OP::cols(tile[1], 32 * t + li, c_);
      sc = OP::template mma<true>(q, kf[c_], sc);
      dp = OP::template mma<true>(o, vf[c_], dp);
      if (has_gq) gm = OP::template mma<true>(OP::cols(tile[2], 32 * t + li, c_), kf[c_], gm);
      if (has_gk) gm = OP::template mma<true>(q, gkf[c_], gm);
      if (has_gv) w = OP::template mma<true>(o, gvf[c_], w);
    }
#pragma unroll
    for (int qd = 0; qd < 4; ++qd) {
      const int o = 32 * t + 8 * qd + 4 * g;
      const f32x4_t m4 = *reinterpret_cast<const f32x4_t*>(sRow[0] + o), i4 = *reinterpret_cast<const f32x4_t*>(sRow[1] + o),
                    z4 = *reinterpret_cast<const f32x4_t*>(sRow[2] + o), r4 = *reinterpret_cast<const f32x4_t*>(sRow[3] + o),
                    t4 = *reinterpret_cast<const f32x4_t*>(sRow[4] + o);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 4 * qd + e;
        float pv = fast_exp2(mul_rn(sc[r], c2) - m4[e]) * i4[e];
        if (s.causal && my > o + e) pv = 0.f;
        const float gr = s.scale * gm[r] - r4[e], dz = dp[r] - z4[e];
        gm[r] = pv * gr;                           // Gbar_dP
        w[r] = pv * (fmaf(gr, dz, w[r]) - t4[e]);  // Gbar_S
        dp[r] = pv * dz;                           // dS
      }
    }
    if (32 * t + 32 > s.T) {  // rows past the end: P = 0, but the score of their zeros against an infinite key is NaN
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (32 * t + acc_row(r, g) >= s.T) gm[r] = w[r] = dp[r] = 0.f;
    }
#pragma unroll
    for (int cc = 0; cc < NPC; ++cc) {
      const auto gs = K_::terms(w, cc), ds = K_::terms(dp, cc), gd = K_::terms(gm, cc);
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) {
        accV[dt] = K_::mma_a(gd, OP::rows(tile[1], 32 * t, cc, dt * 32), accV[dt]);
        accK[dt] = K_::mma_a(gs, OP::rows(tile[0], 32 * t, cc, dt * 32), accK[dt]);
        if (has_gq) accK[dt] = K_::mma_a(ds, OP::rows(tile[2], 32 * t, cc, dt * 32), accK[dt]);
      }
    }
  }
  K_::store_c(p.out_gk, b, h, w0, s.M, accK, s.scale, s.D);
  K_::store_c(p.out_gv, b, h, w0, s.M, accV, 1.f, s.D);
}

// The row term as the general dQ kernel's (kRowFromO): float32, and 16-bit problems holding a row flagged peaked in
// lse, sum_j P dP / sum_j P; other 16-bit problems dO . O.
template <typename T, int DP>
__global__ __launch_bounds__(128, (sizeof(T) == 4 ? DP <= 64 : true) ? 2 : 1) void small_bwd_kernel(const SmallBwdParams p) {
  using K_ = Small<T, DP>;
  using OP = typename K_::OP;
  using F = typename K_::F;
  constexpr int NKC = K_::NKC, NPC = K_::NPC, NDT = K_::NDT, R = K_::R;
  __shared__ __attribute__((aligned(16))) T tile[2][K_::TILE];
  __shared__ __attribute__((aligned(16))) float sRow[2][R];  // lse * log2(e), delta of each query

  const Shape& s = p.s;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 31, g = lane >> 5;
  const int b = blockIdx.x / s.H, h = blockIdx.x - b * s.H;
  const T *Q = slab<T>(p.q, b, h), *K = slab<T>(p.k, b, h), *V = slab<T>(p.v, b, h), *dO = slab<T>(p.dout, b, h);
  const float c2 = s.scale * kLog2e;
  const int w0 = 32 * wave, my = w0 + li;
  const int64_t row_id = (int64_t)blockIdx.x * s.T + my;
  // loads in flight together, as in small_bwdbwd_kernel
  constexpr bool PRE = DP <= 32;
  typename K_::Stage qs, os;
  typename OP::Raw r0[NKC], r1[NKC];
  auto load_q_side = [&]() {
    qs.load(Q, p.q.sr, 0, s.T, s.D, s.vec);
    os.load(dO, p.dout.sr, 0, s.T, s.D, s.vec);
  };
  const float lse = my < s.T ? p.lse[row_id] : THERIA_INF;
  {
    typename K_::Stage a, c;
    a.load(K, p.k.sr, 0, s.M, s.D, s.vec);
    c.load(V, p.v.sr, 0, s.M, s.D, s.vec);
#pragma unroll
    for (int c_ = 0; c_ < NKC; ++c_) {
      r0[c_] = OP::raw(Q, p.q.sr, my, s.T, c_, s.D, s.vec);
      r1[c_] = OP::raw(dO, p.dout.sr, my, s.T, c_, s.D, s.vec);
    }
    if (PRE) load_q_side();
    OP::store(a, tile[0], true, c, tile[1], true);
  }
  // (a barrier of the workgroup either way)
  bool exact = true;
  if constexpr (sizeof(T) == 2)
    exact = __syncthreads_or(lse_peaked(lse));
  else
    __syncthreads();

  if (w0 < s.T) {
    F qf[NKC], of[NKC];
#pragma unroll
    for (int c = 0; c < NKC; ++c) {
      qf[c] = OP::frag(r0[c]);
      of[c] = OP::frag(r1[c]);
    }
    const float lse2 = lse == -THERIA_INF ? THERIA_INF : lse * kLog2e;  // a row without visible keys has P = 0
    float z = 0.f;
    if constexpr (sizeof(T) == 2) {
      if (!exact) {  // dO . O over this lane's half of the head dim, then the pair
        float part = 0.f;
        if (my < s.T) {
#pragma unroll
          for (int c = 0; c < NKC; ++c)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const int col = 16 * c + 8 * g + e;
              if (col < s.D) {
                const int64_t off = (int64_t)my * p.o.sr + col;
                const float ov = p.o_f32 ? ((const float*)p.o.p + b * p.o.sb + h * p.o.sh)[off]
                                         : (float)((const T*)p.o.p + b * p.o.sb + h * p.o.sh)[off];
                part += ov * (float)of[c][e];
              }
            }
        }
        z = pair_sum(part);
      }
    }
    f32x16_t sc[2], dp[2];
    const int lim = s.causal ? min(s.M, my + 1) : s.M;  // first key this query cannot see
    float l = 0.f, a = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      sc[t] = dp[t] = zero16();
      if (32 * t < s.M) {
#pragma unroll
        for (int c = 0; c < NKC; ++c) {
          sc[t] = OP::mma(OP::cols(tile[0], 32 * t + li, c), qf[c], sc[t]);
          dp[t] = OP::mma(OP::cols(tile[1], 32 * t + li, c), of[c], dp[t]);
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float pv = 32 * t + acc_row(r, g) < lim ? fast_exp2(fmaf(sc[t][r], c2, -lse2)) : 0.f;
        sc[t][r] = pv;
        l += pv;
        a = fmaf(pv, dp[t][r], a);
      }
    }
    if (exact) {
      l = pair_sum(l);
      a = pair_sum(a);
      z = l > 0.f ? a / l : 0.f;
    }
    if (g == 0) {
      sRow[0][my] = lse2;
      sRow[1][my] = z;
      if (my < s.T) p.delta[row_id] = z;
    }
    if (p.dq.p) {
      f32x16_t acc[NDT];
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) acc[dt] = zero16();
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if (32 * t >= s.M) continue;  // uniform
#pragma unroll
        for (int r = 0; r < 16; ++r) dp[t][r] = sc[t][r] * (dp[t][r] - z);  // dS
#pragma unroll
        for (int cc = 0; cc < NPC; ++cc) {
          const auto ds = K_::terms(dp[t], cc);
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) acc[dt] = K_::mma_b(OP::rows(tile[0], 32 * t, cc, dt * 32), ds, acc[dt]);
        }
      }
      if (my < s.T) K_::store_t(p.dq, b, h, my, acc, s.scale, s.D, s.vec);
    }
  }

  if (!PRE) load_q_side();
  F kf[NKC], vf[NKC];  // this lane's key, from the tiles
#pragma unroll
  for (int c_ = 0; c_ < NKC; ++c_) {
    kf[c_] = OP::cols(tile[0], my, c_);
    vf[c_] = OP::cols(tile[1], my, c_);
  }
  __syncthreads();  // both waves are done with the key-side tiles
  OP::store(qs, tile[0], true, os, tile[1], true);
  __syncthreads();
  if (w0 >= s.M) return;
  f32x16_t accK[NDT], accV[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) accK[dt] = accV[dt] = zero16();
  for (int t = 0; 32 * t < s.T; ++t) {
    f32x16_t sc = zero16(), dp = zero16();
#pragma unroll
    for (int c_ = 0; c_ < NKC; ++c_) {
      sc = OP::template mma<true>(OP::cols(tile[0], 32 * t + li, c_), kf[c_], sc);
      dp = OP::template mma<true>(OP::cols(tile[1], 32 * t + li, c_), vf[c_], dp);
    }
#pragma unroll
    for (int qd = 0; qd < 4; ++qd) {
      const int o = 32 * t + 8 * qd + 4 * g;
      const f32x4_t l4 = *reinterpret_cast<const f32x4_t*>(sRow[0] + o), z4 = *reinterpret_cast<const f32x4_t*>(sRow[1] + o);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 4 * qd + e;
        float pv = fast_exp2(fmaf(sc[r], c2, -l4[e]));  // rows past the end: lse = +inf
        if (s.causal && my > o + e) pv = 0.f;
        sc[r] = pv;
        dp[r] = pv * (dp[r] - z4[e]);
      }
    }
    if (32 * t + 32 > s.T) {  // as in small_bwdbwd_kernel
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (32 * t + acc_row(r, g) >= s.T) sc[r] = dp[r] = 0.f;
    }
#pragma unroll
    for (int cc = 0; cc < NPC; ++cc) {
      const auto pf = K_::terms(sc, cc), ds = K_::terms(dp, cc);
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) {
        accV[dt] = K_::mma_a(pf, OP::rows(tile[1], 32 * t, cc, dt * 32), accV[dt]);
        accK[dt] = K_::mma_a(ds, OP::rows(tile[0], 32 * t, cc, dt * 32), accK[dt]);
      }
    }
  }
  if (p.dk.p) K_::store_c(p.dk, b, h, w0, s.M, accK, s.scale, s.D);
  K_::store_c(p.dv, b, h, w0, s.M, accV, 1.f, s.D);
}

bool small_problem(const Shape& s) {
  return s.T >= 1 && s.T <= 64 && s.M >= 1 && s.M <= 64 && s.D <= (s.dtype == 0 ? 64 : 128);
}

template <template <typename, int> class L, typename T, typename P>
static hipError_t small_dispatch(const P& p, hipStream_t st) {
  const dim3 grid((unsigned)(p.s.B * p.s.H)), block(128);
  if (grid.x == 0) return hipSuccess;
  if (p.s.D <= 16)
    L<T, 16>::go(p, grid, block, st);
  else if (p.s.D <= 32)
    L<T, 32>::go(p, grid, block, st);
  else if (p.s.D <= 64)
    L<T, 64>::go(p, grid, block, st);
  else if constexpr (sizeof(T) == 2)
    L<T, 128>::go(p, grid, block, st);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}
template <template <typename, int> class L, typename P>
static hipError_t small_dispatch(const P& p, hipStream_t st) {
  switch (p.s.dtype) {
    case 0: return small_dispatch<L, float>(p, st);
    case 1: return small_dispatch<L, _Float16>(p, st);
    case 2: return small_dispatch<L, __bf16>(p, st);
    default: return hipErrorInvalidValue;
  }
}
template <typename T, int DP>
struct SmallBwd {
  static void go(const SmallBwdParams& p, dim3 grid, dim3 block, hipStream_t st) {
    hipLaunchKernelGGL((small_bwd_kernel<T, DP>), grid, block, 0, st, p);
  }
};
template <typename T, int DP>
struct SmallBwdBwd {
  static void go(const BwdBwdParams& p, dim3 grid, dim3 block, hipStream_t st) {
    hipLaunchKernelGGL((small_bwdbwd_kernel<T, DP>), grid, block, 0, st, p);
  }
};
hipError_t launch_small_bwd(const SmallBwdParams& p, hipStream_t st) { return small_dispatch<SmallBwd>(p, st); }
hipError_t launch_small_bwdbwd(const BwdBwdParams& p, hipStream_t st) { return small_dispatch<SmallBwdBwd>(p, st); }

}  // namespace theria
