// Fused SDPA forward for gfx950.
//
// Replaces _fused_sdpa_kernel (reference theria/attention/triton_qk.py:242-304):
// O = softmax(scale * Q K^T) V with an online softmax, saving lse (and the reference's m, l).
//
// Work decomposition: one workgroup = 4 waves; each wave owns QT tiles of 32 query rows of one
// (batch, head) for the whole kernel. The score tile is computed transposed, S^T = K Q^T, so that in
// the accumulator layout each lane owns one query (column li) and 16 keys: the row max and row sum
// are in-lane reductions plus one permlane32 swap, and the output accumulator O^T = V^T P^T is also
// lane-per-query, so the online-softmax rescale is a per-lane scalar multiply. Q stays in registers
// as the B operand; K/V tiles of 64 keys are staged in LDS (register-prefetched one tile ahead), and
// every K fragment and every V^T fragment (LDS transpose read) read from LDS feeds QT MFMAs: with
// one MFMA per fragment the 32x32x16 MFMA rate equals the CU's LDS bandwidth, so QT = 2 halves the
// LDS traffic per FLOP. exp is evaluated as exp2 with scale*log2(e) folded into one FMA. The running
// max used for P is only moved when a row's max grows by more than 2^8 (P <= 256 stays exact in
// float32 and representable in bf16/fp16), so the O rescale is skipped on almost every tile.
#include <algorithm>
#include <type_traits>

#include "dispatch.hpp"
#include "sdpa_common.hpp"
#include "fwd_split.hpp"

#ifndef FWD_MINW
#define FWD_MINW 2
#endif
constexpr int FWD_MAX_SPLITS = 64;  // what the combining kernel takes

namespace theria {

// NW waves per workgroup: four, or two for at most 64 queries (QT = 1), where two of four would have no rows (us, four
// -> two waves: float32 B400 H4 T64 D16 17.9 -> 13.8, B128 H8 T32 D32 11.7 -> 8.1, bfloat16 B64 H8 T64 D128 13.5 -> 9.1).
// SPLIT: one part of the keys per workgroup (FwdParams::nsplit), no causal mask.
template <typename T, int DP, bool CAUSAL, int QT, int BN, int NW = 4, bool SPLIT = false>
__global__ __launch_bounds__(64 * NW, (DP <= 64 ? FWD_MINW : 1)) void fwd_kernel(const FwdParams p) {
  using OP = Ops<T, DP>;
  using F = typename OP::F;
  constexpr int KC = OP::KC;
  constexpr int BM = 32 * NW * QT, NT = 64 * NW;
  constexpr int PITCH = OP::PITCH;
  constexpr int NDT = DP / 32, NKC = DP / KC, NPC = 32 / KC, NST = BN / 32;
  __shared__ __attribute__((aligned(16))) T sK[BN * PITCH];
  __shared__ __attribute__((aligned(16))) T sV[BN * PITCH];

  const Shape& s = p.s;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 31, g = lane >> 5;
  const int nqb = (s.T + BM - 1) / BM;
  const int bid = xcd_remap(blockIdx.x, gridDim.x);
  const int unit = bid / nqb;  // (batch, head) and, with SPLIT, the part of its keys
  int qb = bid - unit * nqb;
  const int bh = SPLIT ? unit / p.nsplit : unit, part = SPLIT ? unit - bh * p.nsplit : 0;
  if (CAUSAL) qb = nqb - 1 - qb;  // longest rows first
  const int b = bh / s.H, h = bh - b * s.H;
  const T* Q = (const T*)p.q.p + b * p.q.sb + h * p.q.sh;
  const FwdPart kp = fwd_part(s, SPLIT ? p.nsplit : 1, part);
  const int M = SPLIT ? kp.keys : s.M;  // this workgroup's keys
  const T* K = (const T*)p.k.p + b * p.k.sb + h * p.k.sh + (SPLIT ? kp.key0 * p.k.sr : 0);
  const T* V = (const T*)p.v.p + b * p.v.sb + h * p.v.sh + (SPLIT ? kp.key0 * p.v.sr : 0);
  const int q0w = qb * BM + wave * 32 * QT;  // query tile j of this wave starts at q0w + 32 j
  const int64_t rowbase = (int64_t)bh * s.T;

  F qf[QT][NKC];
  f32x16_t o[QT][NDT];
  float m_use[QT], m_max[QT], l_part[QT];
#pragma unroll
  for (int j = 0; j < QT; ++j) {
    const int myq = q0w + 32 * j + li;
    typename OP::Raw qraw[NKC];
#pragma unroll
    for (int c = 0; c < NKC; ++c) qraw[c] = OP::raw(Q, p.q.sr, myq, s.T, c, s.D, s.vec);
#pragma unroll
    for (int c = 0; c < NKC; ++c) qf[j][c] = OP::frag(qraw[c]);
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) o[j][dt] = zero16();
    m_use[j] = -THERIA_INF;  // offset of P in the log2 domain
    m_max[j] = -THERIA_INF;  // exact running row max (log2 domain)
    l_part[j] = 0.f;         // this lane's share of the row sum
  }
  const float c2 = s.scale * kLog2e;

  int kend = M;
  if (CAUSAL) kend = min(M, qb * BM + BM);
  const int nkt = (kend + BN - 1) / BN;
  TileStage<T, BN, DP, NT> stK, stV;
  if (nkt > 0) {
    stK.load_any(K, p.k.sr, 0, M, s.D, s.vec);
    stV.load_any(V, p.v.sr, 0, M, s.D, s.vec);
  }
  // MASK: the tile reaches past the last key or (causal) past the block's first query; those tiles take their own copy of
  // the loop (a mask behind a uniform branch becomes a compare and a select per score in every tile).
  auto step = [&](auto mask_tag, int kt) __attribute__((always_inline)) {
    constexpr bool MASK = decltype(mask_tag)::value;
    const int k0 = kt * BN;
    __syncthreads();
    OP::store(stK, sK, true, stV, sV, true);
    __syncthreads();
    if (kt + 1 < nkt) {
      stK.load_any(K, p.k.sr, k0 + BN, M, s.D, s.vec);
      stV.load_any(V, p.v.sr, k0 + BN, M, s.D, s.vec);
    }
    if (CAUSAL && k0 > q0w + 32 * QT - 1) return;  // tile entirely above this wave's diagonal

    f32x16_t sc[QT][NST];
#pragma unroll
    for (int t = 0; t < NST; ++t) {
#pragma unroll
      for (int j = 0; j < QT; ++j) sc[j][t] = zero16();
#pragma unroll
      for (int c = 0; c < NKC; ++c) {
        const F kfr = OP::cols(sK, t * 32 + li, c);
#pragma unroll
        for (int j = 0; j < QT; ++j) sc[j][t] = OP::mma(kfr, qf[j][c], sc[j][t]);
      }
    }
    // masked scores become -inf, so P = 0 there
    if (MASK && ((k0 + BN > M) || (CAUSAL && k0 + BN - 1 > q0w))) {
#pragma unroll
      for (int j = 0; j < QT; ++j) {
        const int lim = CAUSAL ? min(M, q0w + 32 * j + li + 1) : M;  // first key this query cannot see
#pragma unroll
        for (int t = 0; t < NST; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (k0 + t * 32 + acc_row(r, g) >= lim) sc[j][t][r] = -THERIA_INF;
      }
    }
#pragma unroll
    for (int j = 0; j < QT; ++j) {
      {
        float mx = -THERIA_INF;
#pragma unroll
        for (int t = 0; t < NST; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[j][t][r]);
        mx = pair_max(mx) * c2;
        m_max[j] = fmaxf(m_max[j], mx);
        const bool resc = mx > m_use[j] + 8.f;
        if (__any(resc)) {
          const float alpha = resc ? fast_exp2(m_use[j] - mx) : 1.f;
          m_use[j] = resc ? mx : m_use[j];
          l_part[j] *= alpha;
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[j][dt][r] *= alpha;
        }
      }
      // m_use is -inf only while every key seen so far is masked (then every score is -inf and P = 0)
      const float moff = m_use[j] == -THERIA_INF ? 0.f : m_use[j];
      float ls = 0.f;
#pragma unroll
      for (int t = 0; t < NST; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float e = fast_exp2(fmaf(sc[j][t][r], c2, -moff));
          sc[j][t][r] = e;
          ls += e;
        }
      l_part[j] += ls;
    }
#pragma unroll
    for (int t = 0; t < NST; ++t)
#pragma unroll
      for (int cc = 0; cc < NPC; ++cc) {
        F pf[QT];
#pragma unroll
        for (int j = 0; j < QT; ++j) pf[j] = OP::acc(sc[j][t], cc);
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
          const F vfr = OP::rows(sV, t * 32, cc, dt * 32);
#pragma unroll
          for (int j = 0; j < QT; ++j) o[j][dt] = OP::mma(vfr, pf[j], o[j][dt]);
        }
      }
  };
  // Tiles with every key in range and visible to the block. Two copies of the loop pay in float32 only (16-bit D20 T1000
  // 26.0 -> 27.0 us), and not in its two-wave workgroups above head dim 32, which spill.
  constexpr bool PEEL = sizeof(T) == 4 && (NW == 4 || DP == 32);
  const int nfull = PEEL ? (CAUSAL ? min(M / BN, qb * BM / BN) : M / BN) : 0;
  int kt = 0;
  for (; kt < min(nfull, nkt); ++kt) step(std::false_type{}, kt);
  for (; kt < nkt; ++kt) step(std::true_type{}, kt);

#pragma unroll
  for (int j = 0; j < QT; ++j) {
    const int myq = q0w + 32 * j + li;
    const bool qvalid = myq < s.T;
    const int64_t row_id = rowbase + myq;
    if constexpr (SPLIT) {
      const float l = pair_sum(l_part[j]);
      if (qvalid) {
        float* w = p.ws + ((int64_t)part * s.B * s.H * s.T + row_id) * fwd_split_row_floats(s.D);
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
          for (int qd = 0; qd < 4; ++qd) {
            const int d0 = dt * 32 + 8 * qd + 4 * g;
            if (d0 < s.D)  // (columns past D are zero)
              *reinterpret_cast<f32x4_t*>(w + d0) =
                  f32x4_t{o[j][dt][4 * qd], o[j][dt][4 * qd + 1], o[j][dt][4 * qd + 2], o[j][dt][4 * qd + 3]};
          }
        if (g == 0)
          *reinterpret_cast<f32x4_t*>(w + fwd_split_row_floats(s.D) - 4) =
              f32x4_t{m_use[j], l, m_max[j], m_max[j] == -THERIA_INF ? 0.f : fast_exp2(m_max[j] - m_use[j])};
      }
    } else {
      const float l = pair_sum(l_part[j]);
      const float inv = l > 0.f ? 1.f / l : 0.f;
      if (qvalid) {
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
          for (int qd = 0; qd < 4; ++qd) {
            const int d0 = dt * 32 + 8 * qd + 4 * g;
            if (d0 < s.D) {
              const float a0 = o[j][dt][4 * qd] * inv, a1 = o[j][dt][4 * qd + 1] * inv;
              const float a2 = o[j][dt][4 * qd + 2] * inv, a3 = o[j][dt][4 * qd + 3] * inv;
              if (p.o_f32) {
                float* O = (float*)p.o.p + b * p.o.sb + h * p.o.sh;
                store4<float>(O, p.o.sr, myq, d0, s.D, a0, a1, a2, a3, s.vec);
              } else {
                T* O = (T*)p.o.p + b * p.o.sb + h * p.o.sh;
                store4<T>(O, p.o.sr, myq, d0, s.D, a0, a1, a2, a3, s.vec);
              }
            }
          }
        if (g == 0) {
          // 16-bit: flag a peaked row, largest probability exp2(m_max - m_use) / l above 1/4 (log2: -2)
          const float lse2 = m_use[j] + __builtin_log2f(l);
          const bool peaked = sizeof(T) == 2 && m_max[j] - lse2 > -2.f;
          p.lse[row_id] = l > 0.f ? (sizeof(T) == 2 ? lse_with_flag(lse2 * kLn2, peaked) : lse2 * kLn2) : -THERIA_INF;
          if (p.row_max) p.row_max[row_id] = m_max[j] * kLn2;
          if (p.row_sum) p.row_sum[row_id] = l > 0.f ? l * fast_exp2(m_use[j] - m_max[j]) : 0.f;
        }
      }
    }
  }
}

// The parts of a split forward combined: GP groups of 32 lanes (4 columns each) per row, group i taking parts i, i + GP,
// ... (at most 8 each) and all of a row's loads in flight together; the groups sum through LDS. With M* = max_s m_s and
// w_s = exp2(m_s - M*): O = sum_s w_s O_s / L, L = sum_s w_s l_s, lse = (M* + log2 L) ln 2; the row is flagged peaked
// when the largest of the parts' bounds w_s pk_s exceeds L / 4, as in the unsplit kernels.
template <typename T, int GP>
__global__ __launch_bounds__(256) void fwd_combine_kernel(const FwdParams p) {
  constexpr int RPB = 8 / GP;  // rows per workgroup
  __shared__ __attribute__((aligned(16))) f32x4_t sO[8][32];
  const Shape& s = p.s;
  const int64_t rows = (int64_t)s.B * s.H * s.T;
  const int g32 = threadIdx.x >> 5, grp = g32 % GP, ln = threadIdx.x & 31, d0 = 4 * ln;
  const int64_t row0 = (int64_t)blockIdx.x * RPB + g32 / GP;
  const bool ok = row0 < rows;
  const int64_t row = ok ? row0 : rows - 1;
  const int RF = fwd_split_row_floats(s.D);
  const float* w = p.ws + row * RF;
  // lane ln: the statistics of parts ln and ln + 32
  f32x4_t st[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    st[k] = f32x4_t{-THERIA_INF, 0.f, -THERIA_INF, 0.f};
    if (ln + 32 * k < p.nsplit) st[k] = *reinterpret_cast<const f32x4_t*>(w + (ln + 32 * k) * rows * RF + RF - 4);
  }
  f32x4_t x[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int i = grp + GP * j;
    x[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (i < p.nsplit && d0 < s.D) x[j] = *reinterpret_cast<const f32x4_t*>(w + i * rows * RF + d0);
  }
  float mt = fmaxf(st[0][0], st[1][0]), mm = fmaxf(st[0][2], st[1][2]);
#pragma unroll
  for (int k = 16; k > 0; k >>= 1) {
    mt = fmaxf(mt, __shfl_xor(mt, k));
    mm = fmaxf(mm, __shfl_xor(mm, k));
  }
  float f[2], l = 0.f, pk = 0.f;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    f[k] = st[k][0] == -THERIA_INF ? 0.f : fast_exp2(st[k][0] - mt);
    l = fmaf(f[k], st[k][1], l);
    pk = fmaxf(pk, f[k] * st[k][3]);
  }
#pragma unroll
  for (int k = 16; k > 0; k >>= 1) {
    l += __shfl_xor(l, k);
    pk = fmaxf(pk, __shfl_xor(pk, k));
  }
  f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int i = grp + GP * j;  // < 64; the first 32 parts' weights are in f[0]
    const float fi = __shfl(GP * j < 32 ? f[0] : f[1], i % 32, 32);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = fmaf(fi, x[j][e], o[e]);
  }
  if constexpr (GP > 1) {
    sO[g32][ln] = o;
    __syncthreads();
    if (grp != 0) return;
#pragma unroll
    for (int i = 1; i < GP; ++i) {
      const f32x4_t y = sO[g32 + i][ln];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] += y[e];
    }
  }
  if (!ok) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  const int64_t bh = row / s.T;
  const int q = (int)(row - bh * s.T), b = (int)(bh / s.H), h = (int)(bh - (int64_t)b * s.H);
  if (d0 < s.D) {
    if (p.o_f32) {
      float* O = (float*)p.o.p + b * p.o.sb + h * p.o.sh;
      store4<float>(O, p.o.sr, q, d0, s.D, o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv, s.vec);
    } else {
      T* O = (T*)p.o.p + b * p.o.sb + h * p.o.sh;
      store4<T>(O, p.o.sr, q, d0, s.D, o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv, s.vec);
    }
  }
  if (d0 == 0) {
    const float lse = (mt + __builtin_log2f(l)) * kLn2;
    p.lse[row] = l > 0.f ? (sizeof(T) == 2 ? lse_with_flag(lse, pk > kPeakedFrac * l) : lse) : -THERIA_INF;
    if (p.row_max) p.row_max[row] = mm * kLn2;
    if (p.row_sum) p.row_sum[row] = l > 0.f ? l * fast_exp2(mt - mm) : 0.f;
  }
}

// Tile choices (compile-time knobs; the defaults are the measured best on MI355X).
#ifndef FWD_BN_QT2
#define FWD_BN_QT2 64
#endif
#ifndef FWD_QT_MAX
#define FWD_QT_MAX 2
#endif
// Query tiles per wave: 2 where the registers allow it and the sequence fills the block.
template <int DP> constexpr int fwd_qt(int T) { return (FWD_QT_MAX >= 2 && DP <= 64 && T > 128) ? 2 : 1; }

// Keys split over workgroups where the 128-query blocks would fill at most a quarter of the CUs (float32, whose tiles
// take three times as long: half), in parts of at least two 64-key tiles, one part per idle CU. The split costs the
// partial rows' round trip and a launch, 5-8 us, so short sweeps stay whole: at 16-bit head dims up to 64 a tile takes
// ~0.7 us and the lines cross at 20 tiles (us, whole -> split: B1 H8 T1024 M1024 D64 14.1 -> 16.2, B1 H4 T2048 M2048 D64
// 24.0 -> 19.8), at larger ones at 10 (B1 H2 T1024 M700 D128 16.0 -> 13.4), and for float32 and the general kernel's 16-bit
// blocks (up to 128 queries) at 8 (float32 B1 H4 T300 M500 D32 18.5 -> 11.6, B1 H16 T100 M500 D128 18.6 -> 12.0). Two parts
// only pay in float32 (bfloat16 B1 H8 T2048 M2048 D128 36.5 -> 37.8, float32 B1 H16 T700 M700 D128 71.6 -> 53.1).
// B1 H16 T100 M6000 D128 bfloat16: 148-168 -> 21 us (16 workgroups -> 256; 50 MB read once, 10 us at a copy's rate); B1 H4
// T512 M8192 D64 81.0 -> 18.6 us.
int fwd_splits(const Shape& s) {
  if (s.causal || s.T < 1) return 1;
  const int64_t blocks = (int64_t)((s.T + 127) / 128) * s.B * s.H, tiles = (s.M + 63) / 64, cus = device_cu_count();
  const bool f32 = s.dtype == 0;
  const int min_tiles = f32 ? 8 : (s.D <= 64 ? 20 : (s.T <= 128 ? 8 : 10));
  if (blocks == 0 || blocks * (f32 ? 2 : 4) > cus || tiles < min_tiles) return 1;
  const int64_t n = std::min<int64_t>({cus / blocks, tiles / 2, FWD_MAX_SPLITS});
  const int64_t per = (tiles + n - 1) / n;  // tiles per part (fwd_part), so that no part is empty
  return (int)((tiles + per - 1) / per);
}

// Pipelined 16-bit forward (sdpa_fwd_pipe.hip); false when it does not cover the problem.
template <typename T, bool CAUSAL>
bool launch_fwd_pipe(const FwdParams& p, hipStream_t st, hipError_t* err);

struct FwdLauncher {
  template <typename T, int DP, bool CAUSAL>
  static hipError_t run(const FwdParams& p, hipStream_t st) {
    if constexpr (!CAUSAL) {
      if (p.nsplit > 1) {
        const int64_t rows = (int64_t)p.s.B * p.s.H * p.s.T, nblk = (int64_t)((p.s.T + 127) / 128) * p.s.B * p.s.H * p.nsplit;
        hipError_t err = hipSuccess;
        bool done = false;
        if constexpr (sizeof(T) == 2) done = launch_fwd_pipe<T, false>(p, st, &err);
        if (!done)
          hipLaunchKernelGGL((fwd_kernel<T, DP, false, 1, 64, 4, true>), dim3((unsigned)nblk), dim3(256), 0, st, p);
        auto combine = [&](auto gp) {
          constexpr int GP = decltype(gp)::value;
          hipLaunchKernelGGL((fwd_combine_kernel<T, GP>), dim3((unsigned)((rows * GP + 7) / 8)), dim3(256), 0, st, p);
        };
        if (p.nsplit <= 8)
          combine(std::integral_constant<int, 1>{});
        else if (p.nsplit <= 16)
          combine(std::integral_constant<int, 2>{});
        else if (p.nsplit <= 32)
          combine(std::integral_constant<int, 4>{});
        else
          combine(std::integral_constant<int, 8>{});
        return err != hipSuccess ? err : hipGetLastError();
      }
    }
    if constexpr (sizeof(T) == 2) {
      hipError_t err;
      if (launch_fwd_pipe<T, CAUSAL>(p, st, &err)) return err;
    }
    // Two query tiles per wave only for 16-bit inputs: with float32 fragments (twice the registers)
    // that variant spills ~150 VGPRs and runs at half the one-tile rate.
    // Two-wave workgroups where four-wave ones (two of whose waves have no rows) would not all be resident at once;
    // below that the wider workgroup stages its tiles sooner (float32 D64 B24 H16 T52: 10.7 against 13.0 us).
    const int64_t nbh = (int64_t)p.s.B * p.s.H;
    if (p.s.T >= 1 && p.s.T <= 64 && nbh > (int64_t)device_cu_count() * (DP <= 64 ? 2 : 1)) {
      hipLaunchKernelGGL((fwd_kernel<T, DP, CAUSAL, 1, 64, 2>), dim3((unsigned)nbh), dim3(128), 0, st, p);
      return hipGetLastError();
    }
    const int qt = sizeof(T) == 2 ? fwd_qt<DP>(p.s.T) : 1;
    const int bm = 128 * qt;
    const int64_t nblk = (int64_t)((p.s.T + bm - 1) / bm) * p.s.B * p.s.H;
    if (nblk == 0) return hipSuccess;
    if constexpr (DP <= 64 && sizeof(T) == 2) {
      if (qt == 2) {
        hipLaunchKernelGGL((fwd_kernel<T, DP, CAUSAL, 2, FWD_BN_QT2>), dim3((unsigned)nblk), dim3(256), 0, st, p);
        return hipGetLastError();
      }
    }
    hipLaunchKernelGGL((fwd_kernel<T, DP, CAUSAL, 1, 64>), dim3((unsigned)nblk), dim3(256), 0, st, p);
    return hipGetLastError();
  }
};

hipError_t launch_fwd(const FwdParams& p, hipStream_t st) { return dispatch_all<FwdLauncher>(p, st); }

}  // namespace theria
