// SDPA double backward for 16-bit inputs on gfx950: the key-split row kernel and the query-split column kernel. The
// formulas are in sdpa_bwdbwd.hip, whose kernels take the other problems.
//
// Both take LDS-DMA tiles and workgroups of two wave groups: the key-split row kernel (bwdbwd_rows_ks_kernel) forms the
// exact row terms, G_Q and G_dO in one launch (the groups split each query block's key tiles and combine through LDS),
// and the query-split column kernel (bwdbwd_cols_qs_kernel) G_K and G_V (the groups split each key block's query tiles).
#include <initializer_list>
#include <type_traits>

#include "sdpa_common.hpp"
#include "sdpa_lds.hpp"
#include "sdpa_params.hpp"

namespace theria {

// The split kernels' LDS-DMA tiles: 16-bit inputs, a head dim that is a multiple of 8 (computed at 64 or 128, the tile
// columns past D zero-filled by the DMA), 16-byte-aligned views, and every (batch, head) slab of the streamed tensors
// (rows x row stride) below 2^31 bytes.
template <typename T>
static bool split_tiles_ok(const BwdBwdParams& p, int64_t rows, std::initializer_list<const View*> streamed) {
  if (!(sizeof(T) == 2 && p.s.D % 8 == 0 && p.s.vec)) return false;
  for (const View* v : streamed)
    if (v->p && !slab_fits_dma(rows, v->sr, p.s.D)) return false;
  return true;
}
template <typename T>
bool rows_ks_ok(const BwdBwdParams& p) {
  return split_tiles_ok<T>(p, p.s.M, {&p.k, &p.v, &p.gk, &p.gv});
}
template <typename T>
bool cols_qs_ok(const BwdBwdParams& p) {
  return split_tiles_ok<T>(p, p.s.T, {&p.q, &p.dout, &p.gq});
}

// The row pass for 16-bit inputs with LDS-DMA tiles, computed at DP = 64 or 128 (FD: the head dim is DP; otherwise a
// multiple of 8, the tile columns past D zero-filled), as two key groups: at DP = 64 of four waves (eight-wave workgroups
// of 128 queries, two waves per SIMD), at 128 of two (64 queries, 32-key tiles, one wave per SIMD at up to 512
// registers; at 128 the general row kernel spilled and swept every key per wave, and the row terms and G_dO were launches
// of their own. Double backward, bfloat16 D128, before -> here: B2 H8 T1024 472 -> 161 us, causal 383 -> 146, B1 H4 T8192
// 3987 -> 1960, B8 H16 T512 596 -> 330, B64 H8 T65 236 -> 159). The keys of each query block are split between the
// groups, whose partial sums meet in LDS. Each group makes two passes over its key tiles:
//   1. with P from the forward's lse: L = sum_j P, sum_j P Gam and the largest P, and the D-wide products
//      A = sum_j (P o Gam) V + sum_j P gV and O = sum_j P V, partial per group, then exchanged. Then
//      sum_j P dP = dO . O and sum_j P (Gam dP + W) = dO . A, which give the row's exact normaliser (P_c = P / L:
//      a 16-bit forward's lse comes from rounded probabilities, so P sums to one only within ~2^-9), the row
//      term z = sum_j P dP / L and the second-order row terms r = sum_j P_c Gam and t = sum_j P_c E1 with
//      E1 = Gam (dP - z) + W, i.e. t = (dO . A - z sum_j P Gam) / L; and G_dO = (A - r O) / L, the JVP of O;
//   2. G_Q = s sum_j (Gbar_S K + dS gK) with Gbar_S = P_c o ((Gam - r)(dP - z) + W - t), the exact form, in two
//      D-wide accumulators.
// P, P o Gam, Gbar_S and dS enter as two 16-bit terms each in waves holding a row flagged peaked in the forward's lse, and
// at DP = 128 in every wave: the general kernel there summed z and t in float32, took the JVP's two-term products for G_dO,
// and redid whole 128-row blocks holding a flagged row in two terms, and with one term in the other waves G_dO's error was
// 1.4 times its rounding and G_Q's up to 1.09 times that kernel's (two terms: no output's error is larger, over 48 calls at
// D 72..128 and std 0.5..2; they take 0 to 20 of the 146 to 330 us above).
// Every row takes the exact form (no centring, no second launch for flagged rows, no separate row-term or JVP
// pass); the gQ fragments sit in LDS, so that each pass's two accumulators, the per-wave Q and dO fragments and
// the products fit 256 registers. Writes G_Q and G_dO, and r, t, z and lse + ln L (flagged peaked when the
// row's largest P_c exceeds 1/4) for the column kernel. ALL: gQ, gK and gV are all given (the presence tests are
// then constants, and the loop bodies have no branches between their products).
template <typename T, bool CAUSAL, bool ALL, bool FD, int DP>
__global__ __launch_bounds__(DP == 64 ? 512 : 256, DP == 64 ? 2 : 1) void bwdbwd_rows_ks_kernel(const BwdBwdParams p) {
  using MM = Mfma<T>;
  using F = typename MM::frag_t;
  static_assert(sizeof(T) == 2, "16-bit inputs only");
  constexpr int NW = DP == 64 ? 4 : 2, GT = 64 * NW, BM = 32 * NW, BN = DP == 64 ? 64 : 32, NST = BN / 32;
  constexpr int NDT = DP / 32, NKC = DP / MM::KC, NPC = 32 / MM::KC;
  constexpr int TB = BN * DP * 2;  // bytes per tile
  // DP = 64: each group fills its own tiles; 128: all four waves fill both groups' (a slab is then 16 rows)
  constexpr bool JOINT = DP == 128;
  using Dma = SwzDma<4, DP>;
  constexpr int NSLAB = BN / Dma::SLAB_ROWS;
  static_assert(NSLAB * Dma::SLAB_ROWS == BN, "key tiles must be whole DMA slabs");
  // [group][set][K, V, gK, gV]; reused for the exchanges between the passes and after the second
  __shared__ __attribute__((aligned(1024))) char smem[2 * 2 * 4 * TB];
  static_assert(sizeof(smem) >= 4 * (4096 + 2 * NDT * 16 * GT), "the exchanges fit in the tile memory");
  // the gQ fragments of the four query slices (both key groups read them; kept here rather than in registers,
  // which the two passes' accumulators fill): fragment c of lane l of slice w at (w * NKC + c) * 64 + l
  __shared__ __attribute__((aligned(16))) F sGQ[NW * NKC * 64];

  const Shape& s = p.s;
  const int lane = threadIdx.x & 63, li = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = (unsigned)wave / NW, wig = (unsigned)wave % NW;  // key group, wave in group
  const int nqb = (s.T + BM - 1) / BM;
  const int bid = xcd_remap(blockIdx.x, gridDim.x);
  const int bh = bid / nqb;
  int qb = bid - bh * nqb;
  if (CAUSAL) qb = nqb - 1 - qb;  // longest first
  const int b = bh / s.H, h = bh - b * s.H;
  const T* Q = (const T*)p.q.p + b * p.q.sb + h * p.q.sh;
  const T* K = (const T*)p.k.p + b * p.k.sb + h * p.k.sh;
  const T* V = (const T*)p.v.p + b * p.v.sb + h * p.v.sh;
  const T* dO = (const T*)p.dout.p + b * p.dout.sb + h * p.dout.sh;
  const bool has_gq = ALL || p.gq.p != nullptr, has_gk = ALL || p.gk.p != nullptr, has_gv = ALL || p.gv.p != nullptr;
  const T* GQ = has_gq ? (const T*)p.gq.p + b * p.gq.sb + h * p.gq.sh : nullptr;
  const T* GK = has_gk ? (const T*)p.gk.p + b * p.gk.sb + h * p.gk.sh : nullptr;
  const T* GV = has_gv ? (const T*)p.gv.p + b * p.gv.sb + h * p.gv.sh : nullptr;
  const int q0w = qb * BM + wig * 32;
  const int myq = q0w + li;
  const bool qvalid = myq < s.T;
  const int64_t row_id = (int64_t)bh * s.T + myq;

  F qf[NKC], dof[NKC];
#pragma unroll
  for (int c = 0; c < NKC; ++c) {
    qf[c] = gload_frag<T>(Q, p.q.sr, myq, s.T, c, s.D, s.vec);
    dof[c] = gload_frag<T>(dO, p.dout.sr, myq, s.T, c, s.D, s.vec);
    // read after the first barrier of the first sweep
    if (has_gq && grp == 0) sGQ[(wig * NKC + c) * 64 + lane] = gload_frag<T>(GQ, p.gq.sr, myq, s.T, c, s.D, s.vec);
  }
  const float c2 = s.scale * kLog2e;
  const float lse_raw = qvalid ? p.lse_fwd[row_id] : THERIA_INF;
  const float lse2 = lse_raw * kLog2e;
  float moff = lse2 == -THERIA_INF ? THERIA_INF : lse2;  // a row without visible keys has P = 0; pass 2: P_c
  float z = 0.f;                                          // pass 2: the row term (pass 1 forms dP itself)
  // two-term products (uniform per wave; the forward's bound: a superset of the peaked rows)
  const bool split = DP == 128 || __any(lse_peaked(lse_raw));

  int kend = s.M;
  if (CAUSAL) kend = min(s.M, qb * BM + BM);
  const int nkt = (kend + BN - 1) / BN;
  const int half = (nkt + 1) / 2;
  const int kt0 = grp * half, kt1 = min(nkt, kt0 + half);  // this group's tiles [kt0, kt1)

  // S^T, Gam^T / s and (FULL) W^T and dP^T - z of 32-key subtile st of the tile in (tK, tV, tgK, tgV); P from S.
  // MASK: the tile reaches past the last key or (causal) past this wave's first query.
  auto products = [&](auto full_tag, auto mask_tag, int k0s, const char* tK, const char* tV, const char* tgK,
                      const char* tgV, int st, f32x16_t& pv, f32x16_t& gm, f32x16_t& w,
                      f32x16_t& dpz) __attribute__((always_inline)) {
    constexpr bool FULL = decltype(full_tag)::value;
    constexpr bool MASK = decltype(mask_tag)::value;
    f32x16_t sc = zero16();
    gm = zero16();
    if constexpr (FULL) {
      w = zero16();
#pragma unroll
      for (int r = 0; r < 16; ++r) dpz[r] = -z;
    }
#pragma unroll
    for (int c = 0; c < NKC; ++c) {
      const F kfr = swz_cols<T, DP>(tK, 32 * st + li, c);
      sc = MM::mma(kfr, qf[c], sc);
      if constexpr (FULL) dpz = MM::mma(swz_cols<T, DP>(tV, 32 * st + li, c), dof[c], dpz);
      if (has_gq) gm = MM::mma(kfr, sGQ[(wig * NKC + c) * 64 + lane], gm);
      if (has_gk) gm = MM::mma(swz_cols<T, DP>(tgK, 32 * st + li, c), qf[c], gm);
      if constexpr (FULL)
        if (has_gv) w = MM::mma(swz_cols<T, DP>(tgV, 32 * st + li, c), dof[c], w);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float x = fast_exp2(fmaf(sc[r], c2, -moff));
      if constexpr (MASK) {
        const int key = k0s + acc_row(r, g);
        if (key >= s.M || (CAUSAL && key > myq)) x = 0.f;
      }
      pv[r] = x;
    }
  };

  // pass 1: sum_j of P and P Gam, and max_j P (this lane's keys); sum_j P dP and sum_j P (Gam dP + W) follow from
  // the G_dO products as dO . sum_j P V and dO . (sum_j (P o Gam) V + sum_j P gV)
  float l_part = 0.f, r_part = 0.f, p_max = 0.f;
  float rx = 0.f, tx = 0.f;  // r, t of the row after the exchange
  f32x16_t acc[NDT], accy[NDT];  // pass 2: sum_j Gbar_S K and sum_j dS gK (transposed, lane per query)

  // G_dO (the JVP of O along (gQ, gK, gV)) from pass 1, as the JVP kernel forms it with normalised P:
  // G_dO = (sum_j (P o Gam) V + sum_j P gV) / L - r (sum_j P V) / L (jvp_kernel's epilogue). The first two sums
  // share one accumulator (their products chain into it).
  f32x16_t acc_a[NDT], acc_o[NDT];  // sum_j (P o Gam) V + sum_j P gV, and sum_j P V (transposed)
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) acc_a[dt] = acc_o[dt] = zero16();

  // PASS 1: the row sums and the G_dO products over this group's keys (SPLIT: P o Gam and P as two 16-bit terms).
  auto compute_sums = [&](auto split_tag, auto mask_tag, int kt, const char* tK, const char* tV, const char* tgK,
                          const char* tgV) __attribute__((always_inline)) {
    constexpr bool SPLIT = decltype(split_tag)::value;
#pragma unroll
    for (int st = 0; st < NST; ++st) {
      const int k0s = kt * BN + 32 * st;
      if (CAUSAL && k0s > q0w + 31) continue;
      f32x16_t pv, gm, w, dpz;
      products(std::false_type{}, mask_tag, k0s, tK, tV, tgK, tgV, st, pv, gm, w, dpz);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float pg = pv[r] * (s.scale * gm[r]);  // P o Gam
        l_part += pv[r];
        r_part += pg;
        p_max = fmaxf(p_max, pv[r]);
        gm[r] = pg;
      }
#pragma unroll
      for (int cc = 0; cc < NPC; ++cc) {
        if constexpr (SPLIT) {
          F ph, pl, gh, gl;
          split_frag<T>(pv, cc, ph, pl);
          split_frag<T>(gm, cc, gh, gl);
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) {
            const F vr = swz_rows<T, DP>(tV, 32 * st, cc, dt * 32);
            acc_a[dt] = MM::mma(vr, gh, acc_a[dt]);
            acc_a[dt] = MM::mma(vr, gl, acc_a[dt]);
            if (has_gv) {
              const F gvr = swz_rows<T, DP>(tgV, 32 * st, cc, dt * 32);
              acc_a[dt] = MM::mma(gvr, ph, acc_a[dt]);
              acc_a[dt] = MM::mma(gvr, pl, acc_a[dt]);
            }
            acc_o[dt] = MM::mma(vr, ph, acc_o[dt]);
            acc_o[dt] = MM::mma(vr, pl, acc_o[dt]);
          }
        } else {
          const F pf = acc_frag<T>(pv, cc), gf = acc_frag<T>(gm, cc);
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) {
            const F vr = swz_rows<T, DP>(tV, 32 * st, cc, dt * 32);
            acc_a[dt] = MM::mma(vr, gf, acc_a[dt]);
            if (has_gv) acc_a[dt] = MM::mma(swz_rows<T, DP>(tgV, 32 * st, cc, dt * 32), pf, acc_a[dt]);
            acc_o[dt] = MM::mma(vr, pf, acc_o[dt]);
          }
        }
      }
    }
  };
  // PASS 2: Gbar_S and dS products (SPLIT: two 16-bit terms each).
  auto compute_exact = [&](auto split_tag, auto mask_tag, int kt, const char* tK, const char* tV, const char* tgK,
                           const char* tgV) __attribute__((always_inline)) {
    constexpr bool SPLIT = decltype(split_tag)::value;
#pragma unroll
    for (int st = 0; st < NST; ++st) {
      const int k0s = kt * BN + 32 * st;
      if (CAUSAL && k0s > q0w + 31) continue;
      f32x16_t pv, gm, w, dpz;
      products(std::true_type{}, mask_tag, k0s, tK, tV, tgK, tgV, st, pv, gm, w, dpz);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float gam = s.scale * gm[r];
        gm[r] = pv[r] * (fmaf(gam - rx, dpz[r], w[r]) - tx);  // Gbar_S
        dpz[r] = pv[r] * dpz[r];                              // dS
      }
#pragma unroll
      for (int cc = 0; cc < NPC; ++cc) {
        if constexpr (SPLIT) {
          F gh, gl, dh, dl;
          split_frag<T>(gm, cc, gh, gl);
          split_frag<T>(dpz, cc, dh, dl);
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) {
            const F kr = swz_rows<T, DP>(tK, 32 * st, cc, dt * 32);
            acc[dt] = MM::mma(kr, gh, acc[dt]);
            acc[dt] = MM::mma(kr, gl, acc[dt]);
            if (has_gk) {
              const F gkr = swz_rows<T, DP>(tgK, 32 * st, cc, dt * 32);
              accy[dt] = MM::mma(gkr, dh, accy[dt]);
              accy[dt] = MM::mma(gkr, dl, accy[dt]);
            }
          }
        } else {
          const F gf = acc_frag<T>(gm, cc), df = acc_frag<T>(dpz, cc);
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) {
            acc[dt] = MM::mma(swz_rows<T, DP>(tK, 32 * st, cc, dt * 32), gf, acc[dt]);
            if (has_gk) accy[dt] = MM::mma(swz_rows<T, DP>(tgK, 32 * st, cc, dt * 32), df, accy[dt]);
          }
        }
      }
    }
  };

  const Dma dma(JOINT ? wave : wig, lane, FD ? DP / 8 : s.D / 8);  // FD: head dim DP; else columns past D zero-filled
  // Byte offsets fit in 32 bits: the host only selects this kernel when each (batch, head) slab of K, V, gK and
  // gV spans less than 2^31 bytes.
  const uint32_t krs = (uint32_t)p.k.sr * 2, vrs = (uint32_t)p.v.sr * 2;
  const uint32_t gkrs = has_gk ? (uint32_t)p.gk.sr * 2 : 0u, gvrs = has_gv ? (uint32_t)p.gv.sr * 2 : 0u;
  const int64_t rb = 2 * (FD ? DP : s.D);  // bytes of a row the DMA reads
  const rsrc_t krsrc = make_rsrc(K, (uint32_t)slab_span(s.M, krs, rb)),
               vrsrc = make_rsrc(V, (uint32_t)slab_span(s.M, vrs, rb));
  const rsrc_t gkrsrc = make_rsrc(has_gk ? (const void*)GK : (const void*)K, (uint32_t)slab_span(s.M, gkrs, rb));
  const rsrc_t gvrsrc = make_rsrc(has_gv ? (const void*)GV : (const void*)V, (uint32_t)slab_span(s.M, gvrs, rb));
  auto tile_of = [&](int gg, int set, int a) { return smem + ((gg * 2 + set) * 4 + a) * TB; };  // a: K, V, gK, gV
  auto tile = [&](int set, int a) { return tile_of(grp, set, a); };
  auto issue_one = [&](int gg, int kt, int set) __attribute__((always_inline)) {
    const int k0 = kt * BN;
    dma.template issue_clamped<NSLAB>(krsrc, krs, k0, s.M, tile_of(gg, set, 0));
    dma.template issue_clamped<NSLAB>(vrsrc, vrs, k0, s.M, tile_of(gg, set, 1));
    if (has_gk) dma.template issue_clamped<NSLAB>(gkrsrc, gkrs, k0, s.M, tile_of(gg, set, 2));
    if (has_gv) dma.template issue_clamped<NSLAB>(gvrsrc, gvrs, k0, s.M, tile_of(gg, set, 3));
  };
  auto issue_joint = [&](int i) __attribute__((always_inline)) {  // step i's tiles of both groups
    if (i < half) issue_one(0, i, i & 1);
    if (i < half && half + i < nkt) issue_one(1, half + i, i & 1);
  };
  // Step i: tile kt0 + i of this group (if it has one) from set i & 1; the next one's copies go to the other set,
  // read in step i - 1, which every wave has finished at the barrier. Both groups run `half` steps (the same
  // barriers); a group with fewer tiles idles through its last one. The tiles from mask_from on may reach past
  // the last key or (causal) past the block's first query and take the masked copy of the loop; the groups may
  // be in different copies at a step, but both meet the same barriers.
  const int mask_from = min(kend % BN ? nkt - 1 : nkt, CAUSAL ? qb * BM / BN : nkt);
  auto sweep = [&](auto body) __attribute__((always_inline)) {
    auto step = [&](auto mask_tag, int i) __attribute__((always_inline)) {
      const int kt = kt0 + i;
      wait_vm_all();
      __syncthreads();
      if constexpr (JOINT)
        issue_joint(i + 1);
      else if (kt + 1 < kt1)
        issue_one(grp, kt + 1, (i + 1) & 1);
      if (kt < kt1) body(mask_tag, kt, tile(i & 1, 0), tile(i & 1, 1), tile(i & 1, 2), tile(i & 1, 3));
    };
    if constexpr (JOINT)
      issue_joint(0);
    else if (kt0 < kt1)
      issue_one(grp, kt0, 0);
    const int isplit = min(half, max(0, mask_from - kt0));
    int i = 0;
    for (; i < isplit; ++i) step(std::false_type{}, i);
    for (; i < half; ++i) step(std::true_type{}, i);
    __syncthreads();  // every wave is done with the tiles
  };
  float* buf = reinterpret_cast<float*>(smem);

  if (DP == 128 || split) {
    sweep([&](auto mask_tag, int kt, const char* a, const char* b_, const char* c, const char* d)
              __attribute__((always_inline)) { compute_sums(std::true_type{}, mask_tag, kt, a, b_, c, d); });
  } else {
    if constexpr (DP == 64)
      sweep([&](auto mask_tag, int kt, const char* a, const char* b_, const char* c, const char* d)
                __attribute__((always_inline)) { compute_sums(std::false_type{}, mask_tag, kt, a, b_, c, d); });
  }
  // dO . sum_j P V and dO . (sum_j (P o Gam) V + sum_j P gV) over this lane's columns of the accumulators
  float a_dot = 0.f, uw_dot = 0.f;
  if (qvalid) {
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const f32x4_t d4 = load4<T>(dO, p.dout.sr, myq, dt * 32 + 8 * qd + 4 * g, s.D, s.vec);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          a_dot = fmaf(d4[e], acc_o[dt][4 * qd + e], a_dot);
          uw_dot = fmaf(d4[e], acc_a[dt][4 * qd + e], uw_dot);
        }
      }
  }
  // the sums of the row: both lane halves of a query, then both key groups; group 1's G_dO accumulators to group 0
  // (sums at [0, 2560) floats, accumulator element e of lane l of wave w at 4096 + e * GT + w * 64 + l):
  // sum_j P, sum_j P dP, sum_j P Gam, sum_j P (Gam dP + W), max_j P
  float sums[5] = {pair_sum(l_part), pair_sum(a_dot), pair_sum(r_part), pair_sum(uw_dot), pair_max(p_max)};
#pragma unroll
  for (int i = 0; i < 5; ++i) buf[(i * 2 * NW + grp * NW + wig) * 64 + lane] = sums[i];
  if (grp == 1) {
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        buf[4096 + ((0 * NDT + dt) * 16 + r) * GT + wig * 64 + lane] = acc_a[dt][r];
        buf[4096 + ((1 * NDT + dt) * 16 + r) * GT + wig * 64 + lane] = acc_o[dt][r];
      }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) sums[i] += buf[(i * 2 * NW + (1 - grp) * NW + wig) * 64 + lane];
  sums[4] = fmaxf(sums[4], buf[(4 * 2 * NW + (1 - grp) * NW + wig) * 64 + lane]);
  const float L = sums[0];
  if (grp == 0 && qvalid) {
    // G_dO = inv (A + C) - (r inv) (O inv) with the normalised P (inv = 1 / L)
    const float inv = L > 0.f ? 1.f / L : 0.f;
    const float cval = sums[2] * inv;
    T* OD = (T*)p.out_gdo.p + b * p.out_gdo.sb + h * p.out_gdo.sh;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const int d0 = dt * 32 + 8 * qd + 4 * g;
        float r4[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = 4 * qd + e;
          const float a = acc_a[dt][i] + buf[4096 + ((0 * NDT + dt) * 16 + i) * GT + wig * 64 + lane];
          const float o = acc_o[dt][i] + buf[4096 + ((1 * NDT + dt) * 16 + i) * GT + wig * 64 + lane];
          r4[e] = inv * a - cval * (o * inv);
        }
        store4<T>(OD, p.out_gdo.sr, myq, d0, s.D, r4[0], r4[1], r4[2], r4[3], s.vec);
      }
  }
  __syncthreads();  // the exchange is read before the tiles are refilled
  float lse_c = lse_raw;
  if (L > 0.f) {
    const float inv = 1.f / L;
    z = sums[1] * inv;
    rx = sums[2] * inv;
    tx = (sums[3] - z * sums[2]) * inv;
    moff += __builtin_log2f(L);
    lse_c = lse_with_flag(lse_raw + __builtin_log2f(L) * kLn2, sums[4] > kPeakedFrac * L);
  }
  if (grp == 0 && qvalid && g == 0) {
    p.r_row[row_id] = rx;
    p.t_row[row_id] = tx;
    p.z_out[row_id] = z;
    p.lse_out[row_id] = lse_c;
  }
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) acc[dt] = accy[dt] = zero16();
  if (DP == 128 || split) {
    sweep([&](auto mask_tag, int kt, const char* a, const char* b_, const char* c, const char* d)
              __attribute__((always_inline)) { compute_exact(std::true_type{}, mask_tag, kt, a, b_, c, d); });
  } else {
    if constexpr (DP == 64)
      sweep([&](auto mask_tag, int kt, const char* a, const char* b_, const char* c, const char* d)
                __attribute__((always_inline)) { compute_exact(std::false_type{}, mask_tag, kt, a, b_, c, d); });
  }

  // group 1's accumulators to group 0 (element e of lane l of wave w at e * GT + w * 64 + l)
  if (grp == 1) {
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        buf[(dt * 16 + r) * GT + wig * 64 + lane] = acc[dt][r];
        buf[((NDT + dt) * 16 + r) * GT + wig * 64 + lane] = accy[dt][r];
      }
  }
  __syncthreads();
  if (grp == 1) return;
  if (qvalid) {
    T* OG = (T*)p.out_gq.p + b * p.out_gq.sb + h * p.out_gq.sh;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const int d0 = dt * 32 + 8 * qd + 4 * g;
        float r4[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = 4 * qd + e;
          const float x = acc[dt][i] + buf[(dt * 16 + i) * GT + wig * 64 + lane];
          const float y = accy[dt][i] + buf[((NDT + dt) * 16 + i) * GT + wig * 64 + lane];
          r4[e] = s.scale * (x + y);
        }
        store4<T>(OG, p.out_gq.sr, myq, d0, s.D, r4[0], r4[1], r4[2], r4[3], s.vec);
      }
  }
}


// The column pass for 16-bit inputs with LDS-DMA tiles (DP and FD as in the row pass), as two query groups: at DP = 64
// of four waves (eight-wave workgroups, two waves per SIMD), at 128 of two. A workgroup owns 128 (64) keys (32 per wave,
// lane per key, as in cols_block); the groups sweep the two halves of its 32-query tiles and sum G_V and G_K in
// registers, and group 1's sums reach group 0 through LDS at the end. Query tiles holding a row flagged peaked in lse are
// skipped by the sweep and run after it, shared out between the groups, with Gbar_dP, Gbar_S and dS entered as
// two 16-bit terms. The gK and gV fragments sit in LDS, so that the K and V fragments, the two accumulators and
// the products fit 256 registers (512 at DP = 128). ALL as in the key-split row kernel.
template <typename T, bool CAUSAL, bool ALL, bool FD, int DP>
__global__ __launch_bounds__(DP == 64 ? 512 : 256, DP == 64 ? 2 : 1) void bwdbwd_cols_qs_kernel(const BwdBwdParams p) {
  using MM = Mfma<T>;
  using F = typename MM::frag_t;
  static_assert(sizeof(T) == 2, "16-bit inputs only");
  constexpr int NW = DP == 64 ? 4 : 2, GT = 64 * NW, NT = 2 * GT, BN = 32 * NW, BM = 32;
  constexpr int NDT = DP / 32, NKC = DP / MM::KC, NPC = 32 / MM::KC;
  constexpr int TB = BM * DP * 2;  // bytes per tile
  constexpr bool JOINT = DP == 128;  // as in the row kernel
  using Dma = SwzDma<4, DP>;
  constexpr int NSLAB = BM / Dma::SLAB_ROWS;
  static_assert(NSLAB * Dma::SLAB_ROWS == BM, "query tiles must be whole DMA slabs");
  constexpr int FLAG = 4 * BM, RB = FLAG + 4;  // row terms [lse * log2(e) | z | r | t] of a tile, then its flag
  constexpr int TILES = 2 * 2 * 3 * TB;        // [group][set][Q, dO, gQ]
  constexpr int NFR = NW * NKC * 64;           // fragments per operand
  // the tiles, then the gK and gV fragments (fragment c of lane l of key slice w at (w * NKC + c) * 64 + l);
  // group 1's accumulators reach group 0 through the same memory at the end
  __shared__ __attribute__((aligned(1024))) char smem[TILES + 2 * NFR * sizeof(F)];
  static_assert(sizeof(smem) >= 2 * NDT * 16 * GT * sizeof(float), "the exchange fits in the tile memory");
  __shared__ __attribute__((aligned(16))) float sRow[2][2][RB];  // [group][set]
  __shared__ int sPk[64];
  __shared__ int sAny;

  const Shape& s = p.s;
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = (unsigned)wave / NW, wig = (unsigned)wave % NW;  // query group, wave in group
  const int ltid = tid % GT;                   // thread in group
  const int nkb = (s.M + BN - 1) / BN;
  const int bid = xcd_remap(blockIdx.x, gridDim.x);
  const int bh = bid / nkb;
  const int kb = bid - bh * nkb;
  const int b = bh / s.H, h = bh - b * s.H;
  const T* Q = (const T*)p.q.p + b * p.q.sb + h * p.q.sh;
  const T* K = (const T*)p.k.p + b * p.k.sb + h * p.k.sh;
  const T* V = (const T*)p.v.p + b * p.v.sb + h * p.v.sh;
  const T* dO = (const T*)p.dout.p + b * p.dout.sb + h * p.dout.sh;
  const bool has_gq = ALL || p.gq.p != nullptr, has_gk = ALL || p.gk.p != nullptr, has_gv = ALL || p.gv.p != nullptr;
  const T* GQ = has_gq ? (const T*)p.gq.p + b * p.gq.sb + h * p.gq.sh : nullptr;
  const T* GK = has_gk ? (const T*)p.gk.p + b * p.gk.sb + h * p.gk.sh : nullptr;
  const T* GV = has_gv ? (const T*)p.gv.p + b * p.gv.sb + h * p.gv.sh : nullptr;
  const int key0 = kb * BN;
  const int kw0 = key0 + wig * 32;
  const int mykey = kw0 + li;
  const bool kvalid = mykey < s.M;

  F* sFr = reinterpret_cast<F*>(smem + TILES);
  F kf[NKC], vf[NKC];
#pragma unroll
  for (int c = 0; c < NKC; ++c) {
    kf[c] = gload_frag<T>(K, p.k.sr, mykey, s.M, c, s.D, s.vec);
    vf[c] = gload_frag<T>(V, p.v.sr, mykey, s.M, c, s.D, s.vec);
    // read after the sweep's first barrier
    if (grp == 0) {
      if (has_gk) sFr[(wig * NKC + c) * 64 + lane] = gload_frag<T>(GK, p.gk.sr, mykey, s.M, c, s.D, s.vec);
      if (has_gv) sFr[NFR + (wig * NKC + c) * 64 + lane] = gload_frag<T>(GV, p.gv.sr, mykey, s.M, c, s.D, s.vec);
    }
  }
  if (tid == 0) sAny = 0;
  f32x16_t accV[NDT], accK[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) accV[dt] = accK[dt] = zero16();
  const float c2 = s.scale * kLog2e;
  const int qbeg = CAUSAL ? (key0 / BM) * BM : 0;
  const int nqt = s.T > qbeg ? (s.T - qbeg + BM - 1) / BM : 0;
  const int half = (nqt + 1) / 2;
  const int it0 = grp * half, it1 = min(nqt, it0 + half);  // this group's tiles [it0, it1) of the sweep
  const int64_t rowbase = (int64_t)bh * s.T;

  // Row terms of a tile for group thread ltid < BM, held raw (rows past the end: lse = +inf) and converted when
  // stored: lse * log2(e) (+inf for rows past the end or without visible keys, so P = 0), z, r, t.
  float r_lse = THERIA_INF, r_z = 0.f, r_r = 0.f, r_t = 0.f;
  auto load_rows = [&](int it, int lim) {
    if (ltid < BM && it < lim) {
      const int qq = qbeg + it * BM + ltid;
      const bool ok = qq < s.T;
      r_lse = ok ? p.lse[rowbase + qq] : THERIA_INF;
      r_z = ok ? p.delta[rowbase + qq] : 0.f;
      r_r = ok ? p.r_row[rowbase + qq] : 0.f;
      r_t = ok ? p.t_row[rowbase + qq] : 0.f;
    }
  };
  auto store_rows = [&](float* sr) {
    if (ltid < BM) {
      sr[ltid] = __builtin_isinf(r_lse) ? THERIA_INF : r_lse * kLog2e;
      sr[BM + ltid] = r_z;
      sr[2 * BM + ltid] = r_r;
      sr[3 * BM + ltid] = r_t;
      const bool pk = __any(lse_peaked(r_lse));  // the tile's rows are the lanes of the group's first wave
      if (ltid == 0) sr[FLAG] = pk ? 1.f : 0.f;
    }
  };

  // Query tile it held in (tQ, tO, tgQ) with its row terms in sr. SPLIT: Gbar_dP, Gbar_S and dS enter the
  // products as two 16-bit terms each.
  auto tile = [&](auto split_tag, int it, const char* tQ, const char* tO, const char* tgQ,
                  const float* sr) __attribute__((always_inline)) {
    constexpr bool SPLIT = decltype(split_tag)::value;
    const int q0 = qbeg + it * BM;
    if (CAUSAL && kw0 > q0 + BM - 1) return;
    f32x16_t sc = zero16(), gm = zero16(), w = zero16(), dpz;
#pragma unroll
    for (int qd = 0; qd < 4; ++qd) {
      const f32x4_t z4 = *reinterpret_cast<const f32x4_t*>(sr + BM + 8 * qd + 4 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) dpz[4 * qd + e] = -z4[e];
    }
#pragma unroll
    for (int c = 0; c < NKC; ++c) {
      const F qfr = swz_cols<T, DP>(tQ, li, c);
      const F ofr = swz_cols<T, DP>(tO, li, c);
      sc = MM::mma(qfr, kf[c], sc);
      dpz = MM::mma(ofr, vf[c], dpz);
      if (has_gq) gm = MM::mma(swz_cols<T, DP>(tgQ, li, c), kf[c], gm);
      if (has_gk) gm = MM::mma(qfr, sFr[(wig * NKC + c) * 64 + lane], gm);
      if (has_gv) w = MM::mma(ofr, sFr[NFR + (wig * NKC + c) * 64 + lane], w);
    }
    const bool diag = CAUSAL && (kw0 + 31 > q0);
#pragma unroll
    for (int qd = 0; qd < 4; ++qd) {
      const int o = 8 * qd + 4 * g;
      const f32x4_t l4 = *reinterpret_cast<const f32x4_t*>(sr + o);
      const f32x4_t r4 = *reinterpret_cast<const f32x4_t*>(sr + 2 * BM + o);
      const f32x4_t t4 = *reinterpret_cast<const f32x4_t*>(sr + 3 * BM + o);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 4 * qd + e;
        float pv = fast_exp2(fmaf(sc[r], c2, -l4[e]));
        if (!kvalid) pv = 0.f;
        if (diag && mykey > q0 + acc_row(r, g)) pv = 0.f;
        const float gam = s.scale * gm[r];
        const float ds = pv * dpz[r];
        const float e1 = fmaf(gam, dpz[r], w[r]);
        gm[r] = pv * (gam - r4[e]);                        // Gbar_dP
        w[r] = pv * e1 - r4[e] * ds - t4[e] * pv;          // Gbar_S
        dpz[r] = ds;                                       // dS
      }
    }
#pragma unroll
    for (int cc = 0; cc < NPC; ++cc) {
      if constexpr (SPLIT) {
        F gdph, gdpl, gsh, gsl, dsh, dsl;
        split_frag<T>(gm, cc, gdph, gdpl);
        split_frag<T>(w, cc, gsh, gsl);
        split_frag<T>(dpz, cc, dsh, dsl);
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
          const F ro = swz_rows<T, DP>(tO, 0, cc, dt * 32);
          accV[dt] = MM::mma(gdph, ro, accV[dt]);
          accV[dt] = MM::mma(gdpl, ro, accV[dt]);
          const F rq = swz_rows<T, DP>(tQ, 0, cc, dt * 32);
          accK[dt] = MM::mma(gsh, rq, accK[dt]);
          accK[dt] = MM::mma(gsl, rq, accK[dt]);
          if (has_gq) {
            const F rg = swz_rows<T, DP>(tgQ, 0, cc, dt * 32);
            accK[dt] = MM::mma(dsh, rg, accK[dt]);
            accK[dt] = MM::mma(dsl, rg, accK[dt]);
          }
        }
      } else {
        const F gdpf = acc_frag<T>(gm, cc), gsf = acc_frag<T>(w, cc), dsf = acc_frag<T>(dpz, cc);
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
          accV[dt] = MM::mma(gdpf, swz_rows<T, DP>(tO, 0, cc, dt * 32), accV[dt]);
          accK[dt] = MM::mma(gsf, swz_rows<T, DP>(tQ, 0, cc, dt * 32), accK[dt]);
          if (has_gq) accK[dt] = MM::mma(dsf, swz_rows<T, DP>(tgQ, 0, cc, dt * 32), accK[dt]);
        }
      }
    }
  };

  const Dma dma(JOINT ? wave : wig, lane, FD ? DP / 8 : s.D / 8);  // FD: head dim DP; else columns past D zero-filled
  // Byte offsets fit in 32 bits: the host only selects this kernel when each (batch, head) slab of Q, dO and gQ
  // spans less than 2^31 bytes.
  const uint32_t qrs = (uint32_t)p.q.sr * 2, ors = (uint32_t)p.dout.sr * 2;
  const uint32_t gqrs = has_gq ? (uint32_t)p.gq.sr * 2 : 0u;
  const int64_t rb = 2 * (FD ? DP : s.D);  // bytes of a row the DMA reads
  const rsrc_t qrsrc = make_rsrc(Q, (uint32_t)slab_span(s.T, qrs, rb)),
               orsrc = make_rsrc(dO, (uint32_t)slab_span(s.T, ors, rb));
  const rsrc_t gqrsrc = make_rsrc(has_gq ? (const void*)GQ : (const void*)Q, (uint32_t)slab_span(s.T, gqrs, rb));
  auto tiles_of = [&](int gg, int set) { return smem + (gg * 2 + set) * 3 * TB; };  // Q, dO, gQ at 0, TB, 2 TB
  auto tiles = [&](int set) { return tiles_of(grp, set); };
  auto issue_one = [&](int gg, int it, int set) __attribute__((always_inline)) {
    const int q0 = qbeg + it * BM;
    char* t = tiles_of(gg, set);
    dma.template issue_clamped<NSLAB>(qrsrc, qrs, q0, s.T, t);
    dma.template issue_clamped<NSLAB>(orsrc, ors, q0, s.T, t + TB);
    if (has_gq) dma.template issue_clamped<NSLAB>(gqrsrc, gqrs, q0, s.T, t + 2 * TB);
  };
  auto issue_joint = [&](int i) __attribute__((always_inline)) {  // step i's tiles of both groups
    if (i < half) issue_one(0, i, i & 1);
    if (i < half && half + i < nqt) issue_one(1, half + i, i & 1);
  };

  // The sweep. Step i: tile it0 + i of this group (if it has one) from set i & 1; the next one's copies and row
  // terms go to the other set, read in step i - 1, which every wave has finished at the barrier. Both groups run
  // `half` steps (the same barriers); a group with fewer tiles idles through its last one.
  bool pk_any = false;  // a tile holding a peaked row was skipped
  if constexpr (JOINT) issue_joint(0);
  if (it0 < it1) {
    if constexpr (!JOINT) issue_one(grp, it0, 0);
    load_rows(it0, it1);
    store_rows(sRow[grp][0]);
    load_rows(it0 + 1, it1);
  }
  for (int i = 0; i < half; ++i) {
    const int it = it0 + i;
    wait_vm_all();
    __syncthreads();
    if constexpr (JOINT) issue_joint(i + 1);
    if (it + 1 < it1) {
      if constexpr (!JOINT) issue_one(grp, it + 1, (i + 1) & 1);
      store_rows(sRow[grp][(i + 1) & 1]);
      load_rows(it + 2, it1);
    }
    if (it < it1) {
      const float* sr = sRow[grp][i & 1];
      const bool pk = __builtin_amdgcn_readfirstlane(__float_as_uint(sr[FLAG])) != 0u;  // uniform
      pk_any |= pk;
      const char* t = tiles(i & 1);
      if (!pk) tile(std::false_type{}, it, t, t + TB, t + 2 * TB, sr);
    }
  }
  if (pk_any && lane == 0) sAny = 1;
  __syncthreads();  // every wave is done with the tiles; sAny is final

  // The tiles holding a peaked row, found 64 at a time from the lse flags; the groups take alternate ones.
  if (sAny) {
    for (int t0 = 0; t0 < nqt; t0 += 64) {
      const int nt = min(64, nqt - t0);
      __syncthreads();  // every thread is done with the previous flags and tiles
      if (tid < 64) sPk[tid] = 0;
      __syncthreads();
      constexpr int RPT = 64 * BM / NT;
      const int r0 = qbeg + t0 * BM, r1 = min(s.T, qbeg + (t0 + nt) * BM);
#pragma unroll
      for (int j = 0; j < RPT; ++j) {
        const int r = r0 + tid + NT * j;
        if (r < r1 && lse_peaked(p.lse[rowbase + r])) sPk[(tid + NT * j) / BM] = 1;
      }
      __syncthreads();
      const uint64_t mask = __ballot(sPk[lane] != 0);  // the same in every wave
      const int npk = __builtin_popcountll(mask);
      for (int j = 0; j < npk; j += 2) {
        // group x's tile: the (j + x)-th flagged one (-1: none)
        auto flagged = [&](int x) {
          if (j + x >= npk) return -1;
          uint64_t m = mask;
          for (int y = 0; y < j + x; ++y) m &= m - 1;
          return t0 + __builtin_ctzll(m);
        };
        const int ti = flagged(grp);
        __syncthreads();  // the tile buffers are free
        if constexpr (JOINT) {
          const int other = flagged(1 - grp);
          if (ti >= 0) issue_one(grp, ti, 0);
          if (other >= 0) issue_one(1 - grp, other, 0);
        } else if (ti >= 0) {
          issue_one(grp, ti, 0);
        }
        if (ti >= 0) {
          load_rows(ti, nqt);
          store_rows(sRow[grp][0]);
        }
        wait_vm_all();
        __syncthreads();
        if (ti >= 0) {
          const char* t = tiles(0);
          tile(std::true_type{}, ti, t, t + TB, t + 2 * TB, sRow[grp][0]);
        }
      }
    }
    __syncthreads();  // every wave is done with the tiles
  }

  // The groups finish NH column tiles each (group g the tiles g NH ..): each hands the other's G_V and G_K partial sums to
  // the other group (element e of accumulator a (V, K) of tile j of lane l of wave w of group g at
  // (((g * NH + j) * 2 + a) * 16 + e) * GT + w * 64 + l), then stores its part of the columns.
  constexpr int NH = NDT / 2;
  float* xb = reinterpret_cast<float*>(smem);
  T* OV = (T*)p.out_gv.p + b * p.out_gv.sb + h * p.out_gv.sh;
  T* OK = (T*)p.out_gk.p + b * p.out_gk.sb + h * p.out_gk.sh;
  auto finish = [&](auto keep_tag) __attribute__((always_inline)) {
    constexpr int KEEP = decltype(keep_tag)::value, GIVE = 1 - KEEP;
#pragma unroll
    for (int j = 0; j < NH; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        xb[(((KEEP * NH + j) * 2 + 0) * 16 + r) * GT + wig * 64 + lane] = accV[GIVE * NH + j][r];
        xb[(((KEEP * NH + j) * 2 + 1) * 16 + r) * GT + wig * 64 + lane] = accK[GIVE * NH + j][r];
      }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NH; ++j) {
      const int dt = KEEP * NH + j, d = dt * 32 + li;
      if (d < s.D) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = kw0 + acc_row(r, g);
          if (key < s.M) {
            const float v = accV[dt][r] + xb[(((GIVE * NH + j) * 2 + 0) * 16 + r) * GT + wig * 64 + lane];
            const float k = accK[dt][r] + xb[(((GIVE * NH + j) * 2 + 1) * 16 + r) * GT + wig * 64 + lane];
            OV[(int64_t)key * p.out_gv.sr + d] = (T)v;
            OK[(int64_t)key * p.out_gk.sr + d] = (T)(k * s.scale);
          }
        }
      }
    }
  };
  // both branches meet the one barrier inside finish
  if (grp == 0)
    finish(std::integral_constant<int, 0>{});
  else
    finish(std::integral_constant<int, 1>{});
}

template <typename T, bool CAUSAL, int DP>
static void rows_ks_go(const BwdBwdParams& p, hipStream_t st) {
  constexpr int BM = DP == 64 ? 128 : 64;
  const bool all = p.gq.p && p.gk.p && p.gv.p, fd = p.s.D == DP;
  const dim3 grid((unsigned)((int64_t)((p.s.T + BM - 1) / BM) * p.s.B * p.s.H)), block(4 * BM);
  if (grid.x == 0) return;
  if (all && fd)
    hipLaunchKernelGGL((bwdbwd_rows_ks_kernel<T, CAUSAL, true, true, DP>), grid, block, 0, st, p);
  else if (all)
    hipLaunchKernelGGL((bwdbwd_rows_ks_kernel<T, CAUSAL, true, false, DP>), grid, block, 0, st, p);
  else if (fd)
    hipLaunchKernelGGL((bwdbwd_rows_ks_kernel<T, CAUSAL, false, true, DP>), grid, block, 0, st, p);
  else
    hipLaunchKernelGGL((bwdbwd_rows_ks_kernel<T, CAUSAL, false, false, DP>), grid, block, 0, st, p);
}
template <typename T, bool CAUSAL, int DP>
static void cols_qs_go(const BwdBwdParams& p, hipStream_t st) {
  constexpr int BN = DP == 64 ? 128 : 64;
  const bool all = p.gq.p && p.gk.p && p.gv.p, fd = p.s.D == DP;
  const dim3 grid((unsigned)((int64_t)((p.s.M + BN - 1) / BN) * p.s.B * p.s.H)), block(4 * BN);
  if (grid.x == 0) return;
  if (all && fd)
    hipLaunchKernelGGL((bwdbwd_cols_qs_kernel<T, CAUSAL, true, true, DP>), grid, block, 0, st, p);
  else if (all)
    hipLaunchKernelGGL((bwdbwd_cols_qs_kernel<T, CAUSAL, true, false, DP>), grid, block, 0, st, p);
  else if (fd)
    hipLaunchKernelGGL((bwdbwd_cols_qs_kernel<T, CAUSAL, false, true, DP>), grid, block, 0, st, p);
  else
    hipLaunchKernelGGL((bwdbwd_cols_qs_kernel<T, CAUSAL, false, false, DP>), grid, block, 0, st, p);
}

template <typename T, bool CAUSAL>
hipError_t launch_rows_ks(const BwdBwdParams& p, hipStream_t st) {
  if (p.s.dp <= 64)
    rows_ks_go<T, CAUSAL, 64>(p, st);
  else
    rows_ks_go<T, CAUSAL, 128>(p, st);
  return hipGetLastError();
}
template <typename T, bool CAUSAL>
hipError_t launch_cols_qs(const BwdBwdParams& p, hipStream_t st) {
  if (p.s.dp <= 64)
    cols_qs_go<T, CAUSAL, 64>(p, st);
  else
    cols_qs_go<T, CAUSAL, 128>(p, st);
  return hipGetLastError();
}

template bool rows_ks_ok<__bf16>(const BwdBwdParams&);
template bool rows_ks_ok<_Float16>(const BwdBwdParams&);
template bool cols_qs_ok<__bf16>(const BwdBwdParams&);
template bool cols_qs_ok<_Float16>(const BwdBwdParams&);
template hipError_t launch_rows_ks<__bf16, false>(const BwdBwdParams&, hipStream_t);
template hipError_t launch_rows_ks<__bf16, true>(const BwdBwdParams&, hipStream_t);
template hipError_t launch_rows_ks<_Float16, false>(const BwdBwdParams&, hipStream_t);
template hipError_t launch_rows_ks<_Float16, true>(const BwdBwdParams&, hipStream_t);
template hipError_t launch_cols_qs<__bf16, false>(const BwdBwdParams&, hipStream_t);
template hipError_t launch_cols_qs<__bf16, true>(const BwdBwdParams&, hipStream_t);
template hipError_t launch_cols_qs<_Float16, false>(const BwdBwdParams&, hipStream_t);
template hipError_t launch_cols_qs<_Float16, true>(const BwdBwdParams&, hipStream_t);

}  // namespace theria
