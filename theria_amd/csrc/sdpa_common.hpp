// Shared device building blocks for the gfx950 SDPA kernels.
//
// Tiling vocabulary used by every kernel:
//  * All matrix products use 32x32 MFMA output tiles. For 16-bit inputs the instruction is
//    v_mfma_f32_32x32x16_{bf16,f16} (k extent 16, 8 elements per lane); float32 inputs take six
//    v_mfma_f32_32x32x16_bf16 over operands split into three bfloat16 terms (MfmaX3 below). Accumulation is float32
//    in all.
//  * Operand fragment of lane l (li = l % 32, g = l / 32): the row (A) or column (B) index is li, and
//    the k elements depend on g. Output ("accumulator") layout: register r of lane l holds the element
//    at row acc_row(r, g) = 8*(r/4) + 4*g + r%4 and column li. These layouts were checked bit-exactly
//    on the MI355X against a host matrix product.
//  * Because the k reduction is order-free, the k elements of a fragment may follow any mapping as long
//    as both operands use the same one. Two mappings are used:
//      KLIN: element e of chunk c sits at k = c*KC + g*EPL + e (contiguous per lane);
//      KACC: element e of chunk c sits at k = acc_row(c*EPL + e, g) (k inside a 32-row block), which is
//            exactly how an accumulator tile's registers are laid out. An accumulator tile can then be
//            fed straight back as an operand (P, dS, ...) whose k index is the tile's row index.
//  * Row-major LDS tiles are read two ways: "cols" fragments (k runs along a row, lane-fixed row) with
//    ds_read_b128 / ds_read_b64, and "rows" fragments (k runs down a column, lane-fixed column) with the
//    gfx950 transpose read ds_read_b64_tr_b16. Its semantics, measured on the device: within each group
//    of 16 lanes, result lane j element e = 16-bit element (j % 4) of the 8 bytes addressed by source
//    lane 4*e + j/4. Giving source lane s the address of row (k0 + s/4), column (c0 + 4*(s%4)) therefore
//    hands lane j the column c0 + j for rows k0..k0+3. No transposed copies are kept in LDS.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace theria {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4_t __attribute__((ext_vector_type(4)));
typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef short i16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
#define THERIA_INF (__builtin_inff())

enum KOrder { KLIN = 0, KACC = 1 };

__device__ __forceinline__ int acc_row(int r, int g) { return 8 * (r >> 2) + 4 * g + (r & 3); }

// ----------------------------------------------------------------------------------------------
// MFMA traits
// ----------------------------------------------------------------------------------------------
template <typename T> struct Mfma;

template <> struct Mfma<__bf16> {
  using frag_t = bf16x8_t;
  static constexpr int KC = 16;
  static constexpr int EPL = 8;
  __device__ __forceinline__ static f32x16_t mma(frag_t a, frag_t b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};

template <> struct Mfma<_Float16> {
  using frag_t = f16x8_t;
  static constexpr int KC = 16;
  static constexpr int EPL = 8;
  __device__ __forceinline__ static f32x16_t mma(frag_t a, frag_t b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

// float32 products on the bfloat16 matrix pipe. Each operand is split into three bfloat16 terms, h = bf16(x),
// m = bf16(x - h), l = bf16(x - h - m), which hold all 24 bits of it (rounding to nearest leaves |m| <= 2^-8 |x|
// and |l| <= 2^-17 |x|), and a b is summed as the six products down to 2^-16: the three dropped ones (m l, l m,
// l l) are at most 2^-24 of it and 2^-27 on average, under float32's own rounding. One 16-wide k chunk then takes 6 x 32 cycles of the
// matrix pipe where eight v_mfma_f32_32x32x2_f32 take 8 x 64, and rounds the accumulator fewer times.
// Every float32 kernel forms its products this way and in this order: the kernels of one call rebuild each other's
// scores and probabilities (lse, the row statistics of the double backward), and differences of values rounded two
// ways do not cancel (row statistics from v_mfma_f32_32x32x2_f32 beside split products here: G_Q of a peaked D96 problem
// off by 2.0e-4 where float32 PyTorch is off by 4.9e-5). Ops below is the one place that chooses the product.
// Measured against v_mfma_f32_32x32x2_f32 throughout: forward + backward of B2 H16 T1000 D64 461 -> 281 us, the HVP of
// B8 H8 T512 D64 786 -> 504 us, of B4 H8 T700 D128 3724 -> 1666 us; relative error against float64 7.4e-7 -> 6.4e-7,
// 7.4e-7 -> 6.2e-7 and 8.8e-7 -> 7.5e-7, and not larger in any of eight second-order calls at D 72..128.
struct X3Frag {
  bf16x8_t h, m, l;
};
struct MfmaX3 {
  using frag_t = X3Frag;
  static constexpr int KC = 16;
  static constexpr int EPL = 8;
  // Smallest products first. SW: the roles of a and b exchanged in that order, so that a product formed with its
  // operands swapped (S and S^T) rounds identically.
  template <bool SW = false>
  __device__ __forceinline__ static f32x16_t mma(const frag_t& a, const frag_t& b, f32x16_t c) {
    using M = Mfma<__bf16>;
    c = M::mma(a.m, b.m, c);
    c = SW ? M::mma(a.h, b.l, c) : M::mma(a.l, b.h, c);
    c = SW ? M::mma(a.l, b.h, c) : M::mma(a.h, b.l, c);
    c = SW ? M::mma(a.h, b.m, c) : M::mma(a.m, b.h, c);
    c = SW ? M::mma(a.m, b.h, c) : M::mma(a.h, b.m, c);
    return M::mma(a.h, b.h, c);
  }
};

template <typename T> __device__ __forceinline__ T to_t(float x) { return (T)x; }

__device__ __forceinline__ f32x16_t zero16() {
  f32x16_t z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.f;
  return z;
}

// Lane l and lane l^32 combined (both halves receive the result).
__device__ __forceinline__ float pair_max(float x) {
  auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(w[0]), __uint_as_float(w[1]));
}
__device__ __forceinline__ float pair_sum(float x) {
  auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(w[0]) + __uint_as_float(w[1]);
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// a * b rounded once and never fused into a following add: the float32 kernels form x = fl(S c) - m2 from
// the same fl(S c) that the row max m2 was taken over, so the row's largest score gives x = 0 exactly.
__device__ __forceinline__ float mul_rn(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}

// float32 probability from the row's own statistics (kRowOwnStats): exp2((fl(S c) - m2) - L2). m2 = +inf
// (a row without visible keys, or past the end) gives 0.
__device__ __forceinline__ float own_prob(float s_raw, float c2, float m2, float l2) {
  return fast_exp2((mul_rn(s_raw, c2) - m2) - l2);
}

// Peaked rows. With 16-bit inputs the lowest mantissa bit of each lse the forward writes marks a row whose
// largest probability may exceed 1/4 (kPeakedFrac); the backward kernels read it to take their exact path
// there (two-term 16-bit operands, the row term from a pass over the keys). Setting the bit moves lse by at
// most one unit in the last place. Infinite lse (rows without visible keys) carries no flag.
constexpr float kPeakedFrac = 0.25f;
__device__ __forceinline__ float lse_with_flag(float lse, bool peaked) {
  if (!__builtin_isfinite(lse)) return lse;
  return __uint_as_float((__float_as_uint(lse) & ~1u) | (peaked ? 1u : 0u));
}
__device__ __forceinline__ bool lse_peaked(float lse) {
  return __builtin_isfinite(lse) && (__float_as_uint(lse) & 1u);
}

// ----------------------------------------------------------------------------------------------
// k-index mapping of fragment element 0 / element EPL/2. c is the chunk index (KC wide), g the lane half.
// ----------------------------------------------------------------------------------------------
template <int ORDER> __device__ __forceinline__ int k16_first(int c, int g) {
  return ORDER == KLIN ? c * 16 + 8 * g : c * 16 + 4 * g;
}
template <int ORDER> __device__ __forceinline__ int k16_second(int c, int g) {
  return ORDER == KLIN ? c * 16 + 8 * g + 4 : c * 16 + 4 * g + 8;
}

// ----------------------------------------------------------------------------------------------
// LDS fragment reads
// ----------------------------------------------------------------------------------------------
// "cols" fragment: lane-fixed row `row`, k along the row starting at column kbase.
template <typename T, int ORDER>
__device__ __forceinline__ typename Mfma<T>::frag_t lds_cols(const T* base, int pitch, int row, int kbase, int c) {
  const int g = (threadIdx.x >> 5) & 1;
  using F = typename Mfma<T>::frag_t;
  const T* p0 = base + row * pitch + kbase + k16_first<ORDER>(c, g);
  if constexpr (ORDER == KLIN) {
    return __builtin_bit_cast(F, *reinterpret_cast<const i16x8_t*>(p0));
  } else {
    const T* p1 = base + row * pitch + kbase + k16_second<ORDER>(c, g);
    i16x4_t a = *reinterpret_cast<const i16x4_t*>(p0);
    i16x4_t b = *reinterpret_cast<const i16x4_t*>(p1);
    i16x8_t v = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    return __builtin_bit_cast(F, v);
  }
}

typedef __attribute__((address_space(3))) i16x4_t lds_i16x4_t;

__device__ __forceinline__ i16x4_t ds_read_tr16(const void* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t*)(p));
}

// "rows" fragment: lane-fixed column col0 + li, k down the column starting at row kbase.
template <typename T, int ORDER>
__device__ __forceinline__ typename Mfma<T>::frag_t lds_rows(const T* base, int pitch, int kbase, int c, int col0) {
  const int lane = threadIdx.x & 63;
  const int g = lane >> 5;
  using F = typename Mfma<T>::frag_t;
  const int s = lane & 15, hh = (lane >> 4) & 1;
  const int col = col0 + 16 * hh + 4 * (s & 3);
  const T* p0 = base + (kbase + k16_first<ORDER>(c, g) + (s >> 2)) * pitch + col;
  const T* p1 = base + (kbase + k16_second<ORDER>(c, g) + (s >> 2)) * pitch + col;
  i16x4_t a = ds_read_tr16(p0);
  i16x4_t b = ds_read_tr16(p1);
  i16x8_t v = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  return __builtin_bit_cast(F, v);
}

// Accumulator tile -> operand fragment whose k index is the tile row (KACC order), chunk c.
// c must be a compile-time constant after unrolling so the register indices stay static.
template <typename T>
__device__ __forceinline__ typename Mfma<T>::frag_t acc_frag(const f32x16_t& a, int c) {
  typename Mfma<T>::frag_t f;
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] = (T)a[c * 8 + e];
  return f;
}

// Fragment with every element multiplied by x (in float32, rounded once to T).
template <typename T>
__device__ __forceinline__ typename Mfma<T>::frag_t scaled_frag(const typename Mfma<T>::frag_t& f, float x) {
  typename Mfma<T>::frag_t r;
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = (T)((float)f[e] * x);
  return r;
}

// Two-term 16-bit split of accumulator chunk c (16-bit T only): hi = round(x), lo = round(x - hi), so
// hi + lo carries x to ~2^-16 relative and an MFMA pair over (hi, lo) sums x-weighted products with no
// operand rounding of consequence.
template <typename T, typename F>
__device__ __forceinline__ void split_frag(const f32x16_t& a, int c, F& hi, F& lo) {
  static_assert(sizeof(T) == 2, "split_frag is for 16-bit operands");
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const T h = (T)a[c * 8 + e];
    hi[e] = h;
    lo[e] = (T)(a[c * 8 + e] - (float)h);
  }
}

// ----------------------------------------------------------------------------------------------
// Global memory access
// ----------------------------------------------------------------------------------------------
// Fragment of row `row` straight from global memory (k along the row, KLIN order). Rows >= nrows
// and columns >= D read as zero. vec: 16-byte loads are legal (alignment checked by the host).
template <typename T>
__device__ __forceinline__ typename Mfma<T>::frag_t gload_frag(const T* base, int64_t rs, int row, int nrows, int c,
                                                              int D, bool vec) {
  using F = typename Mfma<T>::frag_t;
  const int g = (threadIdx.x >> 5) & 1;
  const int col = c * 16 + 8 * g;
  i16x8_t v = {0, 0, 0, 0, 0, 0, 0, 0};
  if (row < nrows) {
    const T* p = base + (int64_t)row * rs + col;
    if (vec && col + 8 <= D) {
      v = *reinterpret_cast<const i16x8_t*>(p);
    } else {
      const short* ps = reinterpret_cast<const short*>(p);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (col + e < D) ? ps[e] : (short)0;
    }
  }
  return __builtin_bit_cast(F, v);
}

// Cooperative tile staging: a [ROWS][DP] tile of rows row0.. of a (rows, D) matrix, loaded into
// registers (16 bytes per chunk) and later stored to a row-major LDS tile of pitch `pitch`.
// Out-of-range rows and columns are zero, so every LDS column < DP is defined.
template <typename T, int ROWS, int DP, int NT>
struct TileStage {
  static constexpr int THREADS = NT;
  static constexpr int VEC = 16 / (int)sizeof(T);
  static constexpr int CPR = DP / VEC;
  static constexpr int NCH = ROWS * CPR;
  static constexpr int PER = (NCH + NT - 1) / NT;
  i16x8_t r[PER];

  // Straight-line 16-byte loads; only for tiles whose rows and columns are all in range with
  // vector-legal alignment (callers check `row0 + ROWS <= nrows && D == DP && vec` first).
  __device__ __forceinline__ void load_fast(const T* base, int64_t rs, int row0) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int ch = (int)threadIdx.x + i * NT;
      if (NCH % NT == 0 || ch < NCH) {
        const int row = ch / CPR, col = (ch % CPR) * VEC;
        r[i] = *reinterpret_cast<const i16x8_t*>(base + (int64_t)(row0 + row) * rs + col);
      }
    }
  }

  // Picks the fast path when the whole tile is in range (a uniform branch).
  __device__ __forceinline__ void load_any(const T* base, int64_t rs, int row0, int nrows, int D, bool vec) {
    if (vec && D == DP && row0 + ROWS <= nrows)
      load_fast(base, rs, row0);
    else
      load(base, rs, row0, nrows, D, vec);
  }

  __device__ __forceinline__ void load(const T* base, int64_t rs, int row0, int nrows, int D, bool vec) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int ch = (int)threadIdx.x + i * NT;
      i16x8_t v = {0, 0, 0, 0, 0, 0, 0, 0};
      if (NCH % NT == 0 || ch < NCH) {
        const int row = ch / CPR, col = (ch % CPR) * VEC;
        const int grow = row0 + row;
        if (grow < nrows && col < D) {
          const T* p = base + (int64_t)grow * rs + col;
          if (vec && col + VEC <= D) {
            v = *reinterpret_cast<const i16x8_t*>(p);
          } else {
            T tmp[VEC];
#pragma unroll
            for (int e = 0; e < VEC; ++e) tmp[e] = (col + e < D) ? p[e] : (T)0.f;
            v = __builtin_bit_cast(i16x8_t, tmp);
          }
        }
      }
      r[i] = v;
    }
  }

  __device__ __forceinline__ void store(T* lds, int pitch) const {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int ch = (int)threadIdx.x + i * NT;
      if (NCH % NT == 0 || ch < NCH) {
        const int row = ch / CPR, col = (ch % CPR) * VEC;
        *reinterpret_cast<i16x8_t*>(lds + row * pitch + col) = r[i];
      }
    }
  }
};

// ----------------------------------------------------------------------------------------------
// Block scheduling
// ----------------------------------------------------------------------------------------------
// The dispatcher hands workgroup ids to the 8 XCDs round-robin, and each XCD has its own L2. This
// renumbering gives consecutive logical ids (the tiles of one (batch, head), which share K and V) to
// the same XCD, so each head's K/V is fetched from HBM into one L2 instead of eight.
__device__ __forceinline__ int xcd_remap(int bid, int nblocks) {
  constexpr int NX = 8;
  const int q = nblocks / NX, rem = nblocks % NX;
  const int xcd = bid % NX, local = bid / NX;
  return xcd < rem ? xcd * (q + 1) + local : rem * (q + 1) + (xcd - rem) * q + local;
}

// Store 4 consecutive elements (columns col..col+3 of row `row`) from float values, bounds-checked.
template <typename T>
__device__ __forceinline__ void store4(T* base, int64_t rs, int row, int col, int D, float a, float b, float c,
                                       float d, bool vec) {
  T* p = base + (int64_t)row * rs + col;
  if (vec && col + 4 <= D) {
    if constexpr (sizeof(T) == 2) {
      T v[4] = {(T)a, (T)b, (T)c, (T)d};
      *reinterpret_cast<i16x4_t*>(p) = __builtin_bit_cast(i16x4_t, v);
    } else {
      *reinterpret_cast<f32x4_t*>(p) = f32x4_t{a, b, c, d};
    }
  } else {
    if (col + 0 < D) p[0] = (T)a;
    if (col + 1 < D) p[1] = (T)b;
    if (col + 2 < D) p[2] = (T)c;
    if (col + 3 < D) p[3] = (T)d;
  }
}

// gload_frag for 16-bit T and a head dim D that is a multiple of 8, with 16-byte aligned rows: a lane's 8
// columns are all in range or all out of range, so one vector load (or zero) covers them.
template <typename T>
__device__ __forceinline__ typename Mfma<T>::frag_t gload_frag8(const T* base, int64_t rs, int row, int nrows, int c,
                                                               int D) {
  static_assert(sizeof(T) == 2, "16-bit operands only");
  const int col = c * 16 + 8 * ((threadIdx.x >> 5) & 1);
  i16x8_t v = {0, 0, 0, 0, 0, 0, 0, 0};
  if (row < nrows && col < D) v = *reinterpret_cast<const i16x8_t*>(base + (int64_t)row * rs + col);
  return __builtin_bit_cast(typename Mfma<T>::frag_t, v);
}

// store4 for a head dim D that is a multiple of 8 and a column that is a multiple of 4 (vector access).
template <typename T>
__device__ __forceinline__ void store4_8(T* base, int64_t rs, int row, int col, int D, float a, float b, float c,
                                         float d) {
  if (col >= D) return;
  T* p = base + (int64_t)row * rs + col;
  if constexpr (sizeof(T) == 2) {
    T v[4] = {(T)a, (T)b, (T)c, (T)d};
    *reinterpret_cast<i16x4_t*>(p) = __builtin_bit_cast(i16x4_t, v);
  } else {
    *reinterpret_cast<f32x4_t*>(p) = f32x4_t{a, b, c, d};
  }
}

// Load 4 consecutive elements (columns col..col+3 of row `row`) as float, zero beyond D.
template <typename T>
__device__ __forceinline__ f32x4_t load4(const T* base, int64_t rs, int row, int col, int D, bool vec) {
  const T* p = base + (int64_t)row * rs + col;
  f32x4_t out;
  if (vec && col + 4 <= D) {
    if constexpr (sizeof(T) == 2) {
      i16x4_t v = *reinterpret_cast<const i16x4_t*>(p);
      T t[4];
      __builtin_memcpy(t, &v, 8);
      out = f32x4_t{(float)t[0], (float)t[1], (float)t[2], (float)t[3]};
    } else {
      out = *reinterpret_cast<const f32x4_t*>(p);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = (col + e < D) ? (float)p[e] : 0.f;
  }
  return out;
}

// ----------------------------------------------------------------------------------------------
// float32 as three bfloat16 terms (MfmaX3)
// ----------------------------------------------------------------------------------------------
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

// Element i of a register array of 8 floats -> element i of the three terms.
// Two elements at a time, so that one v_cvt_pk_bf16_f32 rounds both and the rounded values are read back from its result
// (element by element the compiler converts each value a second time for the residual: 56 conversions instead of 24 for
// 16 elements).
// LV: 0 for |x| below 2^9, 1 below 2^16, 2 for every x; a value is split alike at every level that takes it. A product that overflows has to be float32's
// infinity, but a term of it such as a.h b.m may overflow with the other sign, and infinity - infinity is NaN (a key masked
// by -3.4e38 against a query of 1002.5). So that no term can: from 2^9 on h is x truncated and m has x's sign, l rounded
// (|l| <= 1/2 below 2^16, so that a.h b.l stays finite), from 2^16 on m is truncated too and l has x's sign; below 2^9,
// |m| <= 1. An infinity is h = +-1, m = 0, l = +-inf: l only meets the other operand's h. The dropped products of two
// operands between 2^9 and 2^16 are at most 2^-22 of theirs and 2^-25 on average (an emulation over two million pairs), of
// two operands beyond 2^-21 and 2^-24; one rounding to float32 is 2^-24 and 2^-26.
// Below 2^-110 l falls under bfloat16's smallest normal number and the split loses its low bits.
typedef float f32x2_t __attribute__((ext_vector_type(2)));
constexpr float kLarge1 = 0x1p9f, kLarge2 = 0x1p16f;
// The larger of mx and |x| (mx if x is NaN) in one instruction; fmaxf would canonicalise x in another.
__device__ __forceinline__ float max_abs(float mx, float x) {
  return __builtin_amdgcn_fmed3f(mx, __builtin_fabsf(x), THERIA_INF);
}
template <int LV>
__device__ __forceinline__ void split3_pair(float x0, float x1, bf16x2_t& h, bf16x2_t& m, bf16x2_t& l) {
  auto lo = [](bf16x2_t p) { return __uint_as_float(__builtin_bit_cast(uint32_t, p) << 16); };
  auto hi = [](bf16x2_t p) { return __uint_as_float(__builtin_bit_cast(uint32_t, p) & 0xffff0000u); };
  auto trunc = [](float x) { return __uint_as_float(__float_as_uint(x) & 0xffff0000u); };
  auto first = [&](float x) {
    if (LV == 0) return x;
    if (LV == 2 && __builtin_isinf(x)) return __builtin_copysignf(1.f, x);
    return __builtin_fabsf(x) >= kLarge1 ? trunc(x) : x;
  };
  auto second = [&](float x, float r) {
    if (LV < 2) return r;
    if (__builtin_isinf(x)) return 0.f;
    return __builtin_fabsf(x) >= kLarge2 ? trunc(r) : r;
  };
  h = __builtin_convertvector((f32x2_t{first(x0), first(x1)}), bf16x2_t);
  const float r0 = x0 - lo(h), r1 = x1 - hi(h);
  m = __builtin_convertvector((f32x2_t{second(x0, r0), second(x1, r1)}), bf16x2_t);
  l = __builtin_convertvector((f32x2_t{r0 - lo(m), r1 - hi(m)}), bf16x2_t);
}
template <int LV>
__device__ __forceinline__ X3Frag split3(const float (&x)[8]) {
  X3Frag f;
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    bf16x2_t h, m, l;
    split3_pair<LV>(x[e], x[e + 1], h, m, l);
    f.h[e] = h[0], f.h[e + 1] = h[1];
    f.m[e] = m[0], f.m[e + 1] = m[1];
    f.l[e] = l[0], f.l[e + 1] = l[1];
  }
  return f;
}

// Tile layout, fragment access and product of a kernel over elements T at padded head dim DP. float32 has its own form
// with the split products: its LDS tiles hold each row as three bfloat16 planes of DP columns (h | m | l), split once
// when the tile is staged, so that fragments are read as a 16-bit tile's are (ds_read_b128, ds_read_b64_tr_b16).
template <typename T, int DP>
struct Ops {
  using MM = Mfma<T>;
  using F = typename MM::frag_t;
  static constexpr int KC = MM::KC;
  static constexpr int PITCH = DP + 16 / (int)sizeof(T);  // elements T between rows
  __device__ __forceinline__ static F cols(const T* tile, int row, int c) {
    return lds_cols<T, KLIN>(tile, PITCH, row, 0, c);
  }
  __device__ __forceinline__ static F rows(const T* tile, int kbase, int c, int col0) {
    return lds_rows<T, KACC>(tile, PITCH, kbase, c, col0);
  }
  // A fragment from global memory in two steps, raw (the loads) and frag (what the registers need after them), so
  // that a caller can have the loads of all its operands in flight before the first frag waits for one.
  using Raw = F;
  __device__ __forceinline__ static Raw raw(const T* base, int64_t rs, int row, int nrows, int c, int D, bool vec) {
    return gload_frag<T>(base, rs, row, nrows, c, D, vec);
  }
  __device__ __forceinline__ static F frag(const Raw& r) { return r; }
  __device__ __forceinline__ static F acc(const f32x16_t& a, int c) { return acc_frag<T>(a, c); }
  template <bool SW = false>
  __device__ __forceinline__ static f32x16_t mma(const F& a, const F& b, f32x16_t c) {
    return MM::mma(a, b, c);
  }
  // store(t1, lds1, has1, t2, lds2, has2, ...): the staged tiles that are there to LDS. (Flags, not null pointers: the
  // address of an LDS array is compared at run time.)
  template <typename S, typename... A>
  __device__ __forceinline__ static void store(const S& st, T* lds, bool has, A&&... more) {
    if (has) st.store(lds, PITCH);
    if constexpr (sizeof...(more) > 0) store(more...);
  }
};

template <int DP>
struct Ops<float, DP> {
  using MM = MfmaX3;
  using F = X3Frag;
  static constexpr int KC = MM::KC;
  // 3 DP bfloat16 and padding to 52, 100 or 228 words: 16 consecutive rows start in 16 distinct groups of 4 banks
  static constexpr int PITCH = DP == 128 ? 228 : 3 * DP / 2 + 4;
  __device__ __forceinline__ static F cols(const float* tile, int row, int c) {
    const int g = (threadIdx.x >> 5) & 1;
    const char* p = reinterpret_cast<const char*>(tile + row * PITCH) + (16 * c + 8 * g) * 2;
    F f;
    f.h = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const i16x8_t*>(p));
    f.m = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const i16x8_t*>(p + 2 * DP));
    f.l = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const i16x8_t*>(p + 4 * DP));
    return f;
  }
  __device__ __forceinline__ static F rows(const float* tile, int kbase, int c, int col0) {
    F f;
    const short* t = reinterpret_cast<const short*>(tile);
    f.h = __builtin_bit_cast(bf16x8_t, lds_rows<__bf16, KACC>((const __bf16*)t, 2 * PITCH, kbase, c, col0));
    f.m = __builtin_bit_cast(bf16x8_t, lds_rows<__bf16, KACC>((const __bf16*)t + DP, 2 * PITCH, kbase, c, col0));
    f.l = __builtin_bit_cast(bf16x8_t, lds_rows<__bf16, KACC>((const __bf16*)t + 2 * DP, 2 * PITCH, kbase, c, col0));
    return f;
  }
  struct Raw {
    f32x4_t a, b;
  };
  __device__ __forceinline__ static Raw raw(const float* base, int64_t rs, int row, int nrows, int c, int D, bool vec) {
    const int col = 16 * c + 8 * ((threadIdx.x >> 5) & 1);
    Raw r = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
    if (row < nrows) {
      const float* p = base + (int64_t)row * rs + col;
      if (vec && col + 8 <= D) {
        r.a = *reinterpret_cast<const f32x4_t*>(p);
        r.b = *reinterpret_cast<const f32x4_t*>(p + 4);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (col + e < D) r.a[e] = p[e];
          if (col + 4 + e < D) r.b[e] = p[4 + e];
        }
      }
    }
    return r;
  }
  __device__ __forceinline__ static F frag(const Raw& r) {
    const float x[8] = {r.a[0], r.a[1], r.a[2], r.a[3], r.b[0], r.b[1], r.b[2], r.b[3]};
    float mx = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) mx = max_abs(mx, x[e]);
    F f = split3<0>(x);
    if (__builtin_expect(__any(mx >= kLarge1), 0)) f = split3<2>(x);
    return f;
  }
  // (P, dS and their like: always at level 0. An infinity among them gives NaN, as its sum with the row's other keys would.)
  __device__ __forceinline__ static F acc(const f32x16_t& a, int c) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = a[8 * c + e];
    return split3<0>(x);
  }
  template <bool SW = false>
  __device__ __forceinline__ static f32x16_t mma(const F& a, const F& b, f32x16_t c) {
    return MM::template mma<SW>(a, b, c);
  }
  // All the tiles of a step in one call, so that their splits interleave: at level 0, then again, to the same places, for a
  // thread that met a larger value in any of them, in a block out of the loop's line. Operands of 2^9 and more throughout
  // cost 1 to 20% (forward B2 H16 T1000 D64 59 -> 69 us, double backward 630 -> 716); splitting at the right level at once
  // would save most of that and costs the usual operands 2 to 4%, since nothing can start before the look is done.
  template <typename... A>
  __device__ __forceinline__ static void store(A&&... tiles) {
    const float mx = put<0>(tiles...);
    if (__builtin_expect(__any(mx >= kLarge1), 0)) {  // uniform
      if (mx >= kLarge2)
        put<2>(tiles...);
      else if (mx >= kLarge1)
        put<1>(tiles...);
    }
  }

 private:
  // Returns the largest |x| (level 0).
  template <int LV, typename S, typename... A>
  __device__ __forceinline__ static float put(const S& st, float* lds, bool has, A&&... more) {
    float mx = 0.f;
    if (has) {
#pragma unroll
      for (int i = 0; i < S::PER; ++i) {
        const int ch = (int)threadIdx.x + i * S::THREADS;
        if (S::NCH % S::THREADS == 0 || ch < S::NCH) {
          const int row = ch / S::CPR, col = (ch % S::CPR) * S::VEC;
          const f32x4_t x = __builtin_bit_cast(f32x4_t, st.r[i]);
          bf16x4_t h, m, l;
#pragma unroll
          for (int e = 0; e < 4; e += 2) {
            bf16x2_t h2, m2, l2;
            split3_pair<LV>(x[e], x[e + 1], h2, m2, l2);
            h[e] = h2[0], h[e + 1] = h2[1];
            m[e] = m2[0], m[e + 1] = m2[1];
            l[e] = l2[0], l[e + 1] = l2[1];
            if constexpr (LV == 0) mx = max_abs(max_abs(mx, x[e]), x[e + 1]);
          }
          char* p = reinterpret_cast<char*>(lds + row * PITCH) + 2 * col;
          *reinterpret_cast<i16x4_t*>(p) = __builtin_bit_cast(i16x4_t, h);
          *reinterpret_cast<i16x4_t*>(p + 2 * DP) = __builtin_bit_cast(i16x4_t, m);
          *reinterpret_cast<i16x4_t*>(p + 4 * DP) = __builtin_bit_cast(i16x4_t, l);
        }
      }
    }
    if constexpr (sizeof...(more) > 0) mx = max_abs(mx, put<LV>(more...));
    return mx;
  }
};

}  // namespace theria
