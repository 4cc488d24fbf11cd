// Device Boys function F_m(T) = int_0^1 t^(2m) exp(-T t^2) dt for gfx950.
//
// Two evaluations:
//   * exact (production): F_M(T) from a polynomial about the centre of T's grid
//     cell, then downward recursion F_m = (2T F_{m+1} + e^{-T}) / (2m+1), which
//     is stable, with e^{-T} = e^{-T0} e^{T0 - T} from the same cell and a short
//     polynomial.  For T >= 36 the asymptote F_0 = sqrt(pi/T)/2 (error < e^{-T})
//     and the upward recursion F_{m+1} = ((2m+1) F_m - e^{-T}) / (2T) are used.
//     The coefficients are the Taylor series about the cell's centre with its
//     last terms folded down (Chebyshev economisation), computed on the host in
//     long double; a kernel stages its order's block in LDS, so every lookup is
//     an LDS read, not a cache miss.
//   * compat (parity with the reference): the Numerical-Recipes incomplete
//     gamma of libpyquante2 (cints.c:302-373) evaluated per m with its own
//     constants (EPS = 3e-7, ITMAX = 100, x clamped to >= 1e-8), so integrals
//     reproduce the reference's Boys truncation error exactly.  Used only
//     where bit-level agreement with the reference's integrals is requested.
#pragma once
#include <hip/hip_runtime.h>

namespace rchem {

constexpr int kBoysMaxM = 9;                          // highest m served
constexpr double kBoysTMax = 36.0;

// The grid.  A lookup gathers one row of coefficients per lane, and those
// gathers (random rows, so each LDS instruction meets bank conflicts) kept the
// LDS busy for 44 % of the (10|00) and (00|00) kernels' time when a row was 9
// Taylor coefficients on a uniform grid of 1/8.  Cutting the series of a cell
// of half width h at n terms leaves h^n F_{m+n} / n! 2^(1-n) of it in Chebyshev
// polynomials, 2^(1-n) of what cutting the powers of d leaves.
//   * orders 0 and 1: F_{m+n} / F_m falls as T^-n beyond T ~ 4, so cells that
//     double in width from one octave of T + 4 to the next ([4, 8), [8, 16),
//     [16, 32), [32, 40)) need the same n everywhere: 13/4 octaves of 2^bits
//     cells where a uniform grid has 36/4.  FP64: 2^6 cells to an octave (width
//     1/16 below T = 4; 208 rows, 12 and 15 KB of LDS where 289 rows took 21)
//     and 7 terms for order 0, 8 for order 1.  FP32: 4 terms, one 16-byte read.
//   * orders >= 2: the fall begins later (T > m + n), so the grid stays uniform:
//     FP64 1/8 with 8 terms, FP32 1/16 with 4.
// Worst relative errors over 0 <= T < 36 against 80-bit F_m (3e5 arguments, log
// and uniform, cell edges among them; the 9-term rows in brackets): order 0
// 2.5e-16 (2.1e-16; 2.1e-16 outside the two cells above T = 12), order 1 F_0
// 2.1e-16 (2.1e-16) and F_1 7.0e-16 (1.1e-15), order 4 F_0 6.8e-16 (6.8e-16)
// and F_4 2.2e-16 (2.2e-16).  FP32: order 0 1.1e-7 (1.1e-7), F_1 1.6e-7
// (1.6e-7), order 4 F_0 4.3e-7 (4.3e-7).
__host__ __device__ constexpr bool boys_octaves(int M) { return M <= 1; }
__host__ __device__ constexpr int boys_bits(int M, bool f64) { return f64 || M == 0 ? 6 : 8; }
__host__ __device__ constexpr int boys_inv_h(bool f64) { return f64 ? 8 : 16; }
__host__ __device__ constexpr int boys_terms(int M, bool f64) {
  return f64 ? (M == 0 ? 7 : 8) : 4;
}
// Entries from one row to the next: FP64 rows an odd number of doubles (8-term
// rows padded to 9), so that rows start at every bank pair.
__host__ __device__ constexpr int boys_stride(int M, bool f64) {
  return f64 ? (M == 0 ? 7 : 9) : 4;
}
__host__ __device__ constexpr int boys_rows(int M, bool f64) {
  return boys_octaves(M) ? 13 << (boys_bits(M, f64) - 2)  // three octaves and [32, 40)
                         : 36 * boys_inv_h(f64) + 1;
}
__host__ __device__ constexpr int boys_block(int M, bool f64) {
  return boys_rows(M, f64) * boys_stride(M, f64);
}
// Device layout: the orders' blocks one after the other, then (FP64) the row
// of e^{-T0} that the downward recursions of M >= 2 share.  Order 1 holds F_0
// as a polynomial whose derivative is F_1 (dF_0/dT = -F_1), so that one pass
// gives both with no exponential.
__host__ __device__ constexpr int boys_offset(int M, bool f64) {
  int o = 0;
  for (int m = 0; m < M; ++m) o += boys_block(m, f64);
  return o;
}
constexpr int kBoysExpRows = boys_rows(2, true);
constexpr int kBoysExpOffset = boys_offset(kBoysMaxM + 1, true);
constexpr int kBoysTableSize = kBoysExpOffset + kBoysExpRows;
constexpr int kBoysTableSizeF = boys_offset(kBoysMaxM + 1, false);
// Staged entries a kernel of highest order M needs: its block and, for FP64
// and M >= 2, the exp row.
__host__ __device__ constexpr int boys_stage_size(int M, bool f64 = true) {
  return boys_block(M, f64) + (f64 && M >= 2 ? kBoysExpRows : 0);
}

enum BoysMode { kBoysExact = 0, kBoysCompat = 1 };

// 1/sqrt(x) from the hardware estimate.  FP64: the estimate (measured on
// gfx950: 5.2e-8 relative over [0.05, 2e4]) refined by one third-order
// (Halley) step, y (1 + e/2 + 3e^2/8) with e = 1 - x y^2, whose error is
// O(e^3) -- five operations in a chain of five, where two Newton steps take
// six in a chain of seven; ~1 ulp, a fraction of the cost of the IEEE
// division and square root sequences.  FP32: the estimate as it is, within
// 0.86 ulp (measured on gfx950 over [1e-3, 1e5] against FP64); one Newton
// step in FP32 (four operations) measured 1.53 ulp, its own rounding
// outweighing what it corrects.
__device__ __forceinline__ double fast_rsqrt(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = __builtin_fma(-x * y, y, 1.0);
  return __builtin_fma(y * e, __builtin_fma(0.375, e, 0.5), y);
}
__device__ __forceinline__ float fast_rsqrt(float x) { return __builtin_amdgcn_rsqf(x); }

// The cell of T (0 <= T < kBoysTMax) on the grid of 2^BITS cells to an octave
// of T + 4, and d = T0 - T, T0 the cell's centre.  The sum r = T + 4 has the
// octave in its exponent and the cell in its leading BITS mantissa bits: the
// row index is its high word shifted, the centre that word with the rest
// replaced by 100...0.  T0 - T is exact, so rounding r costs nothing but a cell
// entered an ulp early.  r < 40 for every T < 36 (ulps are equal there).
template <int BITS, typename R>
__host__ __device__ __forceinline__ void boys_cell(R T, int* k, R* d) {
  const R r = T + R(4);
  if constexpr (sizeof(R) == 8) {
    constexpr int sh = 20 - BITS;
    union { double f; unsigned long long u; } x{r}, c;
    const unsigned hi = static_cast<unsigned>(x.u >> 32);
    *k = static_cast<int>(hi >> sh) - (0x40100000 >> sh);
    c.u = static_cast<unsigned long long>((hi & (~0u << sh)) | (1u << (sh - 1))) << 32;
    *d = (c.f - 4.0) - T;
  } else {
    constexpr int sh = 23 - BITS;
    union { float f; unsigned u; } x{r}, c;
    *k = static_cast<int>(x.u >> sh) - (0x40800000 >> sh);
    c.u = (x.u & (~0u << sh)) | (1u << (sh - 1));
    *d = (c.f - 4.0f) - T;
  }
}

// The grid point nearest to T (0 <= T < kBoysTMax) of the uniform grid: its
// index k and d = T0 - T, |d| at most half the spacing.  Rounding by adding the
// power of two whose ulp is the spacing: the sum r = kMagic + T0 has k in its
// low mantissa bits (read off the register, no conversion), r - kMagic is T0
// exactly, and T0 - T is exact (a multiple of T's ulp).  A tie rounds to even.
template <typename R>
__host__ __device__ __forceinline__ void boys_grid(R T, int* k, R* d) {
  if constexpr (sizeof(R) == 8) {
    constexpr double kMagic = 562949953421312.0;  // 2^49: ulp 1/8 on [2^49, 2^50)
    static_assert(boys_inv_h(true) == 8, "kMagic");
    const union { double f; unsigned long long u; } r{T + kMagic};
    *k = static_cast<int>(static_cast<unsigned>(r.u));
    *d = (r.f - kMagic) - T;
  } else {
    constexpr float kMagic = 524288.0f;  // 2^19: ulp 1/16 on [2^19, 2^20)
    static_assert(boys_inv_h(false) == 16, "kMagic");
    const union { float f; unsigned u; } r{T + kMagic};
    *k = static_cast<int>(r.u & 0x7fffffu);
    *d = (r.f - kMagic) - T;
  }
}

// Row and offset of T in the block of order M.
template <int M, typename R>
__host__ __device__ __forceinline__ void boys_locate(R T, int* k, R* d) {
  if constexpr (boys_octaves(M)) boys_cell<boys_bits(M, sizeof(R) == 8), R>(T, k, d);
  else boys_grid<R>(T, k, d);
}

// e^d, |d| <= 1/16, by its Taylor series (the recursion multiplies its error,
// so it keeps the ninth term that F_M's polynomial does without).
constexpr int kExpTerms = 9;
constexpr double kExpPoly[kExpTerms] = {1.0,       1.0,       1.0 / 2,    1.0 / 6,    1.0 / 24,
                                        1.0 / 120, 1.0 / 720, 1.0 / 5040, 1.0 / 40320};

// The coefficients of row k of a staged block of order M (FP32 rows are 16-byte
// aligned: one wide LDS read).
template <int M, typename R>
__device__ __forceinline__ void boys_row(const R* __restrict__ table, int k, R* __restrict__ c) {
  constexpr int K = boys_terms(M, sizeof(R) == 8);
  // 0 <= k < rows: a 24-bit multiply (full rate; a 32-bit one is quarter rate)
  const R* __restrict__ row =
      table + __umul24(static_cast<unsigned>(k), boys_stride(M, sizeof(R) == 8));
  if constexpr (sizeof(R) == 4) {
    static_assert(K == 4 || sizeof(R) == 8, "one float4 per FP32 row");
    const float4 v = *reinterpret_cast<const float4*>(row);
    c[0] = v.x;
    c[1] = v.y;
    c[2] = v.z;
    c[3] = v.w;
  } else {
#pragma unroll
    for (int j = 0; j < K; ++j) c[j] = row[j];
  }
}

// F_0 and F_1 (order 1) from the row's polynomial p in d and its derivative:
// the derivative's chain starts at c_{K-1} (its first step, 0 d + p, is not
// left to the compiler, which may not drop a product with 0).
template <int K, typename R>
__device__ __forceinline__ void boys_poly01(const R* c, R d, R* f0, R* f1) {
  R q = c[K - 1];
  R p = q * d + c[K - 2];
#pragma unroll
  for (int j = K - 3; j >= 0; --j) {
    q = q * d + p;
    p = p * d + c[j];
  }
  *f0 = p;
  *f1 = q;
}

// Exact Boys F_0..F_M into F[0..M]; `table` is the staged block of order M
// (then, for FP64 and M >= 2, the exp row), 16-byte aligned, normally in LDS.
template <int M, typename R>
__device__ __forceinline__ void boys_exact(R T, const R* __restrict__ table, R* __restrict__ F) {
  static_assert(M <= kBoysMaxM, "Boys order beyond the table");
  constexpr bool kF64 = sizeof(R) == 8;
  constexpr int K = boys_terms(M, kF64);
  if (T < R(kBoysTMax)) {
    int k;
    R d;  // T0 - T
    boys_locate<M, R>(T, &k, &d);
    R c[K];
    boys_row<M, R>(table, k, c);
    if constexpr (M == 1) {
      boys_poly01<K>(c, d, &F[0], &F[1]);
      return;
    }
    R f = c[K - 1];
#pragma unroll
    for (int j = K - 2; j >= 0; --j) f = c[j] + d * f;
    F[M] = f;
    if constexpr (M > 0 && !kF64) {
      const R e = __expf(-T);  // hardware exp2: ample for the FP32 path
      const R t2 = T + T;
#pragma unroll
      for (int m = M - 1; m >= 0; --m) F[m] = (t2 * F[m + 1] + e) * R(1.0 / (2 * m + 1));
    } else if constexpr (M > 0) {
      R p = R(kExpPoly[kExpTerms - 1]);
#pragma unroll
      for (int j = kExpTerms - 2; j >= 0; --j) p = R(kExpPoly[j]) + d * p;
      const R e = table[boys_block(M, true) + k] * p;  // e^{-T0} e^{d}
      const R t2 = T + T;
#pragma unroll
      for (int m = M - 1; m >= 0; --m) F[m] = (t2 * F[m + 1] + e) * R(1.0 / (2 * m + 1));
    }
  } else {
    const R rt = fast_rsqrt(T);
    F[0] = R(0.88622692545275801365) * rt;  // sqrt(pi)/2 / sqrt(T); erf(sqrt T) = 1 - O(e^-T)
    if constexpr (M == 1) {
      // F_1 = (F_0 - e^{-T}) / (2T): e^{-T} / F_0 < 2e-15 for T >= 36, so the
      // exponential is dropped (the branch costs a few operations per lane)
      F[1] = F[0] * (R(0.5) * rt * rt);
    } else if constexpr (M > 1) {
      // e^{-T} < 2.4e-16 here: it only corrects the upward recursion, so a
      // single-precision exponential is accurate enough
      const R e = static_cast<R>(__expf(-static_cast<float>(T)));
      const R h = R(0.5) * rt * rt;  // 1/(2T)
#pragma unroll
      for (int m = 0; m < M; ++m) F[m + 1] = (R(2 * m + 1) * F[m] - e) * h;
    }
  }
}

// Orders 0 and 1 without a branch: the table form (at the clamped grid point
// for T beyond the table) and the asymptotic form are both evaluated and the
// one that applies is selected, so the caller's loop body stays one basic
// block.  Higher orders take boys_exact.
template <int M, typename R>
__device__ __forceinline__ void boys_exact_select(R T, const R* __restrict__ table,
                                                  R* __restrict__ F) {
  if constexpr (M > 1) {
    boys_exact<M, R>(T, table, F);
  } else {
    constexpr bool kF64 = sizeof(R) == 8;
    constexpr int K = boys_terms(M, kF64);
    const bool near = T < R(kBoysTMax);
    const R Tn = near ? T : R(0);
    int k;
    R d;
    boys_locate<M, R>(Tn, &k, &d);
    R c[K];
    boys_row<M, R>(table, k, c);
    const R rt = fast_rsqrt(near ? R(1) : T);
    const R f0 = R(0.88622692545275801365) * rt;
    if constexpr (M == 1) {
      R p, q;
      boys_poly01<K>(c, d, &p, &q);
      F[0] = near ? p : f0;
      F[1] = near ? q : f0 * (R(0.5) * rt * rt);
    } else {
      R p = c[K - 1];
#pragma unroll
      for (int j = K - 2; j >= 0; --j) p = p * d + c[j];
      F[0] = near ? p : f0;
    }
  }
}

// Copies the block of order M and, where the recursion needs it, the exp row
// into LDS: boys_stage_size(M) entries (every thread of the workgroup calls
// it; a barrier follows).
template <int M, typename R>
__device__ __forceinline__ void stage_boys(R* __restrict__ dst, const R* __restrict__ src) {
  constexpr bool kF64 = sizeof(R) == 8;
  constexpr int m = M <= kBoysMaxM ? M : kBoysMaxM;
  constexpr int off = boys_offset(m, kF64), len = boys_block(m, kF64);
  for (int k = threadIdx.x; k < len; k += blockDim.x) dst[k] = src[off + k];
  if constexpr (boys_stage_size(m, kF64) > len)
    for (int k = threadIdx.x; k < kBoysExpRows; k += blockDim.x)
      dst[len + k] = src[kBoysExpOffset + k];
}

// Compat: the reference's Fgamma(m, x) (cints.c:302-373), NR gser/gcf.
__device__ __forceinline__ double fgamma_compat(double m, double x) {
  const double EPS = 3.0e-7, FPMIN = 1.0e-30;
  if (fabs(x) < 1.0e-8) x = 1.0e-8;
  const double a = m + 0.5;
  const double gln = lgamma(a);
  double val;
  if (x < a + 1.0) {
    double ap = a, del = 1.0 / a, sum = del;
    val = __builtin_nan("");
    for (int n = 1; n <= 100; ++n) {
      ap += 1.0;
      del *= x / ap;
      sum += del;
      if (fabs(del) < fabs(sum) * EPS) {
        const double gamser = sum * exp(-x + a * log(x) - gln);
        val = exp(gln) * gamser;
        break;
      }
    }
  } else {
    double b = x + 1.0 - a, c = 1.0 / FPMIN, d = 1.0 / b, h = d;
    for (int i = 1; i <= 100; ++i) {
      const double an = -i * (i - a);
      b += 2.0;
      d = an * d + b;
      if (fabs(d) < FPMIN) d = FPMIN;
      c = b + an / c;
      if (fabs(c) < FPMIN) c = FPMIN;
      d = 1.0 / d;
      const double del = d * c;
      h *= del;
      if (fabs(del - 1.0) < EPS) break;
    }
    const double gammcf = exp(-x + a * log(x) - gln) * h;
    val = exp(gln) * (1.0 - gammcf);
  }
  return 0.5 * pow(x, -m - 0.5) * val;
}

template <int M>
__device__ __forceinline__ void boys_compat(double T, double* __restrict__ F) {
#pragma unroll
  for (int m = 0; m <= M; ++m) F[m] = fgamma_compat(double(m), T);
}

template <int M, int MODE, typename R, bool SELECT = false>
__device__ __forceinline__ void boys(R T, const R* __restrict__ table, R* __restrict__ F) {
  if constexpr (MODE == kBoysCompat) {
    boys_compat<M>(T, F);
  } else if constexpr (SELECT) {
    boys_exact_select<M, R>(T, table, F);
  } else {
    boys_exact<M, R>(T, table, F);
  }
}

}  // namespace rchem
