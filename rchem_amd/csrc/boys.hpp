// Device Boys function F_m(T) = int_0^1 t^(2m) exp(-T t^2) dt for gfx950.
//
// Two evaluations:
//   * exact (production): F_M(T) from a polynomial about the grid point nearest to
//     T, then downward recursion F_m = (2T F_{m+1} + e^{-T}) / (2m+1), which
//     is stable, with e^{-T} = e^{-T0} e^{T0 - T} from the same row and a short
//     polynomial.  For T >= 36 the asymptote F_0 = sqrt(pi/T)/2 (error < e^{-T})
//     and the upward recursion F_{m+1} = ((2m+1) F_m - e^{-T}) / (2T) are used.
//     The coefficients are computed on the host in long double (boys_table.hpp); a
//     kernel stages its order's block in LDS, so every lookup is an LDS read, not
//     a cache miss.
//   * compat (parity with the reference): the Numerical-Recipes incomplete
//     gamma of libpyquante2 (cints.c:302-373) evaluated per m with its own
//     constants (EPS = 3e-7, ITMAX = 100, x clamped to >= 1e-8), so integrals
//     reproduce the reference's Boys truncation error exactly.  Used only
//     where bit-level agreement with the reference's integrals is requested.
#pragma once
#include <hip/hip_runtime.h>

#include "boys_layout.hpp"

namespace rchem {

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

// The grid point nearest to T (0 <= T < kBoysTMax): its index k and d = T0 - T,
// |d| at most half the spacing.  Rounding by adding the power of two whose ulp is
// the spacing: the sum r = kMagic + T0 has k in its low mantissa bits (read off the
// register, no conversion), r - kMagic is T0 exactly, and T0 - T is exact (a
// multiple of T's ulp).  A tie rounds to even.
template <int M, typename R>
__host__ __device__ __forceinline__ void boys_locate(R T, int* k, R* d) {
  constexpr int inv_h = boys_inv_h(M, sizeof(R) == 8);
  if constexpr (sizeof(R) == 8) {
    constexpr double kMagic = 562949953421312.0;  // 2^49: ulp 1/8 on [2^49, 2^50)
    static_assert(inv_h == 8, "kMagic");
    const union { double f; unsigned long long u; } r{T + kMagic};
    *k = static_cast<int>(static_cast<unsigned>(r.u));
    *d = (r.f - kMagic) - T;
  } else {
    // 2^20 and 2^19: ulps 1/8 and 1/16 up to the next power
    constexpr float kMagic = inv_h == 8 ? 1048576.0f : 524288.0f;
    static_assert(inv_h == 8 || inv_h == 16, "kMagic");
    const union { float f; unsigned u; } r{T + kMagic};
    *k = static_cast<int>(r.u & 0x7fffffu);
    *d = (r.f - kMagic) - T;
  }
}

// e^d, |d| <= 1/16, by its Taylor series.
constexpr int kExpTerms = 9;
constexpr double kExpPoly[kExpTerms] = {1.0,       1.0,       1.0 / 2,    1.0 / 6,    1.0 / 24,
                                        1.0 / 120, 1.0 / 720, 1.0 / 5040, 1.0 / 40320};

// The coefficients of row k of a staged block of order M (FP32 rows are read in
// their 16 bytes or, of 24, in eights).
template <int M, typename R>
__device__ __forceinline__ void boys_row(const R* __restrict__ table, int k, R* __restrict__ c) {
  constexpr int K = boys_terms(M, sizeof(R) == 8);
  // 0 <= k < rows: a 24-bit multiply (full rate; a 32-bit one is quarter rate)
  const R* __restrict__ row = table + __umul24(static_cast<unsigned>(k), K);
  if constexpr (sizeof(R) == 4 && K == 4) {
    const float4 v = *reinterpret_cast<const float4*>(row);
    c[0] = v.x;
    c[1] = v.y;
    c[2] = v.z;
    c[3] = v.w;
  } else if constexpr (sizeof(R) == 4) {
    static_assert(sizeof(R) == 8 || K % 2 == 0, "rows of whole float2");
#pragma unroll
    for (int j = 0; j < K; j += 2) {
      const float2 v = *reinterpret_cast<const float2*>(row + j);
      c[j] = v.x;
      c[j + 1] = v.y;
    }
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
