// The Boys tables in device layout (boys_layout.hpp), computed on the host in
// long double.
#pragma once
#include <cmath>
#include <vector>

#include "boys_layout.hpp"

namespace rchem {

struct BoysTables {
  std::vector<double> f64;
  std::vector<float> f32;
};

// Per row the derivatives of F_M about the grid point T0, F_{M+j}(T0) / j! in
// powers of T0 - T, from the all-positive series
// F_m(T) = e^{-T} sum_k (2T)^k / ((2m+1) ... (2m+2k+1)) at the highest order and
// downward recursion.  Order 0 and those from 2 on: the first terms.  Order 1: the
// series of F_1 is rewritten in Chebyshev polynomials of the cell, cut there
// (which leaves 2^(1-n) of what cutting the powers would) and integrated, so that
// F_0's polynomial starts at F_0(T0) exactly and has F_1's as its derivative.
// FP32 rows are cut the same way throughout, having few terms.
inline BoysTables make_boys_tables() {
  constexpr int kD = 14;  // terms of the series before the cut
  constexpr int kM = kBoysMaxM + kD;
  using Real = long double;
  Real cheb[kD][kD] = {};  // Chebyshev polynomials' coefficients
  cheb[0][0] = 1.0L;
  cheb[1][1] = 1.0L;
  for (int n = 2; n < kD; ++n)
    for (int i = 0; i < kD; ++i)
      cheb[n][i] = (i > 0 ? 2.0L * cheb[n - 1][i - 1] : 0.0L) - cheb[n - 2][i];
  auto boys_at = [](Real T, Real* F) {
    Real term = 1.0L / (2 * kM + 1), sum = term;
    for (int k = 1; k < 4000; ++k) {
      term *= 2.0L * T / (2 * kM + 2 * k + 1);
      sum += term;
      if (term < sum * 1e-21L) break;
    }
    const Real e = std::exp(-T);
    F[kM] = e * sum;
    for (int m = kM - 1; m >= 0; --m) F[m] = (2.0L * T * F[m + 1] + e) / (2 * m + 1);
  };
  // the first K coefficients in d of sum_j a_j d^j over |d| <= h, cut in
  // Chebyshev polynomials of d / h
  auto cut = [&](const Real* a, Real h, int K, Real* out) {
    Real r[kD], keep[kD] = {};
    Real hp = 1.0L;
    for (int j = 0; j < kD; ++j, hp *= h) r[j] = a[j] * hp;
    for (int n = kD - 1; n >= 0; --n) {
      const Real c = r[n] / cheb[n][n];
      for (int i = 0; i <= n; ++i) {
        r[i] -= c * cheb[n][i];
        if (n < K) keep[i] += c * cheb[n][i];
      }
    }
    hp = 1.0L;
    for (int j = 0; j < K; ++j, hp *= h) out[j] = keep[j] / hp;
  };
  BoysTables t;
  t.f64.resize(kBoysTableSize);
  t.f32.resize(kBoysTableSizeF);
  for (const bool f64 : {true, false})
    for (int M = 0; M <= kBoysMaxM; ++M) {
      const int K = boys_terms(M, f64), inv_h = boys_inv_h(M, f64);
      for (int r = 0; r < boys_rows(M, f64); ++r) {
        const Real h = 0.5L / inv_h, T = static_cast<Real>(r) / inv_h;
        Real F[kM + 1], a[kD], c[kD], fact = 1.0L;
        boys_at(T, F);
        for (int j = 0; j < kD; ++j) {
          if (j > 0) fact *= j;
          a[j] = c[j] = F[M + j] / fact;
        }
        if (M == 1) {
          Real q[kD];
          cut(a, h, K - 1, q);
          c[0] = F[0];
          for (int j = 1; j < K; ++j) c[j] = q[j - 1] / j;
        } else if (!f64) {
          cut(a, h, K, c);
        }
        const int o = boys_offset(M, f64) + r * K;
        for (int j = 0; j < K; ++j) {
          if (f64)
            t.f64[o + j] = static_cast<double>(c[j]);
          else
            t.f32[o + j] = static_cast<float>(c[j]);
        }
        if (f64 && M == 2) t.f64[kBoysExpOffset + r] = static_cast<double>(std::exp(-T));
      }
    }
  return t;
}

}  // namespace rchem
