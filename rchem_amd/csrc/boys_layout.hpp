// Layout of the exact Boys function's tables (boys.hpp evaluates them,
// boys_table.hpp computes them).
//
// A lookup takes one row of coefficients, of the grid point T0 nearest to T: F_M
// as a polynomial in T0 - T.  FP64: spacing 1/8 and 9 terms.  FP32: spacing 1/16
// and 4 terms, one 16-byte read; order 1, whose F_1 is the polynomial's derivative,
// 1/8 and 6 terms.  Rows and terms are what F_m's last bits need: worst and
// root-mean-square relative error over 0 <= T < 36 (3e6 arguments, log and
// uniform, 80-bit F_m; in brackets the Taylor rows on 1/8, 9 terms or in FP32 6,
// that this table may not be worse than): FP64 order 0 2.13e-16, 5.80e-17 (the
// same), order 1 F_1 3.2e-16, 8.4e-17 (1.15e-15, 1.25e-16).  FP32 order 0
// 1.144e-7, 3.067e-8 (1.138e-7, 3.076e-8), order 1 F_1 1.71e-7, 4.57e-8 (the same),
// order 4 F_0 4.2e-7, 8.87e-8 (4.2e-7, 8.93e-8).  Shorter rows were tried: cells
// doubling with T + 4 and 7 or 8 terms for orders 0 and 1 (12 KB of LDS where this
// takes 21) had F_0 2.5e-16, 6.3e-17; 8 terms on 1/8 F_1 2.3e-15.
#pragma once

namespace rchem {

constexpr int kBoysMaxM = 9;  // highest m served
constexpr double kBoysTMax = 36.0;

constexpr int boys_inv_h(int M, bool f64) { return f64 || M == 1 ? 8 : 16; }
constexpr int boys_terms(int M, bool f64) { return f64 ? 9 : M == 1 ? 6 : 4; }
constexpr int boys_rows(int M, bool f64) { return 36 * boys_inv_h(M, f64) + 1; }
// Entries from one row to the next: all the terms (FP64 rows an odd number of
// doubles, so that they start at every bank pair).
constexpr int boys_block(int M, bool f64) { return boys_rows(M, f64) * boys_terms(M, f64); }
// Device layout: the orders' blocks one after the other, then (FP64) the row
// of e^{-T0} that the downward recursions of M >= 2 share.  Order 1 holds F_0
// as a polynomial whose derivative is F_1 (dF_0/dT = -F_1), so that one pass
// gives both with no exponential.
constexpr int boys_offset(int M, bool f64) {
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
constexpr int boys_stage_size(int M, bool f64 = true) {
  return boys_block(M, f64) + (f64 && M >= 2 ? kBoysExpRows : 0);
}

}  // namespace rchem
