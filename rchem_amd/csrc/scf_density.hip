// The density of a Fock matrix of at most 128 functions in one launch (gfx950),
// one workgroup to a matrix, many matrices to a launch.
//
//   F' = X F X,  P = the projector onto F''s nocc lowest eigenvectors,
//   D = X P X      (rchem.rs:56-59, 74-78, 101-104; X symmetric, Loewdin's)
//
// rchem forms P from F''s eigenvectors.  Only the projector is wanted, and
// purification forms it by products alone: P_0 = (e_max - F') / (e_max - e_min)
// with Gershgorin's bounds, then P <- P^2 or 2P - P^2, whichever brings the trace
// nearer to nocc (the trace-correcting second-order scheme, Niklasson 2002;
// every step squares the distance of the eigenvalues from 0 or from 1).  A
// matrix without a gap at the Fermi level does not get there; its flag says so
// and the caller takes the eigensolver.
//
// Error against extended precision of the density of a core guess, 56 matrices of 1
// to 8 waters (n = 7 to 104, gaps 0.2 to 4): the largest 1.07 times rocSOLVER's
// eigensolver's in the geometric mean (0.63 to 2.0; 2.5e-15 to 3e-13, most of it
// S^(-1/2)'s), the root mean square 1.00 times; the cubic scheme by library products
// 1.07 times.  (Dense synthetic spectra with core levels at -20: up to 7 times.)
//
// What bounds it: one matrix's products on one CU.  The matrix stays in LDS
// (128 x 130 doubles) from F' to P; a step is the lower triangle of P^2 on the
// matrix cores (v_mfma_f64_16x16x4, 64 cycles each and SIMD) and two
// workgroup barriers, with no launch, no pass over memory and no host between
// steps.  The eigensolver's chain -- a Householder tridiagonalisation of n
// dependent steps, a divide and conquer, ~60 launches in all -- took 1.9 ms for
// n = 104, 1.3 ms for 48 matrices up to n = 84; this kernel takes 0.34 and 0.25
// ms with F' and X P X in it.
//
// Layouts.  v_mfma_f64_16x16x4: lane l holds A[l % 16][l / 16] and
// B[l / 16][l % 16], and of the result rows 4 r + l / 16, column l % 16
// (r = 0..3).  A leading dimension of 2 modulo 16 doubles puts the 32 lanes of a
// read (16 rows or 16 columns by two k) on different bank pairs.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "types.hpp"

namespace rchem {

namespace {

using double4_t = __attribute__((ext_vector_type(4))) double;

constexpr int kTile = 16;
constexpr int kMaxTiles = kDensityMaxN / kTile;     // tiles to a side
constexpr int kMaxWaves = 16;
constexpr int kFull = kMaxTiles * kMaxTiles / kMaxWaves;  // tiles of a full product to a wave
constexpr int kMaxSteps = 100;
constexpr double kIdempotent = 1e-9;  // tr(P - P^2) from which one more pair of steps suffices

__device__ __forceinline__ double sum64(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// One 16 x 16 tile of A B, k < K (a multiple of 16): a(row, k), b(k, column).
template <typename FA, typename FB>
__device__ __forceinline__ double4_t tile_product(int K, int lane, FA a, FB b) {
  const int c = lane & 15, q = lane >> 4;
  double4_t acc = {0.0, 0.0, 0.0, 0.0};
  for (int k = 0; k < K; k += 16) {
    double x[4], y[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      x[u] = a(c, k + 4 * u + q);
      y[u] = b(k + 4 * u + q, c);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x[u], y[u], acc, 0, 0, 0);
  }
  return acc;
}

// Tile t of the lower triangle, row by row.
__device__ __forceinline__ void triangle(int t, int* i, int* j) {
  int r = 0;
  while ((r + 1) * (r + 2) / 2 <= t) ++r;
  *i = r;
  *j = t - r * (r + 1) / 2;
}

// Matrix m: F + m f_stride, X + m x_stride, D + m d_stride with leading
// dimension ld, size nb[m] (n where nb is null) and nocc[m] (nocc1 where null).
// flag[2m + 1]: 0 once D holds the density, 1 if the purification has not
// converged or was not asked for (nocc < 0) (flag[2m] is 0.5: the pair reads as a
// purification step's coefficient and tr(P - P^2)).
__global__ __launch_bounds__(64 * kMaxWaves) void density_small_kernel(
    const double* __restrict__ Fb, const double* __restrict__ Xb, size_t stride, int ld, int n0,
    const int* __restrict__ nb, int nocc1, const int* __restrict__ noccb, double* __restrict__ Db,
    double* __restrict__ flag) {
  extern __shared__ __align__(16) double A[];
  __shared__ double red[2 * kMaxWaves];
  const int m = blockIdx.x;
  const int n = nb ? nb[m] : n0, nocc = noccb ? noccb[m] : nocc1;
  if (nocc < 0) {  // block-uniform
    if (threadIdx.x == 0) {
      flag[2 * m] = 0.5;
      flag[2 * m + 1] = 1.0;
    }
    return;
  }
  const double* __restrict__ F = Fb + m * stride;
  const double* __restrict__ X = Xb + m * stride;
  double* __restrict__ D = Db + m * stride;
  const int nt = (n + kTile - 1) / kTile, N = nt * kTile, la = N + 2;
  const int W = blockDim.x >> 6;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int c = lane & 15, q = lane >> 4;
  const int ntri = nt * (nt + 1) / 2, nfull = nt * nt;
  auto from = [&](const double* __restrict__ M, int r, int s) {
    return r < n && s < n ? M[static_cast<size_t>(r) * ld + s] : 0.0;
  };
  auto lds = [&](int r, int s) -> double& { return A[r * la + s]; };

  // A = F X
  for (int t = wave; t < nfull; t += W) {
    const int ti = kTile * (t / nt), tj = kTile * (t % nt);
    const double4_t v = tile_product(
        N, lane, [&](int r, int k) { return from(F, ti + r, k); },
        [&](int k, int s) { return from(X, k, tj + s); });
#pragma unroll
    for (int r = 0; r < 4; ++r) lds(ti + 4 * r + q, tj + c) = v[r];
  }
  __syncthreads();
  // A = X (F X), symmetric: its lower triangle, mirrored
  double4_t res[kFull];
  auto lower = [&](auto&& tile) {
#pragma unroll
    for (int u = 0; u < kFull; ++u) {
      const int t = wave + u * W;
      if (t < ntri) {
        int i, j;
        triangle(t, &i, &j);
        tile(u, kTile * i, kTile * j);
      }
    }
  };
  lower([&](int u, int ti, int tj) {
    res[u] = tile_product(
        N, lane, [&](int r, int k) { return from(X, ti + r, k); },
        [&](int k, int s) { return lds(k, tj + s); });
  });
  __syncthreads();
  lower([&](int u, int ti, int tj) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = ti + 4 * r + q, j = tj + c;
      if (ti != tj || i >= j) {
        lds(i, j) = res[u][r];
        lds(j, i) = res[u][r];
      }
    }
  });
  __syncthreads();
  // Gershgorin's bounds
  double lo = HUGE_VAL, hi = -HUGE_VAL;
  for (int r = wave; r < n; r += W) {
    double s = 0.0;
    for (int j = lane; j < n; j += 64) s += j == r ? 0.0 : fabs(lds(r, j));
    s = sum64(s);
    lo = fmin(lo, lds(r, r) - s);
    hi = fmax(hi, lds(r, r) + s);
  }
  if (lane == 0) {
    red[wave] = lo;
    red[kMaxWaves + wave] = hi;
  }
  __syncthreads();
  for (int w = 0; w < W; ++w) {
    lo = fmin(lo, red[w]);
    hi = fmax(hi, red[kMaxWaves + w]);
  }
  __syncthreads();
  // P_0 (padding rows and columns zero, and zero they stay); its trace
  const bool all = nocc >= n;  // every orbital occupied: P = 1
  const double inv = 1.0 / (hi - lo);
  double tr = 0.0;
  for (int k = threadIdx.x; k < N * N; k += blockDim.x) {
    const int r = k / N, s = k - r * N;
    double v = 0.0;
    if (r < n && s < n) v = all ? (r == s ? 1.0 : 0.0) : ((r == s ? hi : 0.0) - lds(r, s)) * inv;
    lds(r, s) = v;
    if (r == s) tr += v;
  }
  tr = sum64(tr);
  if (lane == 0) red[wave] = tr;
  __syncthreads();
  tr = 0.0;
  for (int w = 0; w < W; ++w) tr += red[w];
  int left = all ? 0 : -1;  // steps left once tr(P - P^2) is small
  bool good = all;
  for (int step = 0; step < kMaxSteps && left != 0; ++step) {
    double t2 = 0.0;
    lower([&](int u, int ti, int tj) {
      res[u] = tile_product(
          N, lane, [&](int r, int k) { return lds(ti + r, k); },
          [&](int k, int s) { return lds(tj + s, k); });
      if (ti == tj) {
#pragma unroll
        for (int r = 0; r < 4; ++r) t2 += 4 * r + q == c ? res[u][r] : 0.0;
      }
    });
    t2 = sum64(t2);
    __syncthreads();  // red of the last step has been read
    if (lane == 0) red[wave] = t2;
    __syncthreads();  // and so has P
    t2 = 0.0;
    for (int w = 0; w < W; ++w) t2 += red[w];
    const double idem = tr - t2;  // sum of lambda (1 - lambda)
    if (!(fabs(idem) < HUGE_VAL)) break;  // a non-finite F
    bool square = fabs(t2 - nocc) < fabs(2.0 * tr - t2 - nocc);
    if (left > 0) {
      square = left == 2;
      --left;
    } else if (idem < kIdempotent) {
      // the last pair, P^2 then 2P - P^2, takes both ends to rounding
      if (fabs(tr - nocc) > 1e-3) break;
      good = true;
      left = 1;
      square = true;
    }
    lower([&](int u, int ti, int tj) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = ti + 4 * r + q, j = tj + c;
        if (ti != tj || i >= j) {
          const double v = square ? res[u][r] : 2.0 * lds(i, j) - res[u][r];
          lds(i, j) = v;
          lds(j, i) = v;
        }
      }
    });
    tr = square ? t2 : 2.0 * tr - t2;
    __syncthreads();
  }
  good = good && left == 0;
  if (threadIdx.x == 0) {
    flag[2 * m] = 0.5;
    flag[2 * m + 1] = good ? 0.0 : 1.0;
  }
  if (!good) return;  // block-uniform
  // A = P X, then D = X A
#pragma unroll
  for (int u = 0; u < kFull; ++u) {
    const int t = wave + u * W;
    if (t < nfull) {
      const int ti = kTile * (t / nt), tj = kTile * (t % nt);
      res[u] = tile_product(
          N, lane, [&](int r, int k) { return lds(ti + r, k); },
          [&](int k, int s) { return from(X, k, tj + s); });
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kFull; ++u) {
    const int t = wave + u * W;
    if (t < nfull) {
      const int ti = kTile * (t / nt), tj = kTile * (t % nt);
#pragma unroll
      for (int r = 0; r < 4; ++r) lds(ti + 4 * r + q, tj + c) = res[u][r];
    }
  }
  __syncthreads();
  lower([&](int, int ti, int tj) {
    const double4_t v = tile_product(
        N, lane, [&](int r, int k) { return from(X, ti + r, k); },
        [&](int k, int s) { return lds(k, tj + s); });
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = ti + 4 * r + q, j = tj + c;
      if (i < n && j < n && (ti != tj || i >= j)) {
        D[static_cast<size_t>(i) * ld + j] = v[r];
        D[static_cast<size_t>(j) * ld + i] = v[r];
      }
    }
  });
}

}  // namespace

// count matrices of leading dimension ld (and stride ld^2), the largest of size
// nmax <= kDensityMaxN; nb, nocc per matrix or null (n = nmax, nocc1).  flag:
// two doubles per matrix.
hipError_t density_small_launch(const double* F, const double* X, int ld, int nmax, const int* nb,
                                int nocc1, const int* nocc, int count, double* D, double* flag,
                                hipStream_t s) {
  if (count <= 0) return hipSuccess;
  if (nmax <= 0 || nmax > kDensityMaxN || ld < nmax) return hipErrorInvalidValue;
  const int nt = (nmax + kTile - 1) / kTile, N = nt * kTile;
  // a wave holds at most kFull tiles of a product
  const int waves = std::min(kMaxWaves, nt * nt);
  const size_t lds = sizeof(double) * N * (N + 2);
  hipLaunchKernelGGL(density_small_kernel, dim3(count), dim3(64 * waves), lds, s, F, X,
                     static_cast<size_t>(ld) * ld, ld, nmax, nb, nocc1, nocc, D, flag);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Larger matrices: the same scheme, one launch to a step.
// ---------------------------------------------------------------------------

namespace {

// What bounds a step is the latency of a launch on data that other dies wrote,
// not its work (n = 416: 72 MFLOP in the lower triangle): a workgroup forms a
// 32 x 32 tile of P^2, a wave 16 x 16 of it, straight from memory -- P is
// symmetric, so both operands are rows, and a lane's 32 consecutive bytes of
// each are four MFMAs' k (any order of k will do, the same for both) -- with
// the next 64 columns in flight.  (Four waves to each 16 x 16, sharing k, and
// reads that wait for no state took as long.)  tr(P) and tr(P^2) = sum P_ij^2 of
// a step's result are summed as it is written and read by the next step, which
// can so choose its polynomial before its product: one launch, no host, no
// separate trace pass.  Per step: 15.6 us at n = 416, 9.2 at n = 156, where two
// library products, the traces and the update of the cubic scheme took 42 and
// 23; a density takes 51 and 39 steps for 34 and 24, without a host read for
// every step where no graph replays them.  The matrices have a leading
// dimension of ldp, a multiple of 64; padding is and stays zero.
constexpr int kSp2Tile = 32;

struct Sp2State {
  int left;  // steps to go once tr(P - P^2) is small; 0: done, -1: not yet
  int buf;   // which of the two buffers holds P
};

__device__ __forceinline__ double2 sum_block(double2 v, double2* red) {
  v.x = sum64(v.x);
  v.y = sum64(v.y);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double2 t = red[0];
  for (int w = 1; w < 4; ++w) {
    t.x += red[w].x;
    t.y += red[w].y;
  }
  __syncthreads();
  return t;
}

__device__ __forceinline__ void sp2_tile(int t, int* i, int* j) {
  int r = static_cast<int>((sqrtf(8.0f * static_cast<float>(t) + 1.0f) - 1.0f) * 0.5f);
  while ((r + 1) * (r + 2) / 2 <= t) ++r;
  while (r * (r + 1) / 2 > t) --r;
  *i = r;
  *j = t - r * (r + 1) / 2;
}

// Gershgorin's bounds of the rows, P_0 in the first buffer, its sums.  Every
// workgroup reduces the n rows' bounds (lo, hi) itself.
__global__ __launch_bounds__(256) void sp2_start_kernel(const double* __restrict__ F, int n,
                                                        const double* __restrict__ lo,
                                                        const double* __restrict__ hi, int ldp,
                                                        double* __restrict__ P,
                                                        double2* __restrict__ part,
                                                        Sp2State* __restrict__ state) {
  __shared__ double2 red[4];
  __shared__ double bl[4], bh[4];
  double l = HUGE_VAL, h = -HUGE_VAL;
  for (int k = threadIdx.x; k < n; k += 256) {
    l = fmin(l, lo[k]);
    h = fmax(h, hi[k]);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    l = fmin(l, __shfl_xor(l, off, 64));
    h = fmax(h, __shfl_xor(h, off, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    bl[threadIdx.x >> 6] = l;
    bh[threadIdx.x >> 6] = h;
  }
  __syncthreads();
  for (int w = 0; w < 4; ++w) {
    l = fmin(l, bl[w]);
    h = fmax(h, bh[w]);
  }
  const double inv = 1.0 / (h - l);
  int ti, tj;
  sp2_tile(blockIdx.x, &ti, &tj);
  double2 s = make_double2(0.0, 0.0);
  for (int k = threadIdx.x; k < kSp2Tile * kSp2Tile; k += 256) {
    const int i = ti * kSp2Tile + k / kSp2Tile, j = tj * kSp2Tile + k % kSp2Tile;
    if (i < j) continue;
    double v = 0.0;
    if (i < n && j < n) {
      // F' is symmetric but for the last bits of its products
      const double f = 0.5 * (F[static_cast<size_t>(i) * n + j] + F[static_cast<size_t>(j) * n + i]);
      v = ((i == j ? h : 0.0) - f) * inv;
    }
    P[static_cast<size_t>(i) * ldp + j] = v;
    P[static_cast<size_t>(j) * ldp + i] = v;
    if (i == j) s.x += v;
    s.y += (i == j ? 1.0 : 2.0) * v * v;
  }
  s = sum_block(s, red);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
  if (blockIdx.x == 0 && threadIdx.x == 0) state[0] = Sp2State{-1, 0};
}

// Step `step`: reads state[step] and part[step][ntri], writes state[step + 1],
// part[step + 1][ntri] and coef[2 step + 1] = tr(P - P^2) (0 once done).
__global__ __launch_bounds__(256) void sp2_step_kernel(double* __restrict__ P0,
                                                       double* __restrict__ P1, int ldp, int nocc,
                                                       int step, int ntri,
                                                       double2* __restrict__ part,
                                                       Sp2State* __restrict__ state,
                                                       double* __restrict__ coef) {
  __shared__ double2 red[4];
  const Sp2State st = state[step];
  const bool first = blockIdx.x == 0 && threadIdx.x == 0;
  if (st.left == 0) {  // done: P stays where it is
    if (first) {
      state[step + 1] = st;
      coef[2 * step] = 0.5;
      coef[2 * step + 1] = 0.0;
    }
    return;
  }
  double2 t = make_double2(0.0, 0.0);
  const double2* __restrict__ pin = part + static_cast<size_t>(step) * ntri;
  for (int k = threadIdx.x; k < ntri; k += 256) {
    t.x += pin[k].x;
    t.y += pin[k].y;
  }
  t = sum_block(t, red);
  const double idem = t.x - t.y;
  bool square = fabs(t.y - nocc) < fabs(2.0 * t.x - t.y - nocc);
  int left = st.left;
  if (left > 0) {
    square = false;
    --left;
  } else if (idem < kIdempotent && fabs(t.x - nocc) < 1e-3) {
    left = 1;  // the last pair: P^2, then 2P - P^2
    square = true;
  }
  if (first) {
    state[step + 1] = Sp2State{left, st.buf ^ 1};
    coef[2 * step] = 0.5;
    // idempotent at another trace than nocc does not count as converged
    coef[2 * step + 1] = left < 0 && idem < kIdempotent ? 1.0 : idem;
  }
  const double* __restrict__ P = st.buf ? P1 : P0;
  double* __restrict__ Q = st.buf ? P0 : P1;
  int ti, tj;
  sp2_tile(blockIdx.x, &ti, &tj);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int c = lane & 15, q = lane >> 4;
  const int i0 = ti * kSp2Tile + 16 * (wave >> 1), j0 = tj * kSp2Tile + 16 * (wave & 1);
  const double* __restrict__ a = P + static_cast<size_t>(i0 + c) * ldp + 4 * q;
  const double* __restrict__ b = P + static_cast<size_t>(j0 + c) * ldp + 4 * q;
  double4_t acc = {0.0, 0.0, 0.0, 0.0};
  double2 xa[8], xb[8], ya[8], yb[8];
  auto load = [&](int k, double2 (&u)[8], double2 (&v)[8]) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      u[2 * w] = *reinterpret_cast<const double2*>(a + k + 16 * w);
      u[2 * w + 1] = *reinterpret_cast<const double2*>(a + k + 16 * w + 2);
      v[2 * w] = *reinterpret_cast<const double2*>(b + k + 16 * w);
      v[2 * w + 1] = *reinterpret_cast<const double2*>(b + k + 16 * w + 2);
    }
  };
  auto multiply = [&](const double2 (&u)[8], const double2 (&v)[8]) {
#pragma unroll
    for (int w = 0; w < 8; ++w) {
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(u[w].x, v[w].x, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(u[w].y, v[w].y, acc, 0, 0, 0);
    }
  };
  load(0, xa, xb);
  for (int k = 0; k < ldp; k += 128) {
    const bool more = k + 64 < ldp;
    if (more) load(k + 64, ya, yb);
    multiply(xa, xb);
    if (k + 128 < ldp) load(k + 128, xa, xb);
    if (more) multiply(ya, yb);
  }
  double2 s = make_double2(0.0, 0.0);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = i0 + 4 * r + q, j = j0 + c;
    if (i < j) continue;
    const double v = square ? acc[r] : 2.0 * P[static_cast<size_t>(i) * ldp + j] - acc[r];
    Q[static_cast<size_t>(i) * ldp + j] = v;
    Q[static_cast<size_t>(j) * ldp + i] = v;
    if (i == j) s.x += v;
    s.y += (i == j ? 1.0 : 2.0) * v * v;
  }
  s = sum_block(s, red);
  if (threadIdx.x == 0) part[static_cast<size_t>(step + 1) * ntri + blockIdx.x] = s;
}

// The n x n projector out of the buffer that holds it; out[0] = 1 where it is
// one (0: the steps were not enough).
__global__ __launch_bounds__(256) void sp2_finish_kernel(const double* __restrict__ P0,
                                                         const double* __restrict__ P1, int ldp,
                                                         int n, const Sp2State* __restrict__ state,
                                                         double* __restrict__ P,
                                                         double* __restrict__ out) {
  const Sp2State st = *state;
  const double* __restrict__ S = st.buf ? P1 : P0;
  const int i = blockIdx.x;
  for (int j = threadIdx.x; j < n; j += 256)
    P[static_cast<size_t>(i) * n + j] = S[static_cast<size_t>(i) * ldp + j];
  if (i == 0 && threadIdx.x == 0) out[0] = st.left == 0 ? 1.0 : 0.0;
}

int sp2_ntri(int n) {
  const int nt = (n + kSp2Tile - 1) / kSp2Tile;
  return nt * (nt + 1) / 2;
}
int sp2_ld(int n) { return (n + 63) / 64 * 64; }

}  // namespace

// Workspace of a purification of at most `steps` steps, in doubles: two
// buffers, the sums and the states.
size_t sp2_workspace(int n, int steps) {
  const size_t ld = sp2_ld(n);
  return 2 * ld * ld + 2 * static_cast<size_t>(steps + 1) * sp2_ntri(n) + (steps + 1) + 1;
}

namespace {

struct Sp2Work {
  double *P0, *P1;
  double2* part;
  Sp2State* state;
};
Sp2Work sp2_split(double* work, int n, int steps) {
  const size_t ld = sp2_ld(n);
  Sp2Work w;
  w.P0 = work;
  w.P1 = work + ld * ld;
  w.part = reinterpret_cast<double2*>(work + 2 * ld * ld);
  w.state = reinterpret_cast<Sp2State*>(w.part + static_cast<size_t>(steps + 1) * sp2_ntri(n));
  return w;
}

}  // namespace

// P_0 from F' (n x n) and its rows' bounds; the workspace's padding must be
// zero (it stays so: one fill when the workspace is made).
hipError_t sp2_start_launch(const double* Fp, int n, const double* lo, const double* hi,
                            double* work, int steps, hipStream_t s) {
  const Sp2Work w = sp2_split(work, n, steps);
  hipLaunchKernelGGL(sp2_start_kernel, dim3(sp2_ntri(n)), dim3(256), 0, s, Fp, n, lo, hi,
                     sp2_ld(n), w.P0, w.part, w.state);
  return hipGetLastError();
}

hipError_t sp2_step_launch(double* work, int n, int nocc, int steps, int step, double* coef,
                           hipStream_t s) {
  if (step < 0 || step >= steps) return hipErrorInvalidValue;
  const Sp2Work w = sp2_split(work, n, steps);
  hipLaunchKernelGGL(sp2_step_kernel, dim3(sp2_ntri(n)), dim3(256), 0, s, w.P0, w.P1, sp2_ld(n),
                     nocc, step, sp2_ntri(n), w.part, w.state, coef);
  return hipGetLastError();
}

hipError_t sp2_finish_launch(double* work, int n, int steps, int step, double* P, double* out,
                             hipStream_t s) {
  const Sp2Work w = sp2_split(work, n, steps);
  hipLaunchKernelGGL(sp2_finish_kernel, dim3(n), dim3(256), 0, s, w.P0, w.P1, sp2_ld(n), n,
                     w.state + step, P, out);
  return hipGetLastError();
}

}  // namespace rchem
