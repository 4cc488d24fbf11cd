// Streaming ERI kernel for the classes whose contracted accumulators do not fit
// one lane (total angular momentum L >= 5: (dp|pp) ... (dd|dd)): their bounds,
// tensors and single quartets, and their Fock builds where the partwise kernel
// (eri_part.hpp) is switched off.
//
// One wavefront evaluates one contracted shell quartet at a time, one
// primitive quartet per lane (64 at a time; a quartet with more runs in
// passes).  Each lane forms its primitive quartet's prefactors and Boys
// function as the per-lane kernels do, then runs the class's straight-line
// Head-Gordon--Pople VRR (EriClass::vrr_stream, generated by gen_eri.py) and
// hands every target [e0|f0]^(0) over as soon as it is formed: groups of 16
// targets are summed over the wave through an LDS transpose (each lane writes
// its 16 values as one row, four lanes per target add up a quarter of the
// rows each, two shuffles finish the sum) into the quartet's contracted
// accumulators in LDS.  A lane therefore keeps no accumulators, only the VRR
// values still to be used.  The horizontal recurrence and the outputs are the
// wave-cooperative kernel's (eri_coop.hpp, tables from gen_eri_prog.py).
// The recurrences are chgp.c:412-586 (VRR) and chgp.c:44-135 (HRR).
#pragma once
#include <utility>

#include "eri_common.hpp"
#include "eri_coop.hpp"

namespace rchem {

constexpr int kStreamRedRow = 18;   // doubles per lane row of the transpose (16 + 2 pad)

// LDS doubles of one wave: the accumulator / HRR buffer and the transpose.
__host__ __device__ inline size_t stream_wave_doubles(const GenericProgram& p) {
  return static_cast<size_t>(p.nh) + 64 * kStreamRedRow;
}

template <int NACC>
struct StreamAcc {
  double buf[16];
  double* red;  // this wave's transpose rows, 64 x kStreamRedRow
  double* acc;  // this wave's contracted accumulators (NACC)
  int lane;

  template <int K>
  __device__ __forceinline__ void put(double v) {
    buf[K & 15] = v;
    if constexpr ((K & 15) == 15 || K == NACC - 1) flush<K & ~15, (K & 15) + 1>();
  }

  // acc[BASE + i] += sum over the wave of buf[i], i < N
  template <int BASE, int N>
  __device__ __forceinline__ void flush() {
    double* row = red + lane * kStreamRedRow;
#pragma unroll
    for (int i = 0; i < N; ++i) row[i] = buf[i];
    wsync<2>();
    const int i = lane & 15, quarter = lane >> 4;
    double s = 0.0;
    if (i < N) {
      const double* col = red + quarter * 16 * kStreamRedRow + i;
#pragma unroll
      for (int j = 0; j < 16; ++j) s += col[j * kStreamRedRow];
    }
    s += __shfl_xor(s, 16, 64);
    s += __shfl_xor(s, 32, 64);
    if (lane < N) acc[BASE + lane] += s;
    wsync<2>();
  }
};

// The streamed VRR of class C in its parts (each part a subset of the targets,
// recomputing the intermediates it needs), one after the other.
template <typename C, int PART, typename SA>
__device__ __forceinline__ void stream_parts(const double* __restrict__ G, double PAx, double PAy,
                                             double PAz, double WPx, double WPy, double WPz,
                                             double QCx, double QCy, double QCz, double WQx,
                                             double WQy, double WQz, double oo2z, double oo2e,
                                             double oo2ze, double roz, double roe, SA& acc) {
  C::template vrr_stream<PART>(G, PAx, PAy, PAz, WPx, WPy, WPz, QCx, QCy, QCz, WQx, WQy, WQz,
                               oo2z, oo2e, oo2ze, roz, roe, acc);
  if constexpr (PART + 1 < C::NSTREAM)
    stream_parts<C, PART + 1>(G, PAx, PAy, PAz, WPx, WPy, WPz, QCx, QCy, QCz, WQx, WQy, WQz,
                              oo2z, oo2e, oo2ze, roz, roe, acc);
}

// W waves per workgroup; persistent over tiles when the launch has a device
// tile range, else one tile per wave.  LDS: the Boys block of order L, the
// HRR and output tables when stage_coop (else they are read from device
// memory), then per wave stream_wave_doubles(p).
// The pair, primitive and tile arrays come as separate restrict-qualified
// arguments: nothing the kernel stores aliases them, so the wave-uniform
// records (tile, bra and ket pair) are read through the scalar unit, whose
// waits do not queue behind the vector memory operations (atomics) of the
// previous quartet.
template <int LA, int LB, int LC, int LD, int MODE, int W>
__global__ __launch_bounds__(64 * W, 1) void eri_stream_kernel(
    const EriArgs a, const GenericProgram p, int stage_coop, const PairRec* __restrict__ pairs,
    const PrimRec* __restrict__ prims, const Tile* __restrict__ tiles) {
  using C = EriClass<LA, LB, LC, LD>;
  constexpr int L = C::L;
  extern __shared__ double lds[];
  double* boys_tab = lds;
  stage_boys<L>(boys_tab, a.boys_table);
  char* after_boys = reinterpret_cast<char*>(lds + boys_stage_size(L));
  const CoopTables tbl = coop_tables(p, after_boys, stage_coop != 0);
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  double* H = reinterpret_cast<double*>(after_boys + (stage_coop ? coop_table_bytes(p) : 0)) +
              static_cast<size_t>(wave) * stream_wave_doubles(p);
  double* red = H + p.nh;
  double* dl = red;  // the density blocks of the epilogue reuse the transpose rows
  int begin, end;
  if (a.tile_range) {
    begin = a.tile_range[0];
    end = a.tile_range[1];
  } else {
    begin = 0;
    end = a.ntiles;
  }
  for (int ti = begin + static_cast<int>(blockIdx.x) * W + wave; ti < end;
       ti += static_cast<int>(gridDim.x) * W) {
    const Tile t = tiles[__builtin_amdgcn_readfirstlane(ti)];
    if (MODE == kModeJK && !first_part(t.pad)) continue;  // the first part does the whole quartet
    for (int qi = 0; qi < t.count; ++qi) {
      const int kidx = __builtin_amdgcn_readfirstlane(t.ket0 + qi);
      const int bidx = __builtin_amdgcn_readfirstlane((MODE == kModeDiag) ? kidx : t.bra);
      const PairRec bp = pairs[bidx];
      const PairRec kp = pairs[kidx];
      wsync<2>();  // the previous quartet's outputs have been read
      for (int k = lane; k < C::NACC; k += 64) H[k] = 0.0;
      const double ACx = bp.A[0] - kp.A[0], ACy = bp.A[1] - kp.A[1], ACz = bp.A[2] - kp.A[2];
      const int knp = kp.np;
      const int npq = bp.np * knp;
      StreamAcc<C::NACC> sa;
      sa.red = red;
      sa.acc = H;
      sa.lane = lane;
      for (int base = 0; base < npq; base += 64) {
        const int j = base + lane;
        const bool valid = j < npq;
        const int ib = valid ? j / knp : 0, ik = valid ? j % knp : 0;
        const PrimRec pb = prims[bp.p0 + ib * bp.ps];
        const PrimRec pk = prims[kp.p0 + ik * kp.ps];
        const double zb = pb.zeta, zk = pk.zeta;
        const double rs = fast_rsqrt(zb + zk);  // (zeta + eta)^(-1/2)
        const double ooze = rs * rs;
        const double roz = zk * ooze, roe = zb * ooze;
        // P - Q = (P - A) - ((Q - C) - (A - C))
        const double PQx = pb.pax - (pk.pax - ACx);
        const double PQy = pb.pay - (pk.pay - ACy);
        const double PQz = pb.paz - (pk.paz - ACz);
        const double T = zb * roz * (PQx * PQx + PQy * PQy + PQz * PQz);
        double F[L + 1];
        boys<L, kBoysExact, double, false>(T, boys_tab, F);
        // a lane past the quartet's primitive quartets adds zeros (the VRR is
        // linear in G)
        const double pref = valid ? pb.kab * pk.kab * rs : 0.0;
        double G[L + 1];
#pragma unroll
        for (int m = 0; m <= L; ++m) G[m] = pref * F[m];
        stream_parts<C, 0>(G, pb.pax, pb.pay, pb.paz, -roz * PQx, -roz * PQy, -roz * PQz,
                           pk.pax, pk.pay, pk.paz, roe * PQx, roe * PQy, roe * PQz, pb.oo2z,
                           pk.oo2z, 0.5 * ooze, roz, roe, sa);
      }
      wsync<2>();
      coop_hrr<2>(tbl, p.nhgroups, H, bp.AB[0], bp.AB[1], bp.AB[2], kp.AB[0], kp.AB[1],
                  kp.AB[2], lane);
      epilogue<2, MODE>(a, p, tbl, t, bidx, kidx, bp, kp, H, dl, lane);
    }
  }
}

// blocks: with a device tile range, the number of 4-wave blocks the per-lane
// kernels would use (as many waves here); without one, one wave per tile.
// Four waves per workgroup, or two where four do not fit the LDS; the HRR and
// output tables in LDS where they fit beside them.
template <int LA, int LB, int LC, int LD, int MODE>
hipError_t eri_stream_launch(const EriArgs& a, const GenericProgram& p, int blocks,
                             hipStream_t s, size_t lds_limit) {
  using C = EriClass<LA, LB, LC, LD>;
  if (p.la != LA || p.lb != LB || p.lc != LC || p.ld != LD || p.nacc != C::NACC ||
      p.nh < p.nacc || p.centre >= 0)
    return hipErrorInvalidValue;
  auto bytes = [&](int W, bool sc) {
    return sizeof(double) * (boys_stage_size(C::L) + W * stream_wave_doubles(p)) +
           (sc ? coop_table_bytes(p) : 0);
  };
  int W = 0, sc = 0;
  for (const auto& c : {std::make_pair(4, 1), std::make_pair(2, 1), std::make_pair(4, 0),
                        std::make_pair(2, 0)})
    if (bytes(c.first, c.second != 0) <= lds_limit) {
      W = c.first;
      sc = c.second;
      break;
    }
  if (W == 0) return hipErrorInvalidValue;
  const size_t lds = bytes(W, sc != 0);
  unsigned waves;
  if (a.tile_range) {
    if (blocks <= 0) return hipSuccess;
    waves = static_cast<unsigned>(blocks) * 4u;
  } else {
    if (a.ntiles <= 0) return hipSuccess;
    waves = static_cast<unsigned>(a.ntiles);
  }
  const unsigned grid = (waves + W - 1) / W;
  if (W == 4)
    hipLaunchKernelGGL((eri_stream_kernel<LA, LB, LC, LD, MODE, 4>), dim3(grid), dim3(256), lds,
                       s, a, p, sc, a.pairs, a.prims, a.tiles);
  else
    hipLaunchKernelGGL((eri_stream_kernel<LA, LB, LC, LD, MODE, 2>), dim3(grid), dim3(128), lds,
                       s, a, p, sc, a.pairs, a.prims, a.tiles);
  return hipGetLastError();
}

}  // namespace rchem
