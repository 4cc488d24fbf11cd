// Fock-build kernel of the classes whose contracted accumulators exceed one
// lane (total angular momentum L >= 5: (dp|pp), (dp|dp) ... (dd|dd)).
//
// A workgroup takes the tiles of a chunk in turn (one bra pair against 64 ket
// pairs, one contracted quartet to a lane, as in the per-lane kernels: every
// lane busy with a primitive quartet of its own, the bra's records through the
// scalar unit).  But its waves divide the class's targets [e0|f0] among them:
// each runs the primitive loops for its parts, whose accumulators and VRR values
// fit its registers, and leaves the sums in the workgroup's slab of memory
// ([target][quartet]; 74 to 492 KB, mostly in the caches).  After a barrier the
// waves divide the bra's component pairs (ab|: a lane forms [ab|f0) from the slab
// by the bra's horizontal recurrence in closed form, (ab|cd) by the ket's, and
// digests them before the next ab, so that one ab's integrals are live at a time.
// K goes to rows of a and b in LDS, the ket's Coulomb sums of all waves to LDS
// too: with every sum an atomic in memory the kernels ran at 40 to 60e9 atomics/s
// whatever their arithmetic ((dp|pp), in eight parts then, 47.5 ms against 19.2,
// (dd|dp) 29 against 18.5).
//
// The per-lane kernels spilled (512 registers and up to 1.2 KB a lane), and the
// streaming kernel (eri_stream.hpp: one wave to a quartet, lanes on its
// primitives, every target summed over the wave through LDS, the recurrence and
// the digestion of one quartet at a time by tables) waited for LDS with one wave
// on a SIMD: VALU 0.22-0.31 of the cycles; here 0.64-0.75 (0.52 in
// (dd|dd), one wave on a SIMD), which is the bound,
// with the product and Boys work that each part repeats (130 of 535 vector
// instructions of a (dp|dp) part) the larger part of the excess.  A build of 210
// s/p/d shells of 3 primitives (n = 430), ms, per-lane or streaming and now:
// (dp|pp) 17.6, 13.5; (dp|dp) 68.6, 14.2; (dd|ds) 20.5, 7.0; (dd|pp) 42.0, 7.6;
// (dd|dp) 55.0, 14.6; (dd|dd) 32.0, 6.5.  The build: 298 -> 132 on one box (108 to
// 132 over boxes).
//
// A tile is one lane's chain of primitive quartets, so where a class has fewer
// tiles than the chip workgroups they are split over the primitives as in the
// per-lane kernels (PrimSplit, part_split_limit).
// The recurrences are chgp.c:412-586 (VRR) and chgp.c:44-135 (HRR).
#pragma once
#include "eri_common.hpp"

namespace rchem {

// c AB_x^px AB_y^py AB_z^pz [e 0|
struct PartTerm {
  int e, px, py, pz;
  double c;
};

template <int LA, int LB, int LC, int LD>
struct EriParts;

#include "generated/eri_parts.inc"

// The targets of part PART of the lane's quartet, contracted, into the slab.
template <int LA, int LB, int LC, int LD, int PART>
__device__ __forceinline__ void part_compute(const TileSrc& src, const PairRec& bp, const Tile& t,
                                             int lane, int lane_off,
                                             const double* __restrict__ boys_tab,
                                             const PrimRec* __restrict__ prim, double* slab) {
  using C = EriParts<LA, LB, LC, LD>;
  constexpr int L = LA + LB + LC + LD;
  constexpr int N = C::begin(PART + 1) - C::begin(PART);
  double acc[N];
#pragma unroll
  for (int i = 0; i < N; ++i) acc[i] = 0.0;
  const KetPlanes& k = src.ket;
  const double2 g0 = (k.geo + t.ket0)[lane_off], g1 = (k.geo + k.npairs + t.ket0)[lane_off];
  const double ACx = bp.A[0] - g0.x, ACy = bp.A[1] - g0.y, ACz = bp.A[2] - g1.x;
  const PairRec& k0 = src.pairs[t.ket0];
  const int kps = k0.ps, row = k0.p0;
  const PrimRec* __restrict__ bprim = prim + bp.p0;
  const int bps = bp.ps;
  int i0 = 0, i1 = bp.np, j0 = 0, j1 = k0.np;
  if (t.pad != 0) {  // a part of the quartets' primitives (PrimSplit)
    i0 = t.pad & 255;
    i1 = (t.pad >> 8) & 255;
    j0 = (t.pad >> 16) & 255;
    j1 = (t.pad >> 24) & 255;
  }
  for (int j = j0; j < j1; ++j) {
    const PrimRec pk = load_ket_prim<double, true>(k, prim, row + j * kps, lane_off);
    const double QAx = pk.pax - ACx, QAy = pk.pay - ACy, QAz = pk.paz - ACz;
    for (int i = i0; i < i1; ++i) {
      const PrimRec pb = bprim[i * bps];
      const double rs = fast_rsqrt(pb.zeta + pk.zeta);  // (zeta + eta)^(-1/2)
      const double ooze = rs * rs;
      const double roz = pk.zeta * ooze, roe = pb.zeta * ooze;
      const double PQx = pb.pax - QAx, PQy = pb.pay - QAy, PQz = pb.paz - QAz;
      const double T = pb.zeta * roz * (PQx * PQx + PQy * PQy + PQz * PQz);
      double F[L + 1];
      boys<L, kBoysExact, double, false>(T, boys_tab, F);
      const double pref = pb.kab * pk.kab * rs;
      double G[L + 1];
#pragma unroll
      for (int m = 0; m <= L; ++m) G[m] = pref * F[m];
      C::template vrr<PART>(G, pb.pax, pb.pay, pb.paz, -roz * PQx, -roz * PQy, -roz * PQz, pk.pax,
                            pk.pay, pk.paz, roe * PQx, roe * PQy, roe * PQz, pb.oo2z, pk.oo2z,
                            0.5 * ooze, roz, roe, acc);
    }
  }
  unsigned lo = 8u * static_cast<unsigned>(lane);
  asm volatile("" : "+v"(lo), "+s"(slab));  // the addresses are formed here, not kept over the loops
#pragma unroll
  for (int i = 0; i < N; ++i) *at_off(slab + (C::begin(PART) + i) * 64, lo) = acc[i];
}

// Doubles of the Boys table's stage, to an even count.
template <int L>
__host__ __device__ constexpr int part_boys() {
  return (boys_stage_size(L) + 1) / 2 * 2;
}

// Parts wave, wave + W, ... (the wave's index is uniform).
template <int LA, int LB, int LC, int LD, int PART>
__device__ __forceinline__ void part_run(int wave, const TileSrc& src, const PairRec& bp,
                                         const Tile& t, int lane, int lane_off,
                                         const double* __restrict__ boys_tab,
                                         const PrimRec* __restrict__ prim, double* slab) {
  using C = EriParts<LA, LB, LC, LD>;
  if constexpr (PART < C::NPART) {
    if (PART % C::W == wave)
      part_compute<LA, LB, LC, LD, PART>(src, bp, t, lane, lane_off, boys_tab, prim, slab);
    part_run<LA, LB, LC, LD, PART + 1>(wave, src, bp, t, lane, lane_off, boys_tab, prim, slab);
  }
}

__device__ __forceinline__ double part_power(double x, int p) {
  return p == 0 ? 1.0 : p == 1 ? x : x * x;
}

// ROWS: where the digestion's rows of the bra's functions are.  0: K in
// memory, by atomics, and D there, tile after tile.  1: K rows in LDS, flushed
// once a chunk of tiles of one bra (EriArgs::chunks).  2: D rows there as well.
template <int LA, int LB, int LC, int LD, int ROWS,
          int THREADS = 64 * EriParts<LA, LB, LC, LD>::W,
          int MINW = EriParts<LA, LB, LC, LD>::MINW>
__global__ __launch_bounds__(THREADS, MINW) void eri_part_kernel(
    const EriArgs a, double* slabs, const PrimRec* __restrict__ prims,
    const double* __restrict__ D, const double* __restrict__ Dp,
    const PairRec* __restrict__ pairs, const Tile* __restrict__ tiles,
    const Chunk* __restrict__ chunks, const double2* __restrict__ kgeo,
    const int2* __restrict__ kfn, const double2* __restrict__ kprim) {
  using C = EriParts<LA, LB, LC, LD>;
  constexpr int L = LA + LB + LC + LD, W = C::W, NF = C::NF;
  constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
  constexpr int NACC = EriClass<LA, LB, LC, LD>::NACC;
  extern __shared__ __align__(16) double part_lds[];
  const TileSrc src{pairs, tiles, KetPlanes{kgeo, kfn, kprim, nullptr, nullptr, a.ket.npairs,
                                            a.ket.nprims}};
  stage_boys<L>(part_lds, a.boys_table);
  double* const jq = part_lds + part_boys<L>();  // the ket's Coulomb sums [k][quartet]
  double* const jb = jq + NC * ND * 64;          // the bra's
  double* const krows = jb + NA * NB;
  double* slab = slabs + static_cast<size_t>(blockIdx.x) * NACC * 64;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = a.nbf, kw = a.kw;
  double* const drows = krows + (NA + NB) * kw;
  for (int k = tid; k < NC * ND * 64; k += THREADS) jq[k] = 0.0;
  const int begin = ROWS ? a.chunk_range[0] : a.tile_range ? a.tile_range[0] : 0;
  const int end = ROWS ? a.chunk_range[1] : a.tile_range ? a.tile_range[1] : a.ntiles;
  __syncthreads();  // the staged table is complete before a wave's first lookup
  __shared__ int s_next[2];  // by turns: a chunk may have no barrier but its last
  int turn = 0;
  for (int u = begin + static_cast<int>(blockIdx.x); u < end;) {  // block-uniform
    int next = 0;
    if (ROWS && tid == 0) next = atomicAdd(a.next, 1);  // awaited at the chunk's end
    const Chunk ch = ROWS ? chunks[u] : Chunk{tiles[u].bra, u, u + 1, 0};
    const int kc0 = ROWS && a.pair_kc0 ? a.pair_kc0[ch.bra] : 0;
    const PairRec bp = pairs[ch.bra];
    const int fa = bp.fa, fb = bp.fb;
    // cleared by the threads that flushed them: no barrier between
    if (tid < NA * NB) jb[tid] = 0.0;
    if constexpr (ROWS > 0) {
      for (int r = 0; r < NA + NB; ++r) {
        const double* __restrict__ drow =
            D + static_cast<size_t>(r < NA ? fa + r : fb + (r - NA)) * n + kc0;
        for (int k = tid; k < kw; k += THREADS) {
          krows[r * kw + k] = 0.0;
          if (ROWS > 1) drows[r * kw + k] = drow[k];
        }
      }
    }
    for (int ti = ch.tb; ti < ch.te; ++ti) {
      const Tile t = tiles[ti];
      const bool active = lane < t.count;
      const int lane_off = active ? lane : 0;  // an idle lane repeats the first
      part_run<LA, LB, LC, LD, 0>(wave, src, bp, t, lane, lane_off, part_lds, prims, slab);
      __syncthreads();
      // (ab|cd) of the wave's component pairs ab, digested
      unsigned lo = 8u * static_cast<unsigned>(lane);
      double* sl = slab;
      asm volatile("" : "+v"(lo), "+s"(sl));
      const int kidx = t.ket0 + lane_off;
      const int2 kf = (kfn + t.ket0)[lane_off];
      const double2 g1 = (kgeo + a.ket.npairs + t.ket0)[lane_off],
                    g2 = (kgeo + 2 * static_cast<size_t>(a.ket.npairs) + t.ket0)[lane_off];
      const int fc = kf.x, fd = kf.y;
      const int e = (fa != fb ? 1 : 0) + (fc != fd ? 1 : 0) + (t.bra != kidx ? 1 : 0);
      const double s = __hiloint2double(active ? (1023 - 3 + e) << 20 : 0, 0);
      const int oc = fc - kc0, od = fd - kc0;
      const unsigned kq8 = static_cast<unsigned>(kidx - a.jp_ket.begin) * 8u;
      const unsigned kstride = static_cast<unsigned>(a.jp_ket.n);
      double dcd[NC * ND], jcd[NC * ND];
#pragma unroll
      for (int k = 0; k < NC * ND; ++k) {
        dcd[k] = ld_off(Dp + a.jp_ket.base, kq8 + 8u * k * kstride);
        jcd[k] = 0.0;
      }
      // v added at column x (of c or d) of row r (of a, or NA + of b)
      auto add = [&](int r, int x, double v) {
        if constexpr (ROWS > 0)
          atomicAdd(&krows[r * kw + x], v);
        else
          unsafeAtomicAdd(at_off(a.K + static_cast<size_t>(r < NA ? fa + r : fb + (r - NA)) * n,
                                 8u * static_cast<unsigned>(x)),
                          v);
      };
      auto den = [&](int r, int x) {
        if constexpr (ROWS > 1)
          return drows[r * kw + x];
        else
          return ld_off(D + static_cast<size_t>(r < NA ? fa + r : fb + (r - NA)) * n + kc0,
                        8u * static_cast<unsigned>(x));
      };
      double kac[NC], kad[ND];
      const int ab0 = NA * NB * wave / W, ab1 = NA * NB * (wave + 1) / W;
      for (int ab = ab0; ab < ab1; ++ab) {  // wave-uniform
        const int ia = ab / NB, ib = ab - ia * NB;
        double g[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) g[f] = 0.0;
        for (int x = 0; x < 4; ++x) {
          const PartTerm tm = C::term(ab, x);
          if (tm.c == 0.0) break;
          const double c = tm.c * part_power(bp.AB[0], tm.px) * part_power(bp.AB[1], tm.py) *
                           part_power(bp.AB[2], tm.pz);
          const double* row = sl + tm.e * (NF * 64);
#pragma unroll
          for (int f = 0; f < NF; ++f) g[f] += c * ld_off(row + f * 64, lo);
        }
        double I[NC * ND];
        C::ket_hrr(g, g1.y, g2.x, g2.y, I);
        const double dab = D[static_cast<size_t>(fa + ia) * n + fb + ib];
        double jab = 0.0;
#pragma unroll
        for (int k = 0; k < NC * ND; ++k) {
          jab += I[k] * dcd[k];
          jcd[k] += I[k] * dab;
        }
        jab = wave_sum(2.0 * s * jab);
        if (lane == 0) jb[ab] += jab;  // this wave's alone
        double dad[ND], dac[NC], dbd[ND], dbc[NC];
#pragma unroll
        for (int id = 0; id < ND; ++id) {
          dad[id] = den(ia, od + id);
          dbd[id] = den(NA + ib, od + id);
        }
#pragma unroll
        for (int ic = 0; ic < NC; ++ic) {
          dac[ic] = den(ia, oc + ic);
          dbc[ic] = den(NA + ib, oc + ic);
        }
        if (ib == 0 || ab == ab0) {
#pragma unroll
          for (int ic = 0; ic < NC; ++ic) kac[ic] = 0.0;
#pragma unroll
          for (int id = 0; id < ND; ++id) kad[id] = 0.0;
        }
        double kbc[NC], kbd[ND];
#pragma unroll
        for (int ic = 0; ic < NC; ++ic) kbc[ic] = 0.0;
#pragma unroll
        for (int id = 0; id < ND; ++id) kbd[id] = 0.0;
#pragma unroll
        for (int ic = 0; ic < NC; ++ic)
#pragma unroll
          for (int id = 0; id < ND; ++id) {
            const double v = I[ic * ND + id];
            kac[ic] += v * dbd[id];
            kad[id] += v * dbc[ic];
            kbc[ic] += v * dad[id];
            kbd[id] += v * dac[ic];
          }
        if (active) {
#pragma unroll
          for (int ic = 0; ic < NC; ++ic) add(NA + ib, oc + ic, s * kbc[ic]);
#pragma unroll
          for (int id = 0; id < ND; ++id) add(NA + ib, od + id, s * kbd[id]);
          if (ib == NB - 1 || ab == ab1 - 1) {
#pragma unroll
            for (int ic = 0; ic < NC; ++ic) add(ia, oc + ic, s * kac[ic]);
#pragma unroll
            for (int id = 0; id < ND; ++id) add(ia, od + id, s * kad[id]);
          }
        }
      }
#pragma unroll
      for (int k = 0; k < NC * ND; ++k) atomicAdd(&jq[k * 64 + lane], 2.0 * s * jcd[k]);
      __syncthreads();  // the slab is free for the next tile
      for (int k = wave; k < NC * ND; k += W) {
        const double v = jq[k * 64 + lane];
        jq[k * 64 + lane] = 0.0;
        if (active) unsafeAtomicAdd(at_off(a.Jp + a.jp_ket.base, kq8 + 8u * k * kstride), v);
      }
    }
    const int bq = ch.bra - a.jp_bra.begin;
    if (tid < NA * NB && jb[tid] != 0.0)
      unsafeAtomicAdd(&a.Jp[a.jp_bra.base + tid * a.jp_bra.n + bq], jb[tid]);
    if constexpr (ROWS > 0) {
      for (int r = 0; r < NA + NB; ++r) {
        double* krow = a.K + static_cast<size_t>(r < NA ? fa + r : fb + (r - NA)) * n + kc0;
        for (int k = tid; k < kw; k += THREADS) {
          const double v = krows[r * kw + k];
          if (v != 0.0) unsafeAtomicAdd(&krow[k], v);
        }
      }
    }
    if (ROWS && tid == 0) s_next[turn] = next;
    __syncthreads();
    u = ROWS ? begin + static_cast<int>(gridDim.x) + __builtin_amdgcn_readfirstlane(s_next[turn])
             : u + static_cast<int>(gridDim.x);
    turn ^= 1;
  }
}

// Workgroups a compute unit can hold by registers, and the bytes of one's slab.
template <int LA, int LB, int LC, int LD>
constexpr int eri_part_groups() {
  using C = EriParts<LA, LB, LC, LD>;
  return 4 * C::MINW / C::W;
}
template <int LA, int LB, int LC, int LD>
constexpr size_t eri_part_slab() {
  return EriClass<LA, LB, LC, LD>::NACC * 64 * sizeof(double);
}

template <int LA, int LB, int LC, int LD, int ROWS>
hipError_t eri_part_launch_rows(const EriArgs& a, double* slab, size_t lds, int blocks,
                                hipStream_t s) {
  hipLaunchKernelGGL((eri_part_kernel<LA, LB, LC, LD, ROWS>), dim3(blocks),
                     dim3(64 * EriParts<LA, LB, LC, LD>::W), lds, s, a, slab, a.prims, a.D, a.Dp,
                     a.pairs, a.tiles, a.chunks, a.ket.geo, a.ket.fn, a.ket.prim);
  return hipGetLastError();
}

// LDS of a workgroup beside its rows, and whether its K rows of kw columns fit.
template <int LA, int LB, int LC, int LD>
constexpr size_t eri_part_fixed() {
  return sizeof(double) * (part_boys<LA + LB + LC + LD>() + ncart(LC) * ncart(LD) * 64 +
                           ncart(LA) * ncart(LB));
}
template <int LA, int LB, int LC, int LD>
bool eri_part_rows_fit(int kw) {
  return eri_part_fixed<LA, LB, LC, LD>() +
             sizeof(double) * (ncart(LA) + ncart(LB)) * static_cast<size_t>(kw) <=
         kLdsPerCu;
}

template <int LA, int LB, int LC, int LD>
hipError_t eri_part_launch(const EriArgs& a, double* slab, size_t bytes, int cus, hipStream_t s) {
  constexpr int NA = ncart(LA), NB = ncart(LB);
  constexpr int groups = eri_part_groups<LA, LB, LC, LD>();
  // no more workgroups than the slab was reserved for
  const size_t most = bytes / eri_part_slab<LA, LB, LC, LD>();
  if (!a.Dp || !a.Jp || !slab || most == 0) return hipErrorInvalidValue;
  const size_t fixed = eri_part_fixed<LA, LB, LC, LD>();
  const size_t rows = sizeof(double) * (NA + NB) * static_cast<size_t>(a.kw);
  // K rows in LDS where they fit, the density's too unless that costs a workgroup
  const auto held = [&](size_t lds) { return std::min<int>(groups, kLdsPerCu / lds); };
  const auto grid = [&](int n) {
    return static_cast<int>(std::min(most, static_cast<size_t>(n) * cus));
  };
  const int rows2 = held(fixed + 2 * rows), rows1 = held(fixed + rows);
  if (a.chunk_range && rows2 > 0 && rows2 == rows1)
    return eri_part_launch_rows<LA, LB, LC, LD, 2>(a, slab, fixed + 2 * rows, grid(rows2), s);
  if (a.chunk_range && rows1 > 0)
    return eri_part_launch_rows<LA, LB, LC, LD, 1>(a, slab, fixed + rows, grid(rows1), s);
  return eri_part_launch_rows<LA, LB, LC, LD, 0>(a, slab, fixed, grid(held(fixed)), s);
}

}  // namespace rchem
