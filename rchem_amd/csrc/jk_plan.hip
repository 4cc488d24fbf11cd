// Device-side quartet planning for one Fock build (gfx950).
//
// The work of a build is a class-sorted queue of tiles (one bra shell pair x
// up to 64 ket pairs of one bucket).  It is rebuilt on the device for every
// density, with no host round trip, in four steps:
//   1. dmax:   max |D_ij| (order-preserving integer atomics on |D|'s bits);
//   2. plan:   one thread per task (bra pair, ket bucket): the ket range that
//              survives Schwarz screening Q_ab Q_cd >= tau (Q sorted descending
//              inside a bucket, so the survivors are a prefix found by binary
//              search), split into an FP64 prefix (Q_ab Q_cd max|D| >=
//              mixed_thresh) and an FP32 remainder; tile counts per task;
//   3. scan:   exclusive prefix sums of the tile counts (hipCUB; FP64-only
//              builds have one list, and no scan of the other's counts);
//   4. expand: each task writes its tiles;
//   5. chunks: the tiles of one (class, bra pair) unit are cut into chunks of
//              at most the class's chunk size per precision (from the tuning
//              table; a workgroup's unit of work when K is
//              digested in LDS), counted, scanned and written (optionally
//              radix-sorted by first ket pair within each class); per class the
//              [begin, end) tile and chunk ranges of each precision go to device
//              memory, where the persistent ERI kernels read them.
// Small passes take 2 to 5 in one launch (plan_direct_kernel).
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>

#include "types.hpp"

namespace rchem {

// max over the block (256 threads), the result in thread 0
__device__ __forceinline__ unsigned long long block_max_u64(unsigned long long m) {
  __shared__ unsigned long long part[4];
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned long long o = __shfl_xor(m, off, 64);
    m = o > m ? o : m;
  }
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0)
    for (int w = 1; w < 4; ++w) m = part[w] > m ? part[w] : m;
  return m;
}

// One atomic per workgroup (of at most 256): all of them meet on one address.
__global__ __launch_bounds__(256) void dmax_kernel(const double* __restrict__ D, size_t n2,
                                                   unsigned long long* __restrict__ out) {
  unsigned long long m = 0;
  for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < n2;
       i += static_cast<size_t>(gridDim.x) * blockDim.x) {
    const double v = fabs(D[i]);
    const unsigned long long b = __double_as_longlong(v);  // non-negative: bits order = value order
    m = b > m ? b : m;
  }
  m = block_max_u64(m);
  if (threadIdx.x == 0) atomicMax(out, m);
}

// The same over the diagonal blocks [f0_m, f0_m + nb_m)^2 of a multi-molecule
// basis (the rest of D is never read).
__global__ void dmax_blocks_kernel(const double* __restrict__ D, size_t n,
                                   const int* __restrict__ f0, const int* __restrict__ nb,
                                   unsigned long long* __restrict__ out) {
  const int m = blockIdx.y, b = nb[m];
  const size_t o = f0[m];
  unsigned long long mx = 0;
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < b * b; k += gridDim.x * blockDim.x) {
    const double v = fabs(D[(o + k / b) * n + o + k % b]);
    const unsigned long long bits = __double_as_longlong(v);
    mx = bits > mx ? bits : mx;
  }
  mx = block_max_u64(mx);
  if (threadIdx.x == 0) atomicMax(out, mx);
}

// First index in [lo, hi) whose Q falls below `need` (Q non-increasing).
__device__ __forceinline__ int first_below(const double* __restrict__ Q, int lo, int hi,
                                           double need) {
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (Q[mid] >= need) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ double wave_sum_d(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

__device__ __forceinline__ int class_of_task(const PlanArgs& a, int t) {
  int c = 0;
  while (c + 1 < a.nclasses && a.classes[c + 1].task_begin <= t) ++c;
  return c;
}

// The kets of bra pair i in bucket slot `slot`: [lo, mid) in FP64, [mid, hi) in FP32.
struct TaskRange {
  int lo, mid, hi;
};
__device__ __forceinline__ TaskRange task_range(const PlanArgs& a, const PlanClass& pc, int i,
                                                int slot, const int4& bk) {
  int lo = bk.x, hi = bk.y;
  bool all64 = false;
  if (a.segs) {  // the bra's molecule only
    const int mol = a.pair_mol[i];
    const int2 sg = a.segs[static_cast<size_t>(slot) * a.nmol + mol];
    const int state = a.mol_active ? a.mol_active[mol] : 1;
    lo = sg.x;
    hi = state == 0 ? sg.x : sg.y;  // a retired molecule: none
    all64 = state == 2;             // a molecule past its precision switch: no FP32
  }
  if (pc.same) hi = (lo > i) ? lo : min(hi, i + 1);
  const double qi = a.Q[i];
  if (a.tau > 0.0) hi = (qi > 0.0) ? first_below(a.Q, lo, hi, a.tau / qi) : lo;
  int mid = hi;
  if (a.mixed_thresh > 0.0 && hi > lo && !all64) {
    const double dm = *a.dmax;
    const double need = (qi > 0.0 && dm > 0.0) ? a.mixed_thresh / (qi * dm) : HUGE_VAL;
    mid = first_below(a.Q, lo, hi, need);
  }
  return TaskRange{lo, mid, hi};
}

__global__ void plan_kernel(const PlanArgs a) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = t < a.ntasks;
  if (t == a.ntasks) {  // the extra slot makes the exclusive scan's last entry the total
    a.cnt64[t] = 0;
    a.cnt32[t] = 0;
  }
  int c = 0;
  double q64 = 0.0, q32 = 0.0, p64 = 0.0, p32 = 0.0;
  if (valid) {
    c = class_of_task(a, t);
    const PlanClass pc = a.classes[c];
    const int local = t - pc.task_begin;
    const int i = pc.bra_begin + local / pc.nbk;
    const int slot = pc.bk_off + local % pc.nbk;
    const int4 bk = a.buckets[slot];
    const auto [lo, mid, hi] = task_range(a, pc, i, slot, bk);
    a.lo[t] = lo;
    a.mid[t] = mid;
    a.hi[t] = hi;
    const int np = a.pairs[i].np;
    const int parts = PrimSplit(np, bk.z, pc.limit).parts();
    a.cnt64[t] = ((mid - lo + 63) >> 6) * parts;
    a.cnt32[t] = ((hi - mid + 63) >> 6) * parts;
    const double npp = static_cast<double>(np) * bk.z;
    q64 = mid - lo;
    q32 = hi - mid;
    p64 = q64 * npp;
    p32 = q32 * npp;
  }
  // statistics: one atomic per wave when the wave's tasks share a class, into
  // the wave's replica
  double* const stats = a.stats + static_cast<size_t>((t >> 6) & (kPlanStatsReplicas - 1)) *
                                      a.stats_stride;
  const int c0 = __shfl(c, 0, 64);
  const int lastv = __shfl(valid ? 1 : 0, 63, 64);
  const int c63 = __shfl(c, 63, 64);
  if (lastv && c0 == c63) {
    q64 = wave_sum_d(q64);
    q32 = wave_sum_d(q32);
    p64 = wave_sum_d(p64);
    p32 = wave_sum_d(p32);
    if ((threadIdx.x & 63) == 0) {
      double* st = stats + 4 * c0;
      if (q64 > 0) { unsafeAtomicAdd(st + 0, q64); unsafeAtomicAdd(st + 2, p64); }
      if (q32 > 0) { unsafeAtomicAdd(st + 1, q32); unsafeAtomicAdd(st + 3, p32); }
    }
  } else if (valid) {
    double* st = stats + 4 * c;
    if (q64 > 0) { unsafeAtomicAdd(st + 0, q64); unsafeAtomicAdd(st + 2, p64); }
    if (q32 > 0) { unsafeAtomicAdd(st + 1, q32); unsafeAtomicAdd(st + 3, p32); }
  }
}

// off64/off32: exclusive scans of the tile counts (length ntasks + 1).
__global__ void expand_kernel(const PlanArgs a, const int* __restrict__ off64,
                              const int* __restrict__ off32, Tile* __restrict__ tiles64,
                              Tile* __restrict__ tiles32, int cap) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= a.ntasks) return;
  const PlanClass pc = a.classes[class_of_task(a, t)];
  const int local = t - pc.task_begin;
  const int i = pc.bra_begin + local / pc.nbk;
  const int lo = a.lo[t], mid = a.mid[t], hi = a.hi[t];
  const PrimSplit sp(a.pairs[i].np, a.buckets[pc.bk_off + local % pc.nbk].z, pc.limit);
  const int parts = sp.parts();
  int o = off64[t];
  for (int k = lo; k < mid; k += 64)
    for (int p = 0; p < parts && o < cap; ++p, ++o)
      tiles64[o] = Tile{i, k, min(64, mid - k), sp.pad(p)};
  if (!off32) return;
  o = off32[t];
  for (int k = mid; k < hi; k += 64)
    for (int p = 0; p < parts && o < cap; ++p, ++o)
      tiles32[o] = Tile{i, k, min(64, hi - k), sp.pad(p)};
}

__device__ __forceinline__ int class_of_unit(const PlanArgs& a, int u) {
  int c = 0;
  while (c + 1 < a.nclasses && a.classes[c + 1].unit_begin <= u) ++c;
  return c;
}

// Unit u = (class c, bra pair): its tasks are [t0, t0 + nbk).
__device__ __forceinline__ void unit_tasks(const PlanArgs& a, int u, int* c, int* bra, int* t0,
                                           int* t1) {
  *c = class_of_unit(a, u);
  const PlanClass pc = a.classes[*c];
  const int local = u - pc.unit_begin;
  *bra = pc.bra_begin + local;
  *t0 = pc.task_begin + local * pc.nbk;
  *t1 = *t0 + pc.nbk;
}

__global__ void chunk_count_kernel(const PlanArgs a, const int* __restrict__ off64,
                                   const int* __restrict__ off32, int* __restrict__ chc64,
                                   int* __restrict__ chc32) {
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u > a.nunits) return;
  if (u == a.nunits) {
    chc64[u] = 0;
    chc32[u] = 0;
    return;
  }
  int c, bra, t0, t1;
  unit_tasks(a, u, &c, &bra, &t0, &t1);
  const int ch64 = a.classes[c].chunk64, ch32 = a.classes[c].chunk32;
  chc64[u] = (off64[t1] - off64[t0] + ch64 - 1) / ch64;
  if (off32) chc32[u] = (off32[t1] - off32[t0] + ch32 - 1) / ch32;
}

// cap bounds the tile offsets (tile buffers), ccap the chunk records written
// (chunk buffers); every record below min(chunk count, ccap) is written.
// keys64 / keys32 (when set): per chunk, (c << key_shift) | (first ket pair of
// the chunk / 64), c the chunk's class (segment) in this pass.
__global__ void chunk_expand_kernel(const PlanArgs a, const int* __restrict__ off64,
                                    const int* __restrict__ off32, const int* __restrict__ choff64,
                                    const int* __restrict__ choff32, Chunk* __restrict__ chunks64,
                                    Chunk* __restrict__ chunks32, int cap, int ccap,
                                    const Tile* __restrict__ tiles64,
                                    const Tile* __restrict__ tiles32, unsigned* __restrict__ keys64,
                                    unsigned* __restrict__ keys32, int key_shift) {
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= a.nunits) return;
  int c, bra, t0, t1;
  unit_tasks(a, u, &c, &bra, &t0, &t1);
  const unsigned khigh = static_cast<unsigned>(c) << key_shift;
  // a class planned in bra order keeps it: its keys differ only by class, and
  // the sort is stable
  const int order = a.classes[c].order;
  {
    const int ch = a.classes[c].chunk64;
    const int tb = min(off64[t0], cap), te = min(off64[t1], cap);
    int o = choff64[u];
    for (int k = tb; k < te && o < ccap; k += ch, ++o) {
      chunks64[o] = Chunk{bra, k, min(k + ch, te), 0};
      if (keys64) keys64[o] = khigh | ((order & 1) ? static_cast<unsigned>(tiles64[k].ket0 >> 6) : 0u);
    }
  }
  if (off32) {
    const int ch = a.classes[c].chunk32;
    const int tb = min(off32[t0], cap), te = min(off32[t1], cap);
    int o = choff32[u];
    for (int k = tb; k < te && o < ccap; k += ch, ++o) {
      chunks32[o] = Chunk{bra, k, min(k + ch, te), 0};
      if (keys32) keys32[o] = khigh | ((order & 2) ? static_cast<unsigned>(tiles32[k].ket0 >> 6) : 0u);
    }
  }
}

// The whole plan of a pass in one launch, for passes of little work: 16 lanes to a
// unit, each class's tiles and chunks in a range of their own (PlanClass::base;
// the capacities are upper bounds), handed out to the units by counters -- the
// range ends in `ranges`, which begin_kernel has set to the bases -- so a
// class's units come in any order.  One block's units of a class take their
// places with one atomic.
constexpr int kDirectLanes = 16;

__global__ __launch_bounds__(256) void plan_direct_kernel(const PlanArgs a,
                                                          Tile* __restrict__ tiles64,
                                                          Tile* __restrict__ tiles32,
                                                          Chunk* __restrict__ chunks64,
                                                          Chunk* __restrict__ chunks32, int cap,
                                                          int* __restrict__ ranges) {
  constexpr int G = 256 / kDirectLanes;
  __shared__ int sc[G], sn[4][G], sbase[4][G];
  __shared__ double sq[4][G];
  const int g = threadIdx.x / kDirectLanes, l = threadIdx.x % kDirectLanes;
  const int u = blockIdx.x * G + g;
  const bool valid = u < a.nunits;
  int c = -1, bra = 0, t0 = 0, t1 = 0;
  PlanClass pc{};
  if (valid) {
    unit_tasks(a, u, &c, &bra, &t0, &t1);
    pc = a.classes[c];
  }
  const int np = valid ? a.pairs[bra].np : 0;
  int n[2] = {0, 0};  // tiles, FP64 and FP32
  double q[4] = {0.0, 0.0, 0.0, 0.0};
  for (int t = t0 + l; t < t1; t += kDirectLanes) {
    const int slot = pc.bk_off + t - t0;
    const int4 bk = a.buckets[slot];
    const auto [lo, mid, hi] = task_range(a, pc, bra, slot, bk);
    a.lo[t] = lo;
    a.mid[t] = mid;
    a.hi[t] = hi;
    const int parts = PrimSplit(np, bk.z, pc.limit).parts();
    n[0] += ((mid - lo + 63) >> 6) * parts;
    n[1] += ((hi - mid + 63) >> 6) * parts;
    const double npp = static_cast<double>(np) * bk.z;
    q[0] += mid - lo;
    q[1] += hi - mid;
    q[2] += (mid - lo) * npp;
    q[3] += (hi - mid) * npp;
  }
  for (int off = kDirectLanes / 2; off > 0; off >>= 1) {
    for (int p = 0; p < 2; ++p) n[p] += __shfl_xor(n[p], off, kDirectLanes);
    for (int k = 0; k < 4; ++k) q[k] += __shfl_xor(q[k], off, kDirectLanes);
  }
  const int ch[2] = {pc.chunk64, pc.chunk32};
  if (l == 0) {
    sc[g] = c;
    for (int p = 0; p < 2; ++p) {
      sn[p][g] = n[p];
      sn[2 + p][g] = valid ? (n[p] + ch[p] - 1) / ch[p] : 0;
    }
    for (int k = 0; k < 4; ++k) sq[k][g] = q[k];
  }
  __syncthreads();
  int first = g, before[4] = {0, 0, 0, 0};
  for (int h = g - 1; h >= 0 && sc[h] == c; --h) {
    first = h;
    for (int k = 0; k < 4; ++k) before[k] += sn[k][h];
  }
  if (valid && l < 4 && first == g) {  // lane k: list k of the block's units of the class
    int total = 0;
    double s = 0.0;
    for (int h = g; h < G && sc[h] == c; ++h) {
      total += sn[l][h];
      s += sq[l][h];
    }
    sbase[l][g] = total > 0 ? atomicAdd(&ranges[8 * c + 2 * l + 1], total) : 0;
    if (s > 0.0)
      unsafeAtomicAdd(a.stats + static_cast<size_t>(blockIdx.x & (kPlanStatsReplicas - 1)) *
                                    a.stats_stride + 4 * c + l,
                      s);
  }
  __syncthreads();
  if (!valid) return;
  for (int p = 0; p < 2; ++p) {
    if (n[p] == 0) continue;
    Tile* const tiles = p ? tiles32 : tiles64;
    Chunk* const chunks = p ? chunks32 : chunks64;
    const int ob = sbase[p][first] + before[p];
    const int cb = sbase[2 + p][first] + before[2 + p], nch = (n[p] + ch[p] - 1) / ch[p];
    for (int x = l; x < nch; x += kDirectLanes)
      if (cb + x < cap)
        chunks[cb + x] = Chunk{bra, ob + x * ch[p], min(ob + (x + 1) * ch[p], ob + n[p]), 0};
    int o = ob;
    for (int t = t0; t < t1; t += kDirectLanes) {
      int from = 0, to = 0, knp = 0;  // of the lane's own task
      if (t + l < t1) {
        from = p ? a.mid[t + l] : a.lo[t + l];
        to = p ? a.hi[t + l] : a.mid[t + l];
        knp = a.buckets[pc.bk_off + t + l - t0].z;
      }
      for (int j = 0; j < min(kDirectLanes, t1 - t); ++j) {
        const int kb = __shfl(from, j, kDirectLanes), ke = __shfl(to, j, kDirectLanes);
        const PrimSplit sp(np, __shfl(knp, j, kDirectLanes), pc.limit);
        const int parts = sp.parts(), m = ((ke - kb + 63) >> 6) * parts;
        for (int x = l; x < m; x += kDirectLanes) {
          const int k = kb + 64 * (x / parts);
          if (o + x < cap) tiles[o + x] = Tile{bra, k, min(64, ke - k), sp.pad(x % parts)};
        }
        o += m;
      }
    }
  }
}

// Clears a build's accumulators (n2 = 0: J and K are cleared elsewhere) and its
// chunk counters, and sets every class's tile and chunk ranges to its base, empty.
__global__ void begin_kernel(double* __restrict__ J, double* __restrict__ K, size_t n2,
                             double* __restrict__ stats, size_t nstats, double* __restrict__ jp,
                             size_t njp, double* __restrict__ dmax,
                             const PlanClass* __restrict__ classes, int nclasses,
                             int* __restrict__ ranges, int* __restrict__ next) {
  const size_t i0 = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x;
  const size_t step = static_cast<size_t>(gridDim.x) * blockDim.x;
  for (size_t i = i0; i < n2; i += step) {
    J[i] = 0.0;
    K[i] = 0.0;
  }
  for (size_t i = i0; i < njp; i += step) jp[i] = 0.0;
  for (size_t i = i0; i < nstats; i += step) stats[i] = 0.0;
  if (i0 == 0) *dmax = 0.0;
  for (size_t i = i0; i < 8 * static_cast<size_t>(nclasses); i += step)
    ranges[i] = classes[i / 8].base;
  for (size_t i = i0; i < 2 * static_cast<size_t>(nclasses); i += step) next[i] = 0;
}

// keys[i] = all ones for i in [total, n): the entries past the chunk count
// sort to the end.
__global__ void pad_keys_kernel(unsigned* __restrict__ keys, const int* __restrict__ total, int n) {
  const int t = min(*total, n);
  for (int i = t + blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    keys[i] = ~0u;
}

// ranges[8c .. 8c+7] = tiles {b64, e64, b32, e32}, chunks {b64, e64, b32, e32}
// of class c, clamped to the buffer capacity.
__global__ void ranges_kernel(const PlanArgs a, const int* __restrict__ off64,
                              const int* __restrict__ off32, const int* __restrict__ choff64,
                              const int* __restrict__ choff32, int* __restrict__ ranges, int cap,
                              int ccap) {
  const int c = threadIdx.x;
  if (c >= a.nclasses) return;
  const int tb = a.classes[c].task_begin;
  const int te = (c + 1 < a.nclasses) ? a.classes[c + 1].task_begin : a.ntasks;
  const int ub = a.classes[c].unit_begin;
  const int ue = (c + 1 < a.nclasses) ? a.classes[c + 1].unit_begin : a.nunits;
  ranges[8 * c + 0] = min(off64[tb], cap);
  ranges[8 * c + 1] = min(off64[te], cap);
  ranges[8 * c + 2] = off32 ? min(off32[tb], cap) : 0;
  ranges[8 * c + 3] = off32 ? min(off32[te], cap) : 0;
  ranges[8 * c + 4] = min(choff64[ub], ccap);
  ranges[8 * c + 5] = min(choff64[ue], ccap);
  ranges[8 * c + 6] = off32 ? min(choff32[ub], ccap) : 0;
  ranges[8 * c + 7] = off32 ? min(choff32[ue], ccap) : 0;
}

hipError_t dmax_launch(const double* D, size_t n2, unsigned long long* out, hipStream_t s) {
  size_t blocks = (n2 + 255) / 256;
  if (blocks > 512) blocks = 512;
  if (blocks == 0) blocks = 1;
  hipLaunchKernelGGL(dmax_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, D, n2,
                     out);
  return hipGetLastError();
}

// Bits of the class field of a chunk key (classes of one pass).
int plan_class_bits(int nclasses) {
  int bits = 0;
  while ((1 << bits) < nclasses) ++bits;
  return bits;
}

// Temporary-storage bytes of a radix sort of n chunk keys and chunks.
size_t plan_sort_bytes(int n) {
  size_t bytes = 0;
  if (hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, static_cast<unsigned*>(nullptr),
                                         static_cast<unsigned*>(nullptr),
                                         static_cast<Chunk*>(nullptr),
                                         static_cast<Chunk*>(nullptr), n, 0, 32) != hipSuccess)
    return 0;
  return bytes;
}

hipError_t dmax_blocks_launch(const double* D, size_t n, const int* f0, const int* nb, int nmol,
                              int nmax, unsigned long long* out, hipStream_t s) {
  if (nmol <= 0) return hipSuccess;
  const unsigned gx = static_cast<unsigned>(min(64, (nmax * nmax + 255) / 256));
  hipLaunchKernelGGL(dmax_blocks_kernel, dim3(gx, nmol), dim3(256), 0, s, D, n, f0, nb, out);
  return hipGetLastError();
}

// Temporary-storage bytes of a scan over n + 1 entries.
size_t plan_scan_bytes(int n) {
  size_t bytes = 0;
  if (hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, static_cast<int*>(nullptr),
                                       static_cast<int*>(nullptr), n + 1) != hipSuccess)
    return 0;
  return bytes;
}

hipError_t begin_launch(double* J, double* K, size_t n2, double* stats, size_t nstats, double* jp,
                        size_t njp, double* dmax, const PlanClass* classes, int nclasses,
                        int* ranges, int* next, hipStream_t s) {
  const size_t most = std::max({n2, nstats, njp, static_cast<size_t>(8) * nclasses});
  const unsigned blocks = static_cast<unsigned>(std::min<size_t>(2048, (most + 255) / 256));
  hipLaunchKernelGGL(begin_kernel, dim3(std::max(1u, blocks)), dim3(256), 0, s, J, K, n2, stats,
                     nstats, jp, njp, dmax, classes, nclasses, ranges, next);
  return hipGetLastError();
}

hipError_t plan_launch(const PlanArgs& a, const PlanBuffers& b, hipStream_t s) {
  if (b.direct) {
    if (a.nunits <= 0) return hipSuccess;
    constexpr int units = 256 / kDirectLanes;
    hipLaunchKernelGGL(plan_direct_kernel, dim3((a.nunits + units - 1) / units), dim3(256), 0, s,
                       a, b.tiles64, b.tiles32, b.chunks64, b.chunks32, b.cap, b.ranges);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(plan_kernel, dim3(static_cast<unsigned>((a.ntasks + 1 + 255) / 256)),
                     dim3(256), 0, s, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  size_t sb = b.scan_bytes;
  e = hipcub::DeviceScan::ExclusiveSum(b.scan_tmp, sb, a.cnt64, b.off64, a.ntasks + 1, s);
  if (e != hipSuccess) return e;
  const int* off32 = a.mixed_thresh > 0.0 ? b.off32 : nullptr;  // null: no FP32 list
  if (off32) {
    sb = b.scan_bytes;
    e = hipcub::DeviceScan::ExclusiveSum(b.scan_tmp, sb, a.cnt32, b.off32, a.ntasks + 1, s);
    if (e != hipSuccess) return e;
  }
  if (a.ntasks > 0) {
    hipLaunchKernelGGL(expand_kernel, dim3(static_cast<unsigned>((a.ntasks + 255) / 256)),
                       dim3(256), 0, s, a, b.off64, off32, b.tiles64, b.tiles32, b.cap);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(chunk_count_kernel, dim3(static_cast<unsigned>((a.nunits + 1 + 255) / 256)),
                     dim3(256), 0, s, a, b.off64, off32, b.chc64, b.chc32);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  sb = b.scan_bytes;
  e = hipcub::DeviceScan::ExclusiveSum(b.scan_tmp, sb, b.chc64, b.choff64, a.nunits + 1, s);
  if (e != hipSuccess) return e;
  if (off32) {
    sb = b.scan_bytes;
    e = hipcub::DeviceScan::ExclusiveSum(b.scan_tmp, sb, b.chc32, b.choff32, a.nunits + 1, s);
    if (e != hipSuccess) return e;
  }
  const bool sorting = b.key_bits > 0 && b.ccap > 0;
  const bool sort64 = sorting && (b.sort_mask & 1);
  // FP64-only builds have no FP32 chunks
  const bool sort32 = sorting && (b.sort_mask & 2) && a.mixed_thresh > 0.0;
  // chunk records per precision: every record below min(count, ccap) is written
  const int ccap = sorting ? min(b.cap, b.ccap) : b.cap;
  Chunk* out64 = sort64 ? b.chunks_raw : b.chunks64;
  Chunk* out32 = sort32 ? b.chunks_raw + b.ccap : b.chunks32;
  unsigned* k64 = sort64 ? b.keys_raw : nullptr;
  unsigned* k32 = sort32 ? b.keys_raw + b.ccap : nullptr;
  if (a.nunits > 0) {
    hipLaunchKernelGGL(chunk_expand_kernel, dim3(static_cast<unsigned>((a.nunits + 255) / 256)),
                       dim3(256), 0, s, a, b.off64, off32, b.choff64, b.choff32, out64, out32,
                       b.cap, ccap, b.tiles64, b.tiles32, k64, k32,
                       b.key_bits - plan_class_bits(a.nclasses));
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  for (int p = 0; p < 2; ++p) {
    if (!(p ? sort32 : sort64)) continue;
    unsigned* kin = b.keys_raw + static_cast<size_t>(p) * b.ccap;
    const unsigned pad_blocks = static_cast<unsigned>(min((b.ccap + 255) / 256, 1024));
    hipLaunchKernelGGL(pad_keys_kernel, dim3(pad_blocks), dim3(256), 0, s, kin,
                       (p ? b.choff32 : b.choff64) + a.nunits, b.ccap);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    size_t sb = b.sort_bytes;
    e = hipcub::DeviceRadixSort::SortPairs(b.sort_tmp, sb, kin, b.keys_sorted,
                                           b.chunks_raw + static_cast<size_t>(p) * b.ccap,
                                           p ? b.chunks32 : b.chunks64, b.ccap, 0, b.key_bits, s);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(ranges_kernel, dim3(1), dim3(64), 0, s, a, b.off64, off32, b.choff64,
                     b.choff32, b.ranges, b.cap, ccap);
  return hipGetLastError();
}

}  // namespace rchem
