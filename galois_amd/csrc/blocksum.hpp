// Deterministic row sums over a CSR/CSC in two streaming phases, for vectors
// whose gathers the row sweep (rowsweep.hpp) would send to the L2 one by one:
// that sweep is bound by about 130 G gathers/s, while here an edge gathers
// from LDS.
//
//   layout  edges sorted by (chunk of the gathered index, row): a chunk is
//           2^shift gathered entries, staged in LDS.  A group is the edges of
//           one row inside one chunk.  Rows are cut into bins; a run is the
//           consecutive groups of one (chunk, bin) pair, cut after 64 groups
//           and where the edges of one wavefront of phase 1 end, so that a row
//           appears at most once in a run.  Built once per graph.
//   phase 1 (gather_kernel) one workgroup per piece of a chunk: stages the
//           chunk, then its wavefronts stream the edges (2 bytes of index per
//           edge, bit 15 set on the last edge of a group; 4 bytes of weight
//           where there are weights), add each group's products in FP64 and
//           write one FP64 partial sum per group in layout order.
//   phase 2 (sum_kernel) one wavefront per bin adds the bin's runs, in chunk
//           order, to FP64 sums in LDS (for FP64 vectors with what the additions
//           round off) and finalises the bin's rows.
//
// Every order is fixed: a group is summed by one wavefront front to back, and
// a row's partial sums are added by one wavefront, whose LDS additions are
// served in order (no two lanes of one addition hold the same row).  So the
// results are bit-reproducible run to run without exact sums, for any sign,
// scale, infinity or NaN.
//
// Bytes per sweep: 2 per edge (6 with weights), 18 per group (a partial sum
// written and read, its row), 8 per run, R (the size of a vector's entry) + what
// the finaliser reads and writes per row.
//
// Bound: phase 1 by memory (67M edges with weights, FP32: 0.60 GB in 147 us, 4.1
// TB/s), phase 2 by the latency of its short runs (25M groups: 110-114 us).  One
// such sweep takes 510-555 us by the row sweep; 20.6M edges in FP64 156 us, 38 +
// 49 us here.  With FP32 partial sums for FP32 vectors, each rounded, the phases
// took 122 and 77-91 us; with one sum a row for FP64 vectors phase 2 took 40.
#pragma once

#include <algorithm>

#include "gx_device.hpp"
#include "gx_internal.hpp"
#include "rowsweep.hpp"

namespace gx {
namespace bs {

constexpr int kItems = 8;                // edges per lane and tile
constexpr int kTile = kWave * kItems;    // 512
constexpr int kRangeTiles = 4;           // tiles of one wavefront's range: a group never crosses its end
constexpr uint32_t kEnd = 1u << 15;      // idx16 flag: last edge of a group
constexpr int kSumGrid = 256 * 16;       // most wavefronts of phase 2

// Gathered entries per chunk: 64 KB of LDS.  With the tiles' group sums (FP64 for
// both precisions, 64 KB) a CU holds one workgroup of phase 1, 16 wavefronts.
constexpr int kGatherBlock = 1024;
template <class Real>
struct Shape;
template <>
struct Shape<float> {
  static constexpr int kShift = 14;
};
template <>
struct Shape<double> {
  static constexpr int kShift = 13;
};

struct Piece {
  uint32_t chunk, tile0, tile1, pad;
};

struct Bin {
  uint32_t row0;
  uint32_t rows;  // with kPair: a row's sum is kept as two, see sum_kernel
  uint32_t run0, run1;
};
constexpr uint32_t kPair = 1u << 31;

struct Plan {
  const Piece* pieces;
  const uint16_t* idx16;     // ntiles * kTile
  const uint32_t* tile_grp;  // ntiles + 1: first group of every tile
  const uint32_t* eid;       // ntiles * kTile: edge id of every position, ~0 = padding (weighted layouts)
  const uint16_t* row16;     // per group: row in its bin
  const uint2* runs;         // per bin, in chunk order: first group, length (at most kWave)
  const Bin* bins;           // nbins, most runs first
  int64_t npieces, ntiles, ngroups, nruns, nbins;
  int lds_sums;              // LDS doubles a bin has for its sums
};

// Whether the layout pays for and can be built for this shape (see blocksum.hip).
bool pays(int64_t n, int64_t m);
// Builds (or returns the cached) layout of the row offsets `rowoff` and gathered
// indices `col`; perm != null: edge ids are perm[position] (CSC slot -> CSR
// edge).  shift: Shape<Real>::kShift.
Plan build(gx_graph* g, const int32_t* rowoff, const int32_t* col, const int32_t* perm, int64_t n, int64_t m,
           int shift, bool weighted, BlockSums& cache);

// Runs `prepare` (build and the scratch that goes with it); false, with nothing
// left of the layout, where device memory does not hold them: the build works in
// 32 bytes an edge, where the row sweep's plan takes one.  The sums then go
// through the row sweep.
template <class F>
bool fits(BlockSums& cache, F prepare) {
  try {
    prepare();
    return true;
  } catch (const Error& e) {
    if (e.code != GX_ERR_ALLOC) throw;
  }
  (void)hipGetLastError();  // the failed allocation is dealt with
  cache = BlockSums{};
  return false;
}

// wt[p] = w[eid[p]] (0 where padded).
void layout_weights(const Plan& P, const float* w, float* wt, hipStream_t s);

__device__ __forceinline__ uint32_t wave_exclusive_sum(uint32_t v, int lane) {
  uint32_t x = v;
  const int in_row = lane & 15;
  uint32_t o;
  o = __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);
  x += in_row >= 1 ? o : 0u;
  o = __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
  x += in_row >= 2 ? o : 0u;
  o = __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
  x += in_row >= 4 ? o : 0u;
  o = __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
  x += in_row >= 8 ? o : 0u;
  o = __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
  x += (lane & 16) ? o : 0u;
  o = __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
  x += (lane & 32) ? o : 0u;
  return x - v;
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// The loads of one tile: 8 consecutive edges per lane.
template <bool W>
struct TileLoad {
  u32x4 idx;
  f32x4 w[W ? 2 : 1];
  __device__ __forceinline__ void load(const uint16_t* __restrict__ idx16, const float* __restrict__ wt, int64_t T,
                                       int lane) {
    idx = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(idx16 + T * kTile) + lane);
    if constexpr (W) {
      const f32x4* p = reinterpret_cast<const f32x4*>(wt + T * kTile) + 2 * lane;
      w[0] = __builtin_nontemporal_load(p);
      w[1] = __builtin_nontemporal_load(p + 1);
    }
  }
};

// Phase 1 (see the file comment).  y: n entries.
template <class Real, bool W>
__global__ void __launch_bounds__(kGatherBlock) gather_kernel(Plan P, const float* __restrict__ wt,
                                                              const Real* __restrict__ y, int64_t n,
                                                              double* __restrict__ partial,
                                                              const unsigned* __restrict__ skip) {
  if (skip && *skip) return;
  constexpr int kSpan = 1 << Shape<Real>::kShift, kWaves = kGatherBlock / kWave;
  __shared__ Real ys[kSpan];
  __shared__ double stage[kWaves][kTile];
  const Piece pc = P.pieces[blockIdx.x];
  const int64_t base = static_cast<int64_t>(pc.chunk) * kSpan;
  const int cnt = static_cast<int>(n - base < kSpan ? n - base : kSpan);
  for (int i = threadIdx.x; i < cnt; i += kGatherBlock) ys[i] = y[base + i];
  __syncthreads();
  const int lane = static_cast<int>(lane_id());
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  double* st = stage[wid];
  for (int64_t r0 = pc.tile0 + wid * kRangeTiles; r0 < pc.tile1; r0 += kWaves * kRangeTiles) {
    const int64_t r1 = r0 + kRangeTiles < pc.tile1 ? r0 + kRangeTiles : pc.tile1;
    double open = 0;  // sum of the group open at the start of the tile (uniform)
    TileLoad<W> cur, nxt;
    cur.load(P.idx16, wt, r0, lane);
    for (int64_t T = r0; T < r1; ++T) {
      if (T + 1 < r1) nxt.load(P.idx16, wt, T + 1, lane);
      const uint32_t g0 = P.tile_grp[T], g1 = P.tile_grp[T + 1];
      double v[kItems];
      uint32_t ends = 0;
#pragma unroll
      for (int u = 0; u < kItems; ++u) {
        const uint32_t word = (cur.idx[u / 2] >> (16 * (u & 1))) & 0xffffu;
        ends |= (word >> 15) << u;
        v[u] = static_cast<double>(ys[word & (kSpan - 1)]);
        if constexpr (W) v[u] *= static_cast<double>(cur.w[u / 4][u & 3]);
      }
      double tail = 0;
#pragma unroll
      for (int u = 0; u < kItems; ++u) {
        tail += v[u];
        if ((ends >> u) & 1u) tail = 0;
      }
      const uint64_t heads = __ballot(ends != 0);
      const uint64_t upto = heads & (~0ull >> (63 - lane));
      const double seg = rs::wave_seg_scan(tail, upto ? 63 - __builtin_clzll(upto) : 0, lane);
      double before = __shfl_up(seg, 1);
      if (lane == 0) before = 0;
      if ((heads & ((1ull << lane) - 1)) == 0) before += open;
      const double last = __shfl(seg, kWave - 1);
      open = heads ? last : open + last;
      uint32_t slot = wave_exclusive_sum(static_cast<uint32_t>(__popc(ends)), lane);
      double acc = 0;
#pragma unroll
      for (int u = 0; u < kItems; ++u) {
        acc += v[u];
        if ((ends >> u) & 1u) {
          st[slot++] = before + acc;
          before = acc = 0;
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      for (uint32_t j = lane; j < g1 - g0; j += kWave) partial[g0 + j] = st[j];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      cur = nxt;
    }
  }
}

// Phase 2: one wavefront per workgroup, bin b on workgroup b mod the grid.  It
// is a chain of short loads (a run is about half a wavefront's lanes), so 16
// runs are in flight at a time and the next 64 runs' descriptors are loaded
// ahead: with 4 in flight it took 2-3 times as long.
//
// PAIRS (FP64 vectors): a row of k partial sums, added one after another, is off
// by 0.3 * sqrt(k / 3) units of its last place, where a sweep that sums values
// among themselves first stays near half a unit.  In bins with rows of more than
// kPairRow edges a row therefore has two sums, and the second collects what the
// additions to the first round off (Knuth's TwoSum; the LDS addition returns what
// it was added to), so that the row is rounded once.  Relative L2 errors over 8
// graphs of 700,000 vertices 1.65e-16 -> 1.34e-16 (gather by gather, 512-lane
// merge-path tiles: 1.40e-16), 600,000 vertices without hubs 1.06 -> 0.67e-16
// (0.89); PageRank of 1.5 M vertices 2.07 -> 2.31 ms a
// solve.
template <bool PAIRS, class Fin>
__global__ void __launch_bounds__(kWave) sum_kernel(Plan P, const double* __restrict__ partial, Fin fin,
                                                    double* __restrict__ part0, double* __restrict__ part1,
                                                    const unsigned* __restrict__ skip) {
  if (skip && *skip) return;
  fin.load();
  extern __shared__ double acc[];
  const int lane = static_cast<int>(lane_id());
  rs::DoubleSum a0, a1;  // a lane meets 64 rows a bin, often of one and the same value
  constexpr int kRuns = 16;
  for (int64_t b = blockIdx.x; b < P.nbins; b += gridDim.x) {
    const Bin bin = P.bins[b];
    const uint32_t row0 = bin.row0, q0 = bin.run0, q1 = bin.run1;
    const int rows = static_cast<int>(bin.rows & ~kPair);
    const bool pair = PAIRS && (bin.rows & kPair);
    double* const low = acc + rows;  // with pair
    uint2 next{0, 0};
    if (q0 + lane < q1) next = P.runs[q0 + lane];
    for (int i = lane; i < (pair ? 2 * rows : rows); i += kWave) acc[i] = 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (uint32_t q = q0; q < q1; q += kWave) {
      const uint2 mine = next;  // lanes past the last run: length 0
      next = make_uint2(0, 0);
      if (q + kWave + lane < q1) next = P.runs[q + kWave + lane];
      const int nr = static_cast<int>(q1 - q < kWave ? q1 - q : kWave);
      for (int i = 0; i < nr; i += kRuns) {
        uint32_t r[kRuns];
        double x[kRuns];
#pragma unroll
        for (int k = 0; k < kRuns; ++k) {
          const uint32_t g = __builtin_amdgcn_readlane(mine.x, i + k), len = __builtin_amdgcn_readlane(mine.y, i + k);
          r[k] = 0;
          x[k] = 0;
          if (static_cast<uint32_t>(lane) < len) {
            r[k] = P.row16[g + lane];
            x[k] = partial[g + lane];
          }
        }
        auto in_run = [&](int k) {
          return static_cast<uint32_t>(lane) < static_cast<uint32_t>(__builtin_amdgcn_readlane(mine.y, i + k));
        };
        if (pair) {
          double was[kRuns];
#pragma unroll
          for (int k = 0; k < kRuns; ++k)
            if (in_run(k)) was[k] = atomicAdd(&acc[r[k]], x[k]);
#pragma unroll
          for (int k = 0; k < kRuns; ++k)
            if (in_run(k)) {
              const double t = was[k] + x[k], b = t - was[k];
              atomicAdd(&low[r[k]], (was[k] - (t - b)) + (x[k] - b));
            }
        } else {
#pragma unroll
          for (int k = 0; k < kRuns; ++k)
            if (in_run(k)) atomicAdd(&acc[r[k]], x[k]);
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    constexpr int kU = 4;
    for (int i = lane; i < rows; i += kU * kWave) {
      typename Fin::Pre pre[kU];
#pragma unroll
      for (int k = 0; k < kU; ++k)
        if (i + k * kWave < rows) pre[k] = fin.pre(row0 + i + k * kWave);
      double t0 = 0, t1 = 0;
#pragma unroll
      for (int k = 0; k < kU; ++k)
        if (const int j = i + k * kWave; j < rows)
          fin(row0 + j, pair ? rs::DoubleSum{acc[j], low[j]}.value() : acc[j], pre[k], t0, t1);
      a0.add(t0);
      a1.add(t1);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  const double s0 = wave_sum(a0.value()), s1 = wave_sum(a1.value());
  if (lane == 0) {
    part0[blockIdx.x] = s0;
    part1[blockIdx.x] = s1;
  }
}

// Host: one sweep; wt null: unweighted.  Returns the number of partials
// written to part0/part1 (at most kSumGrid).
template <class Real, class Fin>
int launch(const Plan& P, const float* wt, const Real* y, int64_t n, double* partial, const Fin& fin,
           const unsigned* skip, double* part0, double* part1, hipStream_t s) {
  if (P.npieces > 0) {
    if (wt)
      gather_kernel<Real, true><<<static_cast<unsigned>(P.npieces), kGatherBlock, 0, s>>>(P, wt, y, n, partial, skip);
    else
      gather_kernel<Real, false><<<static_cast<unsigned>(P.npieces), kGatherBlock, 0, s>>>(P, wt, y, n, partial, skip);
    GX_LAUNCHED("bs::gather_kernel");
  }
  const int grid = static_cast<int>(std::min<int64_t>(P.nbins, kSumGrid));
  sum_kernel<sizeof(Real) == 8, Fin><<<grid, kWave, P.lds_sums * sizeof(double), s>>>(P, partial, fin, part0, part1, skip);
  GX_LAUNCHED("bs::sum_kernel");
  return grid;
}

}  // namespace bs
}  // namespace gx
