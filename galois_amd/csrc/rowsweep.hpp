// Deterministic, load-balanced row sums over a CSR/CSC: sum_{e in row r}
// value(e, col[e]) for every row, the pull step of PageRank (over the
// transpose) and of its adjoint (over the CSR).
//
// Layout.  The edges are cut into tiles of kTile = 512 (8 per lane of one
// wavefront); `kt` consecutive tiles are a chunk, which one wavefront sums
// from front to back.  A static plan holds, per lane and tile, which of the
// lane's 8 edges end a row and how many rows of the tile end before them
// (one word), per tile the index of its first row among the rows that have
// edges, and those rows' ids in order.  Rows without edges are listed behind
// them and finalised in a pass of their own, so that a tile costs the same
// whatever the degrees.
//
// Tile work (one wavefront, no workgroup barrier).
//  1. The columns of the tile are loaded with consecutive lanes on consecutive
//     edges (gathers of neighbouring sources then share cache lines), the
//     values gathered and laid down in LDS.
//  2. Each lane reads its 8 consecutive values and sums what follows its last
//     row end; a segmented scan of those sums over the lanes (DPP, fixed
//     order) gives every lane the open sum it continues.
//  3. The lane walks its values once more and stores a row sum to LDS at each
//     row end, the first one with the open sum added: values are summed among
//     themselves before they meet the sum of a long row.
//  4. Consecutive lanes finalise consecutive rows.
// The sum left open at a tile's end is carried in a register to the next tile
// of the chunk.  A row that began in an earlier chunk is not finalised where
// it ends: the chunk stores its part (head), every chunk stores the sum of
// the row open at its end (tail), and a second launch adds the tails of the
// earlier chunks and the head, in a fixed order, and finalises those rows.
// Sums are FP64 for both precisions (the FP32 values are summed in FP64, which
// on this GPU takes one conversion and one addition where a compensated FP32
// sum takes six operations); every order is fixed, so results are
// bit-reproducible run to run.
//
// Bound: the gathers.  One request per edge reaches the L2 at about 130 G/s
// whatever the occupancy (67M edges, 4.2M rows, FP32 with weights: 555 us;
// 20.6M edges, 1.5M rows, FP64: 156 us, where a version with 512-lane
// workgroups, a merge-path search per lane and workgroup barriers took 172 us
// and 15 wavefronts fewer per CU), so what is left to save here is the fixed
// cost of a small sweep.
//
// Src  : static constexpr bool kCol (false: the value does not need the column)
//        __device__ Real operator()(int64_t e, int32_t c) const  (value of
//        edge slot e whose column id is c)
// Fin  : __device__ void load()  (read per-sweep scalars, once per thread)
//        struct Pre; __device__ Pre pre(uint32_t r) const  (per-row operands,
//        loaded early so their latency overlaps the tile's gathers)
//        __device__ void operator()(uint32_t r, double sum, const Pre&,
//        double& a0, double& a1) const  (finalise row r; two FP64
//        per-workgroup accumulators, e.g. residual and dangling mass)
#pragma once

#include <algorithm>
#include <climits>
#include <cmath>

#include "gx_device.hpp"
#include "gx_internal.hpp"

namespace gx {
namespace rs {

constexpr int kBlock = 256;          // 4 wavefronts
constexpr int kWaves = kBlock / kWave;
constexpr int kItems = 8;            // edges per lane and tile
constexpr int kTile = kWave * kItems;
constexpr int kSweepGrid = 256 * 8;  // workgroups of the sweep: 8 per CU
constexpr int kFixGrid = 256;        // most workgroups of the spanning-row launch
constexpr int kParts = kSweepGrid + kFixGrid;

// Workgroup sum of one double per lane in a fixed order (valid in lane 0);
// NT = threads of the workgroup, lds holds NT / 64 doubles.
template <int NT = kBlock>
__device__ __forceinline__ double block_sum(double v, double* lds) {
  v = wave_sum(v);
  const unsigned w = threadIdx.x / kWave;
  if (lane_id() == 0) lds[w] = v;
  __syncthreads();
  double r = 0;
  if (threadIdx.x == 0)
    for (int i = 0; i < NT / kWave; ++i) r += lds[i];
  __syncthreads();
  return r;
}

// A sum and, in lo, what its additions rounded off (Knuth's TwoSum): a long row's
// is rounded once, however many parts it has.
struct DoubleSum {
  double hi = 0, lo = 0;
  __device__ __forceinline__ void add(double x) {
    const double t = hi + x, b = t - hi;
    lo += (hi - (t - b)) + (x - b);
    hi = t;
  }
  // hi alone where the sum is not finite (lo then means nothing).
  __device__ __forceinline__ double value() const { return isfinite(lo) ? hi + lo : hi; }
};

template <class T>
__device__ __forceinline__ T ld_stream(const T* p) {
  return __builtin_nontemporal_load(p);
}

constexpr uint32_t kNoRow = 0xffffffffu;

struct RowPlan {
  const int32_t* rowoff;      // n+1
  const int32_t* col;         // len
  int64_t n;                  // rows
  int64_t len;                // edges
  const uint32_t* rid;        // rows with edges, ascending, then the rows without
  int64_t full;               // rows with edges
  const uint32_t* tile_row;   // ntiles+1: index in rid of the row of each tile's first edge
  const uint32_t* lane_info;  // ntiles*64: bits 0..7 row ends, bits 8.. rows of the tile ended before
  const uint32_t* span_row;    // nchunks: row that spans chunks and ends in this one, or kNoRow
  const uint32_t* span_first;  // nchunks: the chunk it begins in
  int64_t ntiles, nchunks;
  int kt;                     // tiles per chunk
};

// Builds (or returns the cached) plan of a row-offset array; defined in
// rowsweep.hip.
RowPlan build_plan(gx_graph* g, const int32_t* rowoff, const int32_t* col, int64_t n, int64_t m, PullPlan& cache);

// Tiles per chunk.
inline int tiles_per_chunk(int64_t ntiles) {
  return static_cast<int>(std::min<int64_t>(8, std::max<int64_t>(1, ntiles / (4 * kSweepGrid * kWaves))));
}

template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_f64(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b), CTRL, ROWS, 0xf, false);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), CTRL, ROWS, 0xf, false);
  return __builtin_bit_cast(double, (static_cast<uint64_t>(hi) << 32) | lo);
}

// Inclusive sum over lanes first..lane (first <= lane, the same for every lane
// of a segment).  Fixed order: within rows of 16 lanes by shifts, then across
// rows by broadcasts of their last lanes.
__device__ __forceinline__ double wave_seg_scan(double v, int first, int lane) {
  const int in_row = lane & 15;
  double o;
  o = dpp_f64<0x111, 0xf>(v);
  if (in_row >= 1 && lane - 1 >= first) v += o;
  o = dpp_f64<0x112, 0xf>(v);
  if (in_row >= 2 && lane - 2 >= first) v += o;
  o = dpp_f64<0x114, 0xf>(v);
  if (in_row >= 4 && lane - 4 >= first) v += o;
  o = dpp_f64<0x118, 0xf>(v);
  if (in_row >= 8 && lane - 8 >= first) v += o;
  o = dpp_f64<0x142, 0xa>(v);  // lane 15 of rows 0 and 2 to rows 1 and 3
  if ((lane & 16) && (lane | 15) - 16 >= first) v += o;
  o = dpp_f64<0x143, 0xc>(v);  // lane 31 to rows 2 and 3
  if ((lane & 32) && 31 >= first) v += o;
  return v;
}

// One LDS area per wavefront: first the tile's values (one pad word per kItems,
// which spreads the lanes' reads over the banks), then its row sums.
template <class Real>
union WaveShared {
  Real val[kTile + kTile / kItems];
  double sum[kTile];
};

// One launch over every chunk (chunk c on wavefront c mod the grid's) and the
// rows without edges.  Workgroup partials of the two accumulators go to
// part0/part1[blockIdx.x].  Returns at once when *skip is non-zero (a
// converged iteration loop).  carry: 2 * nchunks.
template <class Real, class Src, class Fin>
__global__ void __launch_bounds__(kBlock) sweep_kernel(RowPlan P, Src src, Fin fin, const unsigned* __restrict__ skip,
                                                       double* __restrict__ part0, double* __restrict__ part1,
                                                       double* __restrict__ carry) {
  if (skip && *skip) return;
  fin.load();
  __shared__ WaveShared<Real> shared[kWaves];
  __shared__ double red[kWaves];
  const int lane = static_cast<int>(lane_id());
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  WaveShared<Real>& sh = shared[wid];
  double a0 = 0, a1 = 0;
  const int64_t nwaves = static_cast<int64_t>(gridDim.x) * kWaves;
  for (int64_t c = static_cast<int64_t>(blockIdx.x) * kWaves + wid; c < P.nchunks; c += nwaves) {
    const int64_t T0 = c * P.kt, T1 = T0 + P.kt < P.ntiles ? T0 + P.kt : P.ntiles;
    uint32_t k0 = P.tile_row[T0];
    // The chunk's first row began in an earlier chunk.
    bool defer = P.rowoff[P.rid[k0]] < T0 * kTile;
    double open = 0;  // sum of the row open at the start of the tile (uniform)
    for (int64_t T = T0; T < T1; ++T) {
      const int64_t e0 = T * kTile;
      const int ned = static_cast<int>(P.len - e0 < kTile ? P.len - e0 : kTile);
      const uint32_t k1 = P.tile_row[T + 1];
      const int nrow = static_cast<int>(k1 - k0);  // rows that end in this tile
      int32_t cc[kItems];
      if constexpr (Src::kCol) {
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
          const int j = lane + i * kWave;
          cc[i] = j < ned ? ld_stream(&P.col[e0 + j]) : 0;
        }
      }
      const uint32_t info = ld_stream(&P.lane_info[T * kWave + lane]);
      const uint32_t row = lane < nrow ? P.rid[k0 + lane] : 0u;
      const typename Fin::Pre pre = lane < nrow ? fin.pre(row) : typename Fin::Pre{};
      Real v[kItems];
#pragma unroll
      for (int i = 0; i < kItems; ++i) {
        const int j = lane + i * kWave;
        v[i] = j < ned ? src(e0 + j, Src::kCol ? cc[i] : 0) : Real(0);
      }
#pragma unroll
      for (int i = 0; i < kItems; ++i) {
        const int j = lane + i * kWave;
        sh.val[j + j / kItems] = v[i];
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int u = 0; u < kItems; ++u) v[u] = sh.val[lane * (kItems + 1) + u];
      // Sum after the lane's last row end, scanned over the lanes.
      const uint32_t ends = info & 0xffu;
      double tail = 0;
#pragma unroll
      for (int u = 0; u < kItems; ++u) {
        tail += static_cast<double>(v[u]);
        if ((ends >> u) & 1u) tail = 0;
      }
      const uint64_t heads = __ballot(ends != 0);
      const uint64_t upto = heads & (~0ull >> (63 - lane));
      const double seg = wave_seg_scan(tail, upto ? 63 - __builtin_clzll(upto) : 0, lane);
      double before = __shfl_up(seg, 1);
      if (lane == 0) before = 0;
      if ((heads & ((1ull << lane) - 1)) == 0) before += open;
      const double last = __shfl(seg, kWave - 1);
      open = heads ? last : open + last;
      // Row sums (the values are in registers: the LDS area is free).
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      uint32_t slot = info >> 8;
      double acc = 0;
#pragma unroll
      for (int u = 0; u < kItems; ++u) {
        acc += static_cast<double>(v[u]);
        if ((ends >> u) & 1u) {
          sh.sum[slot++] = before + acc;
          before = acc = 0;
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (lane < nrow) {
        const double s = sh.sum[lane];
        if (lane == 0 && defer)
          carry[c] = s;  // head of a row that began in an earlier chunk
        else
          fin(row, s, pre, a0, a1);
      }
      for (int j = lane + kWave; j < nrow; j += kWave) {
        const uint32_t r = P.rid[k0 + j];
        fin(r, sh.sum[j], fin.pre(r), a0, a1);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (nrow > 0) defer = false;
      k0 = k1;
    }
    if (lane == 0) carry[P.nchunks + c] = open;
  }
  // Rows without edges.
  for (int64_t i = P.full + static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < P.n;
       i += static_cast<int64_t>(gridDim.x) * kBlock) {
    const uint32_t r = P.rid[i];
    fin(r, 0.0, fin.pre(r), a0, a1);
  }
  a0 = block_sum(a0, red);
  a1 = block_sum(a1, red);
  if (threadIdx.x == 0) {
    part0[blockIdx.x] = a0;
    part1[blockIdx.x] = a1;
  }
}

// Rows that span chunks: the tails of the chunks before the one where the row
// ends, then that chunk's head.  A lane per chunk; the wavefront sums the tails
// of long spans together (a hub's are thousands).
// The accumulators are this lane's.
template <int NT, class Fin>
__device__ __forceinline__ void finalize_spans(const RowPlan& P, const Fin& fin, const double* __restrict__ carry,
                                               double& a0, double& a1) {
  const int lane = static_cast<int>(lane_id());
  const int64_t stride = static_cast<int64_t>(gridDim.x) * NT;
  for (int64_t b = static_cast<int64_t>(blockIdx.x) * NT + (threadIdx.x & ~(kWave - 1)); b < P.nchunks; b += stride) {
    const int64_t c = b + lane;
    const uint32_t r = c < P.nchunks ? P.span_row[c] : kNoRow;
    const bool spans = r != kNoRow;
    const uint32_t first = spans ? P.span_first[c] : 0u;
    const double head = spans ? carry[c] : 0.0;
    const typename Fin::Pre pre = spans ? fin.pre(r) : typename Fin::Pre{};
    DoubleSum sum;
    // Short spans by their own lane, long ones by the whole wavefront.
    constexpr int kAlone = 8;
    if (spans && c - first <= kAlone)
      for (int64_t t = first; t < c; ++t) sum.add(carry[P.nchunks + t]);
    for (uint64_t todo = __ballot(spans && c - first > kAlone); todo; todo &= todo - 1) {
      const int i = __ffsll(static_cast<unsigned long long>(todo)) - 1;
      const int64_t f = __shfl(first, i), e = b + i;
      DoubleSum s;
      for (int64_t t = f + lane; t < e; t += kWave) s.add(carry[P.nchunks + t]);
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        const double oh = __shfl_xor(s.hi, off), ol = __shfl_xor(s.lo, off);
        s.add(oh);
        s.lo += ol;
      }
      if (lane == i) sum = s;
    }
    if (spans) {
      sum.add(head);
      fin(r, sum.value(), pre, a0, a1);
    }
  }
}

template <class Fin>
__global__ void __launch_bounds__(kBlock) span_finalize_kernel(RowPlan P, Fin fin, const unsigned* __restrict__ skip,
                                                               const double* __restrict__ carry,
                                                               double* __restrict__ part0,
                                                               double* __restrict__ part1) {
  if (skip && *skip) return;
  fin.load();
  __shared__ double red[kWaves];
  double a0 = 0, a1 = 0;
  finalize_spans<kBlock>(P, fin, carry, a0, a1);
  a0 = block_sum(a0, red);
  a1 = block_sum(a1, red);
  if (threadIdx.x == 0) {
    part0[blockIdx.x] = a0;
    part1[blockIdx.x] = a1;
  }
}

// The same in one workgroup, which also adds up the accumulators of the sweep
// (nparts partials) and hands their sums to close, once: the end of an
// iteration in one launch instead of two.  For up to kCloseChunks chunks, two
// rounds of the workgroup (1 M edges; the launch it saves takes 4 us, a further
// round 3; which rows span is in the plan): FP64 PageRank of 4096 vertices
// 327 -> 289 us, of 77,000 (0.5 M edges) 700 -> 640, adjoint of 4096 2.49 -> 2.14
// ms.
constexpr int kCloseBlock = 1024;
constexpr int64_t kCloseChunks = 2 * kCloseBlock;
template <class Fin, class Close>
__global__ void __launch_bounds__(kCloseBlock) span_close_kernel(RowPlan P, Fin fin,
                                                                 const unsigned* __restrict__ skip,
                                                                 const double* __restrict__ carry,
                                                                 const double* __restrict__ part0,
                                                                 const double* __restrict__ part1, int nparts,
                                                                 Close close) {
  if (skip && *skip) return;
  fin.load();
  __shared__ double red[kCloseBlock / kWave];
  double a0 = 0, a1 = 0;
  for (int i = threadIdx.x; i < nparts; i += kCloseBlock) {
    a0 += part0[i];
    a1 += part1[i];
  }
  finalize_spans<kCloseBlock>(P, fin, carry, a0, a1);
  a0 = block_sum<kCloseBlock>(a0, red);
  a1 = block_sum<kCloseBlock>(a1, red);
  if (threadIdx.x == 0) close(a0, a1);
}

// A sweep that leaves its accumulators as partials.
struct NoClose {};

// Host: one full sweep (tile launch + spanning-row launch) on stream s.
// part0/part1 hold kParts entries each and carry 2 * P.nchunks; returns the
// number of partials written (at most kParts, contiguous from 0), or 0 when
// `close` has got their sums (small sweeps, see span_close_kernel).  `timer`
// brackets the tile launch.
template <class Real, class Src, class Fin, class Close = NoClose>
int launch_sweep(const RowPlan& P, const Src& src, const Fin& fin, const unsigned* skip, double* part0,
                 double* part1, double* carry, hipStream_t s, KernelTimer* timer, const Close& close = Close{}) {
  const int64_t items = std::max<int64_t>(P.nchunks * kWave, P.n - P.full);
  const int grid = static_cast<int>(grid_for(items, kBlock, kSweepGrid));
  if (timer) timer->begin();
  sweep_kernel<Real, Src, Fin><<<grid, kBlock, 0, s>>>(P, src, fin, skip, part0, part1, carry);
  if (timer) timer->end();
  GX_LAUNCHED("sweep_kernel");
  if constexpr (!std::is_same<Close, NoClose>::value) {
    if (P.nchunks <= kCloseChunks) {
      span_close_kernel<Fin, Close><<<1, kCloseBlock, 0, s>>>(P, fin, skip, carry, part0, part1, grid, close);
      GX_LAUNCHED("span_close_kernel");
      return 0;
    }
  }
  const int fix = static_cast<int>(grid_for(P.nchunks, kBlock, kFixGrid));
  span_finalize_kernel<Fin><<<fix, kBlock, 0, s>>>(P, fin, skip, carry, part0 + grid, part1 + grid);
  GX_LAUNCHED("span_finalize_kernel");
  return grid + fix;
}

}  // namespace rs
}  // namespace gx
