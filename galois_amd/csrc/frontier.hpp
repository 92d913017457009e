// Load-balanced neighbour expansion shared by the frontier-driven kernels
// (BFS, SSSP, k-core, CC hooking, BC forward).
//
// A workgroup of BLOCK lanes takes up to `most` frontier vertices (fewer when the
// frontier has fewer than that for every workgroup of the launch, see
// batch_vertices), exclusive-scans their degrees in LDS and walks the
// concatenated edge list with all lanes; the owning vertex of edge slot e is
// found by binary search over the LDS offsets.  Vertices whose degree exceeds `hub_thresh` are not expanded here:
// they are appended to a hub queue and their edges are later spread over the
// whole grid by expand_hubs.  This gives three effective tiers — short
// adjacencies packed many-per-wavefront, medium ones spread over the
// workgroup, hubs spread over the grid.
//
// The per-edge operation is called by every lane of the workgroup the same
// number of times (with `valid` false and edge 0 for padding lanes), so it may
// use wavefront-collective operations (ballot, shuffles).  With U > 1 a lane
// takes U edges of a step at once (op.run), so that their loads are in flight
// together.  After every step of BLOCK * U edges, every lane calls
// op.after_step() (workgroup-uniform), where an operation may flush its
// LDS-staged output (LdsQueue below).
//
// Counters shared by a whole launch (queue ends, sums) are single words, and
// atomics on one word are served one after another, about 12 ns each on this
// GPU whether or not the result is used (256 workgroups: 3 us, 2048: 25 us).
// So the operations count per workgroup first, a workgroup's counts go out in
// one packed 64-bit atomic where they can, and the launches with the most such
// traffic use few wide workgroups (kWideBlock lanes, kWideGrid workgroups).
#pragma once

#include "gx_device.hpp"

namespace gx {

constexpr int kWideBlock = 1024;
constexpr int kWideGrid = 256 * 2;
constexpr int kWideWaves = kWideBlock / kWave;
constexpr int kWideEdges = 4;                       // edges per lane and step of the wide launches
constexpr int kWideStep = kWave * kWideEdges;       // most items a wavefront pushes per step
constexpr int kWaveQCap = 2 * kWideStep;            // items a wavefront stages

// Frontier vertices a workgroup takes at a time: an equal share of the frontier
// between kBatchMin and `most`.  With whole blocks a frontier of a few thousand
// vertices kept a dozen workgroups busy, each walking up to 32K edges alone
// (BFS on 4096 vertices, 97K edges: one level 77 us).  More than kBatchMax at a
// time leave the last workgroups of a launch with uneven shares (directed BFS of
// 3 M vertices 628 us with 1024, 613 with 256).  Graphs without hubs take up to
// BLOCK: their edges are few and alike (`most`; k-core of a 2048 x 2048 lattice,
// all vertices at once, 271 us with 256, 209 with 1024).
constexpr unsigned kBatchMin = 4, kBatchMax = 256;
template <int BLOCK>
__device__ __forceinline__ unsigned batch_vertices(unsigned qcount, unsigned most) {
  const unsigned share = (qcount + gridDim.x - 1) / gridDim.x;
  if (most > BLOCK) most = BLOCK;
  return share < kBatchMin ? kBatchMin : (share < most ? share : most);
}

// Identity frontier (q null): vertex first + i for i in [0, count).
// Otherwise q[i].  With ADMIT, op.admit(v) is asked once per frontier vertex
// and a vertex it rejects contributes no edges (a fused filter).
template <int BLOCK, class Op, bool ADMIT = false, int U = 1>
__device__ __forceinline__ void expand_queue(const int32_t* __restrict__ row, const uint32_t* __restrict__ q,
                                             unsigned qcount, uint32_t hub_thresh, uint32_t* __restrict__ hubq,
                                             unsigned* hub_count, unsigned cap, unsigned* overflow, Op& op,
                                             uint32_t first = 0, unsigned most = kBatchMax) {
  __shared__ int32_t s_start[BLOCK];
  __shared__ uint32_t s_off[BLOCK];
  __shared__ uint32_t s_src[BLOCK];
  __shared__ uint64_t s_scan[BLOCK / kWave + 1];
  __shared__ unsigned s_hub_base;
  const unsigned tid = threadIdx.x;
  const unsigned per = batch_vertices<BLOCK>(qcount, most);
  for (uint64_t base = static_cast<uint64_t>(blockIdx.x) * per; base < qcount;
       base += static_cast<uint64_t>(gridDim.x) * per) {
    const unsigned i = static_cast<unsigned>(base) + tid;
    uint32_t v = 0, deg = 0;
    int32_t start = 0;
    bool hub = false;
    if (tid < per && i < qcount) {
      v = q ? q[i] : first + i;
      bool in = true;
      if constexpr (ADMIT) in = op.admit(v);
      if (in) {
        start = row[v];
        deg = static_cast<uint32_t>(row[v + 1] - start);
        if (deg > hub_thresh) {
          hub = true;
          deg = 0;
        }
      }
    }
    // One scan gives both the edge offsets (low 40 bits) and the hub slots
    // (high bits), so the hub list takes one global atomic per workgroup
    // batch instead of one per wavefront.
    uint64_t total64;
    const uint64_t ex64 = block_exclusive_scan<BLOCK>(static_cast<uint64_t>(deg) | (static_cast<uint64_t>(hub) << 40),
                                                      s_scan, &total64);
    constexpr uint64_t kLow = (uint64_t(1) << 40) - 1;
    const uint32_t excl = static_cast<uint32_t>(ex64 & kLow), total = static_cast<uint32_t>(total64 & kLow);
    const uint32_t hub_total = static_cast<uint32_t>(total64 >> 40);  // workgroup-uniform
    if (hubq && hub_total && tid == 0) s_hub_base = atomicAdd(hub_count, hub_total);
    s_start[tid] = start;
    s_off[tid] = excl;
    s_src[tid] = v;
    __syncthreads();
    if (hubq && hub) {
      const unsigned slot = s_hub_base + static_cast<uint32_t>(ex64 >> 40);
      if (slot < cap)
        hubq[slot] = v;
      else
        atomicOr(overflow, 1u);
    }
    for (uint32_t e0 = 0; e0 < total; e0 += BLOCK * U) {
      bool valid[U];
      uint32_t u[U];
      int32_t edge[U];
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const uint32_t e = e0 + k * BLOCK + tid;
        valid[k] = e < total;
        u[k] = 0;
        edge[k] = 0;
        if (valid[k]) {
          int lo = 0;
          if constexpr (BLOCK <= 256) {  // unrolled; lanes without a vertex hold the total, which is above e
#pragma unroll
            for (int step = BLOCK / 2; step > 0; step >>= 1)
              if (s_off[lo + step] <= e) lo += step;
          } else {
            int hi = static_cast<int>(per) - 1;
            while (lo < hi) {
              const int mid = (lo + hi + 1) >> 1;
              if (s_off[mid] <= e) lo = mid; else hi = mid - 1;
            }
          }
          u[k] = s_src[lo];
          edge[k] = s_start[lo] + static_cast<int32_t>(e - s_off[lo]);
        }
      }
      if constexpr (U == 1) op(valid[0], u[0], edge[0]);
      else op.run(valid, u, edge);
      op.after_step();
    }
    __syncthreads();
  }
}

// Step offsets of the hub list for expand_hubs, computed by
// kHubSlices workgroups: the hub list hubq[0..hubs) (hubs = min(*hub_count,
// cap); the count runs past cap when the hub queue overflowed, which the
// caller reports) is cut into kHubSlices slices of 2^hub_chunk_shift(hubs)
// hubs (the last ones may be empty), and slice k
// writes off[h] = sum over hubs h' < h of its own slice of ceil(deg(hubq[h'])
// / BLOCK) for its hubs h, and its total to off[cap + 1 + k].  expand_hubs
// adds the slice bases; it must be given the same `cap`.  `off` holds
// hub_off_words(cap) words.
constexpr int kHubSlices = 256;
constexpr int64_t hub_off_words(int64_t cap) { return cap + 1 + kHubSlices; }

// log2 of the slice length: the smallest power of two with
// kHubSlices << shift >= hubs (a shift, not a division, in the search).
__device__ __forceinline__ unsigned hub_chunk_shift(unsigned hubs) {
  unsigned sh = 0;
  while ((static_cast<uint64_t>(kHubSlices) << sh) < hubs) ++sh;
  return sh;
}

constexpr int kHubScanThreads = 256;

template <int BLOCK>
__global__ void __launch_bounds__(kHubScanThreads) hub_offsets_kernel(const int32_t* __restrict__ row,
                                                                      const uint32_t* __restrict__ hubq,
                                                                      const unsigned* __restrict__ hub_count,
                                                                      unsigned cap, uint32_t* __restrict__ off) {
  constexpr int NT = kHubScanThreads;
  __shared__ uint32_t lds[NT / kWave + 1];
  const unsigned hubs = min(*hub_count, cap);
  const unsigned sh = hub_chunk_shift(hubs);
  const unsigned b0 = static_cast<unsigned>(min(static_cast<uint64_t>(blockIdx.x) << sh, static_cast<uint64_t>(hubs)));
  const unsigned b1 = static_cast<unsigned>(min(static_cast<uint64_t>(b0) + (uint64_t(1) << sh), static_cast<uint64_t>(hubs)));
  uint32_t carry = 0;
  for (unsigned base = b0; base < b1; base += NT) {
    const unsigned i = base + threadIdx.x;
    uint32_t c = 0;
    if (i < b1) {
      const uint32_t v = hubq[i];
      c = static_cast<uint32_t>((row[v + 1] - row[v] + BLOCK - 1) / BLOCK);
    }
    uint32_t total;
    const uint32_t ex = block_exclusive_scan<NT>(c, lds, &total);
    if (i < b1) off[i] = carry + ex;
    carry += total;
  }
  if (threadIdx.x == 0) off[cap + 1 + blockIdx.x] = carry;
}

template <int BLOCK>
inline void launch_hub_offsets(const int32_t* row, const uint32_t* hubq, const unsigned* hub_count, unsigned cap,
                               uint32_t* off, hipStream_t s) {
  hub_offsets_kernel<BLOCK><<<kHubSlices, kHubScanThreads, 0, s>>>(row, hubq, hub_count, cap, off);
}

// Edges of the hub vertices hubq[0..hubs), cut into steps of LANES * U edges
// (a hub's steps are consecutive; hub_offsets_kernel<LANES * U> counted them).
// Each workgroup takes a contiguous range of steps, BLOCK / LANES at a time,
// one per group of LANES lanes: one binary search over the hub offsets (those
// of hub_offsets_kernel plus the scanned slice totals) finds the hub of a
// group's first step, and the following steps advance to the next hubs when
// they pass their first steps, so a step costs no search.
template <int BLOCK, class Op, int LANES = BLOCK, int U = 1>
__device__ __forceinline__ void expand_hubs(const int32_t* __restrict__ row, const uint32_t* __restrict__ hubq,
                                            unsigned hub_count, unsigned cap, const uint32_t* __restrict__ off,
                                            Op& op) {
  static_assert(BLOCK >= kHubSlices, "one slice total per lane");
  static_assert(BLOCK % LANES == 0 && LANES % kWave == 0, "groups are whole wavefronts");
  constexpr uint32_t kGroups = BLOCK / LANES;
  __shared__ uint32_t s_base[kHubSlices];
  __shared__ uint32_t s_scan[BLOCK / kWave + 1];
  __shared__ uint32_t s_total;
  const unsigned hubs = min(hub_count, cap);
  if (hubs == 0) return;
  const unsigned sh = hub_chunk_shift(hubs);
  {
    const uint32_t t = threadIdx.x < kHubSlices ? off[cap + 1 + threadIdx.x] : 0u;
    uint32_t total;
    const uint32_t ex = block_exclusive_scan<BLOCK>(t, s_scan, &total);
    if (threadIdx.x < kHubSlices) s_base[threadIdx.x] = ex;
    if (threadIdx.x == 0) s_total = total;
    __syncthreads();
  }
  const uint32_t total = s_total;
  const uint32_t per = (total + gridDim.x - 1) / gridDim.x;
  const uint32_t c0 = static_cast<uint32_t>(min(static_cast<uint64_t>(blockIdx.x) * per, static_cast<uint64_t>(total)));
  const uint32_t c1 = static_cast<uint32_t>(min(static_cast<uint64_t>(c0) + per, static_cast<uint64_t>(total)));
  if (c0 >= c1) return;
  const uint32_t group = threadIdx.x / LANES, lane = threadIdx.x % LANES;
  auto first_step = [&](unsigned h) { return off[h] + s_base[h >> sh]; };
  const uint32_t mine = min(c0 + group, total - 1);  // a step that exists, for the search
  unsigned lo = 0, hi = hubs - 1;  // last h with first_step(h) <= mine (steps >= 1 per hub: increasing)
  while (lo < hi) {
    const unsigned mid = (lo + hi + 1) >> 1;
    if (first_step(mid) <= mine) lo = mid; else hi = mid - 1;
  }
  unsigned h = lo;
  uint32_t first = first_step(h);
  uint32_t next = h + 1 < hubs ? first_step(h + 1) : total;
  uint32_t v = hubq[h];
  int64_t rb = row[v], re = row[v + 1];
  for (uint32_t base = c0; base < c1; base += kGroups) {  // workgroup-uniform
    const uint32_t c = base + group;
    const bool live = c < c1;
    if (live && c >= next) {  // uniform in the group; every hub has >= 1 step
      do {
        ++h;
        first = next;
        next = h + 1 < hubs ? first_step(h + 1) : total;
      } while (c >= next);
      v = hubq[h];
      rb = row[v];
      re = row[v + 1];
    }
    bool valid[U];
    uint32_t u[U];
    int32_t edge[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const int64_t e = rb + static_cast<int64_t>(c - first) * (LANES * U) + k * LANES + lane;
      valid[k] = live && e < re;
      u[k] = v;
      edge[k] = valid[k] ? static_cast<int32_t>(e) : 0;
    }
    if constexpr (U == 1) op(valid[0], u[0], edge[0]);
    else op.run(valid, u, edge);
    op.after_step();
  }
}

// Workgroup-private output queue in LDS.  Lanes append with one LDS atomic
// per wavefront; the workgroup moves the items to the global queue with one
// global atomic per flush (coalesced stores), instead of one global atomic
// per wavefront per step on a single hot counter.
template <int CAP>
struct LdsQueue {
  uint32_t items[CAP];
  unsigned count;
  unsigned gbase;
};

template <int CAP>
__device__ __forceinline__ void lq_init(LdsQueue<CAP>& q) {
  if (threadIdx.x == 0) q.count = 0;
  __syncthreads();
}

// Room is guaranteed by flushing whenever fewer than one step's worth
// (blockDim.x items) of space is left.
template <int CAP>
__device__ __forceinline__ void lq_push(LdsQueue<CAP>& q, bool pred, uint32_t v) {
  const uint64_t mask = __ballot(pred);
  if (mask == 0) return;
  const unsigned leader = __ffsll(static_cast<unsigned long long>(mask)) - 1;
  unsigned base = 0;
  if (lane_id() == leader) base = atomicAdd(&q.count, static_cast<unsigned>(__popcll(mask)));
  base = __shfl(base, leader);
  if (pred) q.items[base + lanes_below(mask)] = v;
}

// Workgroup-uniform: every lane of the workgroup must call it.  Flushes when
// `force` or when the queue is nearly full.
template <int CAP>
__device__ __forceinline__ void lq_flush(LdsQueue<CAP>& q, uint32_t* __restrict__ gq, unsigned* gcount, unsigned cap,
                                         unsigned* overflow, bool force) {
  __syncthreads();
  const unsigned cnt = q.count;
  __syncthreads();
  if (!force && cnt + blockDim.x <= CAP) return;
  if (cnt == 0) return;
  if (threadIdx.x == 0) q.gbase = atomicAdd(gcount, cnt);
  __syncthreads();
  const unsigned base = q.gbase;
  for (unsigned i = threadIdx.x; i < cnt; i += blockDim.x) {
    if (base + i < cap)
      gq[base + i] = q.items[i];
    else
      atomicOr(overflow, 1u);
  }
  __syncthreads();
  if (threadIdx.x == 0) q.count = 0;
  __syncthreads();
}

// Output queue of one wavefront in LDS, its length in a register: a push costs
// no LDS atomic and a flush no workgroup barrier, so the wavefronts of a
// workgroup run on at their own pace between two batches of vertices.
template <int CAP>
struct WaveQueue {
  uint32_t* items;     // CAP words of LDS of this wavefront
  unsigned count = 0;  // wavefront-uniform
  // U items per lane; room for kWave * U is the caller's to see to.
  template <int U>
  __device__ __forceinline__ void push(const bool (&pred)[U], const uint32_t (&v)[U]) {
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const uint64_t mask = __ballot(pred[k]);
      if (pred[k]) items[count + lanes_below(mask)] = v[k];
      count += static_cast<unsigned>(__popcll(mask));
    }
  }
  __device__ __forceinline__ bool full(unsigned step) const { return count + step > CAP; }
  // Stores the items to gq[base, base + count), bounded by cap.
  __device__ __forceinline__ void store(unsigned base, uint32_t* __restrict__ gq, unsigned cap, unsigned* overflow) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (unsigned i = lane_id(); i < count; i += kWave) {
      if (base + i < cap)
        gq[base + i] = items[i];
      else
        atomicOr(overflow, 1u);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    count = 0;
  }
};

// Workgroup-uniform: the sum of one wavefront-uniform value per wavefront and
// the sum of those of earlier wavefronts.  lds: BLOCK / kWave + 1 words.
template <int BLOCK>
__device__ __forceinline__ unsigned long long waves_exclusive_sum(unsigned long long v, unsigned long long* lds,
                                                                  unsigned long long* total) {
  constexpr int kW = BLOCK / kWave;
  const unsigned w = threadIdx.x / kWave;
  if (lane_id() == 0) lds[w] = v;
  __syncthreads();
  // A lane per wavefront: an unrolled loop over 16 words would hold them all in
  // registers and halve the wavefronts that fit a CU.
  const unsigned lane = lane_id();
  const unsigned long long x = lane < kW ? lds[lane] : 0ull;
  *total = wave_sum(x);
  const unsigned long long before = wave_sum(lane < w ? x : 0ull);
  return before;
}

// Segmented inclusive sum across a wavefront where equal `key`s form
// contiguous runs of lanes (invalid lanes carry a key no valid lane has).
// Returns the run total in the last lane of each run (is_tail set).
template <class T>
__device__ __forceinline__ T wave_segmented_sum(uint32_t key, T v, bool& is_tail) {
  const unsigned lane = lane_id();
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const T ov = __shfl_up(v, off);
    const uint32_t ok = __shfl_up(key, off);
    if (lane >= static_cast<unsigned>(off) && ok == key) v += ov;
  }
  const uint32_t nk = __shfl_down(key, 1);
  is_tail = (lane == kWave - 1) || (nk != key);
  return v;
}

}  // namespace gx
