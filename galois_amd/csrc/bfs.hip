// Breadth-first search: level-synchronous top-down BFS and the
// direction-optimising (push/pull) BFS.
//
// Reference semantics
//  - lonestar/analytics/cpu/bfs/bfs.cpp:245-293 (syncAlgo): level[src] = 0,
//    level[dst] = L+1 the first time dst is seen from a level-L vertex,
//    unreached = DIST_INFINITY (BFS_SSSP.h:31-32).  Levels are unique, so the
//    result is bit-exact whatever the order of discovery.
//  - lonestar/analytics/cpu/bfs/bfsDirectionOpt.cpp:205-342 (syncDOAlgo):
//    push while the scout count (edges out of the new frontier) is at most
//    edges_to_check/alpha; otherwise pull over in-edges against a frontier
//    bitmap, stopping at the first frontier neighbour, and keep pulling while
//    the frontier grows or holds more than n/beta vertices.
//
// Design (gfx950)
//  - Top-down expansion uses the load-balanced workgroup expansion of
//    frontier.hpp (degree above frontier.hub_degree, 128 by default, goes
//    to a grid-wide hub pass).  Discovery is
//    an atomicCAS on the level word, so each vertex enters the next frontier
//    once.  New vertices are staged per wavefront in LDS; a workgroup takes
//    room for what is left at its end, and adds the degrees of what it found,
//    with one atomic on one packed word (see frontier.hpp: with 2048
//    workgroups and two words, two thirds of an RMAT-18 level went into
//    them; RMAT-18 375 -> 286 us, direction-optimising RMAT-24 1209 -> 1004
//    us, 4096 vertices 248 -> 153 us, most of the last from spreading small
//    frontiers over more workgroups).
//  - gx_bfs drives its levels on the device from a state word: runs of small
//    levels in one workgroup (narrow_kernel), larger ones as a fixed kernel
//    sequence (expand, hubs, narrow); a few such levels are captured in a HIP
//    graph and replayed until the frontier is empty.
//  - On symmetric graphs with hubs the heavy levels of gx_bfs are pulled
//    instead (level_begin): RMAT-18 240 -> 115 us, 4 M vertices 1272 -> 282 us,
//    where 130 G neighbour levels a second bound the push.
//  - Pulls test a 1-bit-per-vertex frontier bitmap (n/8 bytes, L2 resident for
//    the graphs here), four neighbours at a time, and stop at the first hit
//    (RMAT-24: the three pulls of the direction-optimising BFS 684 -> 346 us;
//    the call, with one wait per level instead of up to three, 1177 -> 560;
//    with pull_vertex 432).
#include <algorithm>

#include "frontier.hpp"
#include "gx_device.hpp"
#include "gx_internal.hpp"

using namespace gx;

namespace {

constexpr int kBlock = 256;
constexpr uint32_t kInf = GX_DIST_INFINITY;
constexpr uint32_t kNoParent = 0xffffffffu;
// Graphs without hubs (maximum degree at or below the hub threshold, such as
// road-like grids) have small frontiers per level and many levels: a quarter
// of the workgroups start faster.
constexpr int kGridNoHubs = 128;
constexpr int kHubLanes = 64;  // lanes per step of the hub pass
constexpr int kLevelsPerGraph = 4;
// Wide levels of the first replay: what power-law graphs need.  A level that
// is not needed costs 6-7 us, a second replay with its wait 60.  Below 2^18
// edges the one-workgroup levels leave at most three (4096 vertices, 97K edges
// 98 -> 92 us; 1100 to 10,000 vertices 89-103 -> 83-97; with two, 8000 vertices
// go from 100 to 136), above it the fourth is needed.  Graphs without hubs
// have tens of levels: with fewer in the first replay a lattice of 20,000
// vertices goes from 275 us to 305.
constexpr int kLevelsFirst = 4, kLevelsFirstSmall = 3;
constexpr int64_t kSmallEdges = int64_t(1) << 18;

struct BfsState {
  unsigned count[2];      // frontier sizes (double buffered by q)
  unsigned hub_count;
  unsigned overflow;
  unsigned q;             // frontier read this level
  unsigned level;         // level being written
  unsigned active;        // this level has a frontier
  unsigned pull;          // this level is pulled (gx_bfs)
  unsigned done;
  // Vertices discovered this level (low 32 bits: also the end of the queue a
  // push fills) and their degree sum (high 32 bits; it is at most m < 2^31),
  // so that a workgroup adds both with one atomic.
  unsigned long long app;
  unsigned long long scout;  // degree sum of the vertices discovered this level
  unsigned long long edges;  // degree sum of every discovered vertex
  unsigned long long items;
  // Output arrays of the current call, read by the captured level kernels
  // (so the captured graph does not depend on the caller's buffers).
  uint32_t* level_out;
  uint32_t* parent_out;
};

struct Bufs {
  const int32_t* row;
  const int32_t* col;
  uint32_t* level;
  uint32_t* parent;
  uint32_t* q[2];
  uint32_t* hubq;
  BfsState* S;
  unsigned cap;
  uint32_t* hub_off;
  uint32_t hub;   // frontier.hub_degree
  uint32_t* vis;  // visited bitmap (gx_bfs only; null for the DO-BFS)
  uint64_t* front;    // frontier bitmap of a pulled level (gx_bfs)
  int64_t n, m;
  // On the degree-ordered copy: every vertex's first neighbour, and the number
  // of vertices with edges (the first ones); otherwise null and n.
  const uint32_t* first;
  int64_t nonzero;
  uint64_t pull_min;    // fewest edges out of a frontier that is pulled
  uint64_t narrow_max;  // most edges out of a frontier that a narrow level takes
  unsigned batch;       // most vertices a workgroup takes at a time
};

// Levels, parents and the visited bitmap of a search that has found its source,
// and its state.  src_map (may be null): the source's id in the graph the
// search runs on.
__global__ void bfs_init_kernel(Bufs B, int64_t n, uint32_t src, const uint32_t* __restrict__ src_map) {
  if (src_map) src = src_map[src];
  const int64_t first = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t v = first; v < n; v += stride) {
    B.level[v] = (v == src) ? 0u : kInf;
    if (B.parent) B.parent[v] = (v == src) ? src : kNoParent;
  }
  if (B.vis)
    for (int64_t w = first; w < (n + 31) / 32; w += stride) B.vis[w] = w == src / 32 ? 1u << (src & 31) : 0u;
  if (first == 0) {
    BfsState* S = B.S;
    S->level_out = B.level;
    S->parent_out = B.parent;
    S->count[0] = 1;
    S->count[1] = 0;
    S->hub_count = 0;
    S->overflow = 0;
    S->q = 0;
    S->level = 0;
    S->active = 0;
    S->pull = 0;
    S->done = 0;
    S->app = 0;
    S->scout = static_cast<unsigned>(B.row[src + 1] - B.row[src]);
    S->edges = S->scout;
    S->items = 1;
    B.q[0][0] = src;
  }
}

// A level is pulled when the edges out of its frontier are many (pull_min, a
// quarter of the vertices: the pull reads every vertex's level and the rows of
// the unreached) and at least an eighth of those out of the unreached vertices
// (the most a pull could walk; most scans end at their first neighbours).
// RMAT-18, symmetric: the two heavy levels took 89 and 92 us pushed.
constexpr int kPullShare = 8;

__device__ __forceinline__ void level_begin(const Bufs& B) {
  BfsState* S = B.S;
  if (S->done || S->overflow || S->count[S->q] == 0) {
    S->active = 0;
    S->done = 1;
    return;
  }
  S->active = 1;
  S->level += 1;
  S->app = 0;
  S->hub_count = 0;
  S->pull = S->scout > B.pull_min && S->scout * kPullShare > static_cast<uint64_t>(B.m) - S->edges;
}

__device__ __forceinline__ void level_end(BfsState* S) {
  if (!S->active) return;
  S->q ^= 1;
  S->count[S->q] = static_cast<unsigned>(S->app);
  S->scout = S->app >> 32;
  S->items += S->count[S->q];
  S->edges += S->scout;
  S->active = 0;
}

// Plain pointers only: the output arrays come from the device state and the
// next queue is picked by the state's index, so the kernel-argument Bufs is
// never copied or modified (a modified copy, with its runtime-indexed queue
// array, would be kept in scratch memory).
struct TdOp {
  const int32_t* __restrict__ row;
  const int32_t* __restrict__ col;
  uint32_t* level;
  uint32_t* parent;
  uint32_t* qout;
  unsigned cap;
  BfsState* S;
  WaveQueue<kWaveQCap> wq;
  uint32_t nl;
  unsigned long long scout;  // this lane's degree sum of discovered vertices
  uint32_t* vis;
  // With a visited bitmap (n/8 bytes, mostly cache-resident) an edge to an
  // already discovered vertex is dropped without the random read of its
  // level word; a bit set late only sends the edge on to the level check.
  template <int U>
  __device__ __forceinline__ void run(const bool (&valid)[U], const uint32_t (&u)[U], const int32_t (&e)[U]) {
    bool won[U];
    uint32_t v[U], lv[U];
#pragma unroll
    for (int k = 0; k < U; ++k) v[k] = static_cast<uint32_t>(col[e[k]]);
    if (vis) {
#pragma unroll
      for (int k = 0; k < U; ++k) won[k] = valid[k] && !((vis[v[k] >> 5] >> (v[k] & 31)) & 1u);
#pragma unroll
      for (int k = 0; k < U; ++k) lv[k] = won[k] ? level[v[k]] : 0u;
    } else {
#pragma unroll
      for (int k = 0; k < U; ++k) lv[k] = level[v[k]];
    }
#pragma unroll
    for (int k = 0; k < U; ++k) {
      won[k] = valid[k] && lv[k] == kInf && atomicCAS(&level[v[k]], kInf, nl) == kInf;
      if (won[k]) {
        if (vis) atomicOr(&vis[v[k] >> 5], 1u << (v[k] & 31));
        if (parent) parent[v[k]] = u[k];
        scout += static_cast<unsigned long long>(row[v[k] + 1] - row[v[k]]);
      }
    }
    wq.push(won, v);
  }
  // Room in the next queue, and the degree sum of what was found, with one atomic.
  __device__ __forceinline__ void after_step() {
    if (!wq.full(kWideStep)) return;
    unsigned base = 0;
    if (lane_id() == 0) base = static_cast<unsigned>(atomicAdd(&S->app, static_cast<unsigned long long>(wq.count)));
    wq.store(__builtin_amdgcn_readfirstlane(base), qout, cap, &S->overflow);
  }
  // Workgroup-uniform: what is left, for all wavefronts at once.
  __device__ __forceinline__ void finish() {
    __shared__ unsigned long long s_sum[kWideWaves + 1];
    unsigned long long total;
    const unsigned long long before =
        waves_exclusive_sum<kWideBlock>(wq.count | (wave_sum(scout) << 32), s_sum, &total);
    if (threadIdx.x == 0) s_sum[kWideWaves] = total ? atomicAdd(&S->app, total) : 0ull;
    __syncthreads();
    wq.store(static_cast<unsigned>(s_sum[kWideWaves]) + static_cast<unsigned>(before), qout, cap, &S->overflow);
  }
};

__device__ __forceinline__ TdOp make_td(const Bufs& B, uint32_t (&stage)[kWideWaves][kWaveQCap]) {
  BfsState* S = B.S;
  return TdOp{B.row, B.col, S->level_out, S->parent_out, B.q[S->q ^ 1], B.cap, S, {stage[threadIdx.x / kWave]},
              S->level, 0ull, B.vis};
}

// Per lane: whether one of the in-neighbours col[begin, end) is in the frontier
// bitmap, and the first found (`who`).  Called by whole wavefronts (lanes
// without a vertex: begin == end).  A lane tests its first kPullSerial
// neighbours itself, four in flight; what is left of longer lists is walked by
// the wavefront together, one list after another, so that an unreached hub does
// not hold a wavefront for as many steps as it has neighbours.
constexpr uint32_t kPullSerial = 32;

__device__ __forceinline__ bool pull_scan(const int32_t* __restrict__ col, const uint32_t* __restrict__ front,
                                          int32_t begin, int32_t end, uint32_t& who) {
  bool hit = false;
  const uint32_t len = static_cast<uint32_t>(end - begin);
  const uint32_t serial = min(len, kPullSerial);
  for (uint32_t i = 0; i < serial && !hit; i += 4) {
    uint32_t u[4], w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) u[k] = static_cast<uint32_t>(col[list_edge(begin, i + k, len)]);
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = front[u[k] >> 5];
#pragma unroll
    for (int k = 3; k >= 0; --k)
      if ((w[k] >> (u[k] & 31)) & 1u) {
        hit = true;
        who = u[k];
      }
  }
  uint64_t rest = __ballot(!hit && serial < len);
  while (rest) {
    const int i = __ffsll(static_cast<unsigned long long>(rest)) - 1;
    rest &= rest - 1;
    const int32_t b = __builtin_amdgcn_readlane(begin, i);
    const uint32_t n = __builtin_amdgcn_readlane(len, i);
    for (uint32_t j = kPullSerial; j < n; j += kWave) {
      const uint32_t u = static_cast<uint32_t>(col[list_edge(b, j + lane_id(), n)]);
      const uint64_t in = __ballot((front[u >> 5] >> (u & 31)) & 1u);
      if (in) {
        const uint32_t first = __builtin_amdgcn_readlane(u, __ffsll(static_cast<unsigned long long>(in)) - 1);
        if (static_cast<int>(lane_id()) == i) {
          hit = true;
          who = first;
        }
        break;
      }
    }
  }
  return hit;
}

// The frontier of a pulled level as a bitmap, from the levels.
__device__ __forceinline__ void front_bitmap(const Bufs& B) {
  const uint32_t* __restrict__ level = B.S->level_out;
  const uint32_t last = B.S->level - 1;
  for (int64_t b = (blockIdx.x * static_cast<int64_t>(kWideBlock) + threadIdx.x) & ~int64_t(kWave - 1); b < B.n;
       b += static_cast<int64_t>(gridDim.x) * kWideBlock) {
    const int64_t v = b + lane_id();
    const uint64_t in = __ballot(v < B.n && level[v] == last);
    if (lane_id() == 0) B.front[b / kWave] = in;
  }
}

// Per lane: whether unreached vertex v (or none: live false) has a neighbour in
// the frontier, and which.  On the degree-ordered copy most vertices are found
// by their first neighbour, a hub, which is read in sequence from a list of its
// own: the row and, a cache line each, the neighbours are left to the others
// (RMAT-24: the three pulls 346 -> 240 us).
__device__ __forceinline__ bool pull_vertex(const int32_t* __restrict__ row, const int32_t* __restrict__ col,
                                            const uint32_t* __restrict__ first, const uint32_t* __restrict__ front,
                                            bool live, int64_t v, uint32_t& who) {
  bool hit = false;
  int32_t rb = 0, re = 0;
  if (live) {
    if (first) {
      who = first[v];  // v < nonzero: it has one
      hit = (front[who >> 5] >> (who & 31)) & 1u;
    }
    if (!hit) {
      rb = row[v];
      re = row[v + 1];
    }
  }
  uint32_t u;
  if (pull_scan(col, front, rb, re, u)) {
    who = u;
    hit = true;
  }
  return hit;
}

// A pulled level: every unreached vertex looks for a neighbour in the frontier.
__device__ __forceinline__ void pull_level(const Bufs& B, TdOp& op) {
  const uint32_t* front = reinterpret_cast<const uint32_t*>(B.front);
  for (int64_t b = (blockIdx.x * static_cast<int64_t>(kWideBlock) + threadIdx.x) & ~int64_t(kWave - 1); b < B.nonzero;
       b += static_cast<int64_t>(gridDim.x) * kWideBlock) {
    const int64_t v = b + lane_id();
    uint32_t who;
    const bool won[1] = {pull_vertex(B.row, B.col, B.first, front, v < B.nonzero && op.level[v] == kInf, v, who)};
    const uint32_t id[1] = {static_cast<uint32_t>(v)};
    if (won[0]) {
      op.level[v] = op.nl;
      if (op.vis) atomicOr(&op.vis[v >> 5], 1u << (v & 31));
      op.scout += static_cast<unsigned long long>(B.row[v + 1] - B.row[v]);
    }
    op.wq.push(won, id);
    op.after_step();
  }
}

__global__ void __launch_bounds__(kWideBlock) td_expand_kernel(Bufs B) {
  BfsState* S = B.S;
  if (!S->active) return;
  if (S->pull) {
    front_bitmap(B);
    return;
  }
  __shared__ uint32_t stage[kWideWaves][kWaveQCap];
  TdOp op = make_td(B, stage);
  expand_queue<kWideBlock, TdOp, false, kWideEdges>(B.row, B.q[S->q], S->count[S->q], B.hub, B.hubq, &S->hub_count, B.cap, &S->overflow, op, 0,
                                                    B.batch);
  op.finish();
}

// The second half of a level: the hubs' edges, or the pull.
__global__ void __launch_bounds__(kWideBlock) td_hubs_kernel(Bufs B) {
  BfsState* S = B.S;
  const bool pull = S->pull;
  if (!S->active || (S->hub_count == 0 && !pull)) return;
  __shared__ uint32_t stage[kWideWaves][kWaveQCap];
  TdOp op = make_td(B, stage);
  if (pull)
    pull_level(B, op);
  else
    expand_hubs<kWideBlock, TdOp, kHubLanes, kWideEdges>(B.row, B.hubq, S->hub_count, B.cap, B.hub_off, op);
  op.finish();
}

// Expansion of one level.  `hubs` false: no vertex exceeds the hub
// threshold, so the hub list stays empty and its two launches are left out.
void enqueue_expand(const Bufs& B, bool hubs, hipStream_t s) {
  td_expand_kernel<<<hubs ? kWideGrid : kGridNoHubs, kWideBlock, 0, s>>>(B);
  if (hubs) {
    launch_hub_offsets<kHubLanes * kWideEdges>(B.row, B.hubq, &B.S->hub_count, B.cap, B.hub_off, s);
    td_hubs_kernel<<<kWideGrid, kWideBlock, 0, s>>>(B);
  }
}

// Between two wide levels (inside a captured batch): ends the one before, and
// as long as the frontier is small takes the next levels itself, in one
// workgroup, then begins a wide level.  A wide level costs its launches and
// five dependent trips to memory, about 18 us (10 without hubs) however little
// there is to do; here the frontier's rows stay in LDS and a level of a few
// thousand edges is three trips (the neighbours, their levels, the exchange
// and the rows of what was found) and two barriers.  It takes frontiers of up
// to 8192 edges, 4096 without hubs, where the workgroup's own rate (a step of
// 4096 edges in 3-4 us) meets the cost of a wide level: RMAT-18 240 us (16384:
// 240, 4096: 316, all levels wide: 286), a lattice of 100,000 vertices 365
// (8192: 384, 16384: 432, all wide 400), 4096 RMAT vertices 111 (153).
constexpr unsigned kNarrowV = 4096;
constexpr unsigned kNarrowEdges = 1u << 13, kNarrowEdgesNoHubs = 1u << 12;

__global__ void __launch_bounds__(kWideBlock) narrow_kernel(Bufs B) {
  BfsState* S = B.S;
  if (S->done) return;
  __shared__ int32_t s_start[2][kNarrowV];
  __shared__ uint32_t s_deg[2][kNarrowV];
  __shared__ uint32_t s_vtx[2][kNarrowV];  // only with parents
  __shared__ uint32_t s_off[kNarrowV];
  __shared__ uint32_t s_scan[kWideWaves + 1];
  __shared__ unsigned s_count;
  __shared__ unsigned long long s_scout;
  const unsigned tid = threadIdx.x;
  if (tid == 0) level_end(S);
  __syncthreads();
  uint32_t* __restrict__ level = S->level_out;
  uint32_t* __restrict__ parent = S->parent_out;
  unsigned q = S->q, count = S->count[q], nl = S->level;
  const unsigned overflow = S->overflow;
  unsigned long long scout = S->scout, items = S->items, edges = S->edges;
  bool loaded = false;
  int cur = 0;
  while (count > 0 && count <= kNarrowV && scout <= B.narrow_max && !overflow) {  // workgroup-uniform
    if (!loaded) {
      const uint32_t* __restrict__ fq = B.q[q];
      for (unsigned i = tid; i < count; i += kWideBlock) {
        const uint32_t v = fq[i];
        s_start[cur][i] = B.row[v];
        s_deg[cur][i] = static_cast<uint32_t>(B.row[v + 1] - B.row[v]);
        if (parent) s_vtx[cur][i] = v;
      }
      loaded = true;
    }
    __syncthreads();
    if (tid == 0) {
      s_count = 0;
      s_scout = 0;
    }
    constexpr unsigned kPer = kNarrowV / kWideBlock;
    uint32_t deg[kPer], sum = 0, total;
#pragma unroll
    for (unsigned j = 0; j < kPer; ++j) {
      deg[j] = tid * kPer + j < count ? s_deg[cur][tid * kPer + j] : 0u;
      sum += deg[j];
    }
    uint32_t off = block_exclusive_scan<kWideBlock>(sum, s_scan, &total);
#pragma unroll
    for (unsigned j = 0; j < kPer; ++j) {
      s_off[tid * kPer + j] = off;
      off += deg[j];
    }
    __syncthreads();
    ++nl;
    uint32_t* __restrict__ qout = B.q[q ^ 1];
    unsigned long long found = 0;
    for (uint32_t e0 = 0; e0 < total; e0 += kWideBlock * kWideEdges) {
      bool won[kWideEdges];
      uint32_t v[kWideEdges], at_f[kWideEdges];
      int32_t rb[kWideEdges], re[kWideEdges];
#pragma unroll
      for (int k = 0; k < kWideEdges; ++k) {
        const uint32_t e = e0 + k * kWideBlock + tid;
        won[k] = e < total;
        v[k] = at_f[k] = 0;
        if (won[k]) {
          int lo = 0, hi = static_cast<int>(count) - 1;
          while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (s_off[mid] <= e) lo = mid; else hi = mid - 1;
          }
          at_f[k] = static_cast<uint32_t>(lo);
          v[k] = static_cast<uint32_t>(B.col[s_start[cur][lo] + static_cast<int32_t>(e - s_off[lo])]);
        }
      }
#pragma unroll
      for (int k = 0; k < kWideEdges; ++k) won[k] = won[k] && level[v[k]] == kInf;
#pragma unroll
      for (int k = 0; k < kWideEdges; ++k) {
        rb[k] = re[k] = 0;
        if (won[k]) {
          rb[k] = B.row[v[k]];
          re[k] = B.row[v[k] + 1];
        }
      }
      unsigned mine = 0;  // found by the wavefront in this step
#pragma unroll
      for (int k = 0; k < kWideEdges; ++k) {
        won[k] = won[k] && atomicCAS(&level[v[k]], kInf, nl) == kInf;
        if (won[k] && B.vis) atomicOr(&B.vis[v[k] >> 5], 1u << (v[k] & 31));
        mine += static_cast<unsigned>(__popcll(__ballot(won[k])));
      }
      if (mine == 0) continue;  // wavefront-uniform
      unsigned at = 0;
      if (lane_id() == 0) at = atomicAdd(&s_count, mine);
      at = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
      for (int k = 0; k < kWideEdges; ++k) {
        const uint64_t mask = __ballot(won[k]);
        if (won[k]) {
          const unsigned p = at + lanes_below(mask);
          const uint32_t d = static_cast<uint32_t>(re[k] - rb[k]);
          if (p < B.cap) qout[p] = v[k];
          if (p < kNarrowV) {
            s_start[cur ^ 1][p] = rb[k];
            s_deg[cur ^ 1][p] = d;
            if (parent) s_vtx[cur ^ 1][p] = v[k];
          }
          if (parent) parent[v[k]] = s_vtx[cur][at_f[k]];
          found += d;
        }
        at += static_cast<unsigned>(__popcll(mask));
      }
    }
    found = wave_sum(found);
    if (lane_id() == 0 && found) atomicAdd(&s_scout, found);
    __syncthreads();
    count = s_count;
    scout = s_scout;
    items += count;
    edges += scout;
    q ^= 1;
    cur ^= 1;
  }
  if (tid == 0) {
    S->q = q;
    S->count[q] = count;
    S->level = nl;
    S->scout = scout;
    S->items = items;
    S->edges = edges;
    level_begin(B);
  }
}

// `levels` wide levels, with the narrow ones between and after them, and
// before them at the start of a search (the last narrow kernel of a batch has
// begun the first wide level of the next).
void enqueue_levels(const Bufs& B, bool hubs, bool start, int levels, hipStream_t s) {
  if (start) narrow_kernel<<<1, kWideBlock, 0, s>>>(B);
  for (int i = 0; i < levels; ++i) {
    enqueue_expand(B, hubs, s);
    narrow_kernel<<<1, kWideBlock, 0, s>>>(B);
  }
  GX_LAUNCHED("bfs levels");
}

// ------------------------------------------------------------ bottom-up
__global__ void queue_to_bitmap_kernel(const uint32_t* __restrict__ q, const unsigned* __restrict__ count,
                                       uint32_t* __restrict__ bm) {
  const unsigned cnt = *count;
  for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < cnt; i += gridDim.x * blockDim.x) {
    const uint32_t v = q[i];
    atomicOr(&bm[v >> 5], 1u << (v & 31));
  }
}

// Every unreached vertex below `last` looks for a frontier in-neighbour; the
// words of `next` behind it are cleared.
__global__ void __launch_bounds__(kWideBlock) bu_step_kernel(const int32_t* __restrict__ trow,
                                                         const int32_t* __restrict__ tcol,
                                                         const uint32_t* __restrict__ first,
                                                         const int32_t* __restrict__ row,
                                                         uint32_t* __restrict__ level, uint32_t* __restrict__ parent,
                                                         const uint32_t* __restrict__ front,
                                                         uint32_t* __restrict__ next, BfsState* S, int64_t n,
                                                         int64_t last, uint32_t nl) {
  __shared__ unsigned long long red[kWideWaves];
  unsigned long long deg = 0;
  unsigned found = 0;
  for (int64_t b = (blockIdx.x * static_cast<int64_t>(kWideBlock) + threadIdx.x) & ~int64_t(kWave - 1); b < n;
       b += static_cast<int64_t>(gridDim.x) * kWideBlock) {
    const int64_t v = b + lane_id();
    uint32_t u;
    const bool hit = b < last && pull_vertex(trow, tcol, first, front, v < last && level[v] == kInf, v, u);
    // The wavefront owns the two words of its vertices.
    const uint64_t in = __ballot(hit);
    if (lane_id() < 2 && b + 32 * lane_id() < n) next[b / 32 + lane_id()] = static_cast<uint32_t>(in >> (32 * lane_id()));
    if (hit) {
      level[v] = nl;
      if (parent) parent[v] = u;
      deg += static_cast<unsigned long long>(row[v + 1] - row[v]);
      ++found;
    }
  }
  // Degree sum and count in one word, as the pushes add them.
  unsigned long long both;
  waves_exclusive_sum<kWideBlock>(wave_sum((deg << 32) | found), red, &both);
  if (threadIdx.x == 0 && both) atomicAdd(&S->app, both);
}

// A lane per bitmap word: one scan and one atomic per 32768 vertices.
__global__ void __launch_bounds__(kWideBlock) bitmap_to_queue_kernel(const uint32_t* __restrict__ bm, int64_t words,
                                                                 uint32_t* __restrict__ q, unsigned* count,
                                                                 unsigned cap, unsigned* overflow) {
  __shared__ uint32_t s_scan[kWideWaves + 1];
  __shared__ unsigned s_base;
  for (int64_t b = blockIdx.x * static_cast<int64_t>(kWideBlock); b < words;
       b += static_cast<int64_t>(gridDim.x) * kWideBlock) {
    const int64_t i = b + threadIdx.x;
    uint32_t bits = i < words ? bm[i] : 0u, total;
    const uint32_t before = block_exclusive_scan<kWideBlock>(static_cast<uint32_t>(__popc(bits)), s_scan, &total);
    if (total == 0) continue;  // workgroup-uniform
    if (threadIdx.x == 0) s_base = atomicAdd(count, total);
    __syncthreads();
    unsigned p = s_base + before;
    for (; bits; bits &= bits - 1, ++p) {
      const uint32_t v = static_cast<uint32_t>(i) * 32 + static_cast<uint32_t>(__ffs(static_cast<int>(bits)) - 1);
      if (p < cap) q[p] = v; else atomicOr(overflow, 1u);
    }
    __syncthreads();
  }
}

__global__ void do_pull_begin_kernel(BfsState* S) {
  if (threadIdx.x == 0) {
    S->app = 0;
  }
}

// The queue made from the last pulled frontier becomes the frontier of a push.
__global__ void do_pull_end_kernel(BfsState* S, uint32_t lvl) {
  if (threadIdx.x == 0) {
    S->level = lvl;
    S->scout = S->app >> 32;
    S->active = 0;
  }
}

__global__ void do_to_queue_begin_kernel(BfsState* S) {
  if (threadIdx.x == 0) {
    S->q = 0;
    S->count[0] = 0;
  }
}

unsigned sweep_grid(int64_t n) { return grid_for(n, kBlock, 256 * 16); }
unsigned wide_grid(int64_t n) { return grid_for(n, kWideBlock, kWideGrid); }

}  // namespace

extern "C" gx_status gx_bfs(gx_graph* g, uint32_t src, uint32_t* level, gx_stats* st) {
  GX_API_BEGIN
  check_graph(g);
  check_ptr(level, "level");
  check_vertex(g, src, "source");
  const int64_t n = g->n;
  hipStream_t s = g->stream;
  const unsigned cap = static_cast<unsigned>(n);
  // Visited bitmap from 2^25 vertices on: below that the 4-byte level array
  // (<= 128 MB) stays cache-resident and the bitmap's clear and atomics cost
  // more than they save.  Directed RMAT graphs of 2^24, 2^25 and 2^26 vertices
  // without it and with it: 3.03 3.20, 6.35 5.99, 12.97 11.08 ms.  Where levels
  // are pulled, which read the levels, it costs: symmetric RMAT-26 2.35 3.05 ms.
  const int64_t words = (n + 31) / 32;
  const bool use_vis = tune_effective("bfs.visited_bitmap", n, g->m) != 0;
  uint32_t* vis = use_vis ? g->scratch<uint32_t>(WS_BITMAP0, words) : nullptr;
  Bufs B{g->row, g->col, level, nullptr, {g->scratch<uint32_t>(WS_Q0, n), g->scratch<uint32_t>(WS_Q1, n)},
         g->scratch<uint32_t>(WS_Q2, n), g->scratch<BfsState>(WS_COUNTERS, 1), cap,
         g->scratch<uint32_t>(WS_HUBOFF, hub_off_words(n)), hub_degree(), vis, nullptr, n, g->m, nullptr, n, ~uint64_t(0), kNarrowEdgesNoHubs, kWideBlock};
  const bool hubs = max_degree(g) > static_cast<int64_t>(B.hub);
  if (hubs) {
    B.narrow_max = kNarrowEdges;
    B.batch = kBatchMax;
  }
  // Symmetric graphs with hubs pull their heavy levels (level_begin): the lists
  // then stand for the in-edges, which a push does not ask of them, so the first
  // search looks whether they do.
  if (hubs && (g->flags & GX_GRAPH_SYMMETRIC) && edges_paired(g)) {
    B.front = g->scratch<uint64_t>(WS_BITMAP1, (n + 63) / 64);
    B.pull_min = static_cast<uint64_t>(n) / 4;
  }
  // Graphs with hubs run on the degree-ordered copy of the CSR
  // (frontier.relabel): the levels of the most often reached vertices then
  // share a few cached megabytes; the source is mapped in, the levels back.
  const bool relabel = hubs && tune_effective("frontier.relabel", n, g->m) != 0;
  const uint32_t* src_map = nullptr;
  if (relabel) {
    build_relabeled(g);
    B.row = g->relab.row.as<int32_t>();
    B.col = g->relab.col.as<int32_t>();
    B.level = g->scratch<uint32_t>(WS_V5, cap);
    src_map = g->relab.new_of_old.as<uint32_t>();
    B.first = g->relab.first.as<uint32_t>();
    B.nonzero = g->relab.nonzero;
  }
  BfsState* host = static_cast<BfsState*>(g->host_pinned(sizeof(BfsState)));
  RegionTimer region(s);
  KernelTimer ktimer(s);
  bfs_init_kernel<<<sweep_grid(n), kBlock, 0, s>>>(B, n, src, src_map);
  GX_LAUNCHED("bfs_init_kernel");
  uint64_t key = 0;
  for (const void* p : {(const void*)B.row, (const void*)B.col, (const void*)B.q[0],
                        (const void*)B.q[1], (const void*)B.hubq, (const void*)B.S, (const void*)B.hub_off,
                        (const void*)B.vis, (const void*)B.front})
    key = mix_key(key, reinterpret_cast<uintptr_t>(p));
  key = mix_key(mix_key(mix_key(key, cap), B.hub), hubs ? 1u : 0u);
  uint32_t replays = 0, slots = 0;
  for (;;) {
    const int first = hubs && g->m < kSmallEdges ? kLevelsFirstSmall : kLevelsFirst;
    const int nl = replays == 0 ? first : kLevelsPerGraph;
    ktimer.begin();
    g->replay(replays == 0 ? g->bfs_head : g->bfs_batch, key, [&](hipStream_t cs) {
      enqueue_levels(B, hubs, replays == 0, nl, cs);
    });
    ktimer.end();
    ++replays;
    slots += static_cast<uint32_t>(nl);
    GX_HIP(hipMemcpyAsync(host, B.S, sizeof(BfsState), hipMemcpyDeviceToHost, s));
    GX_HIP(hipStreamSynchronize(s));
    if (host->overflow) fail(GX_ERR_CAPACITY, "BFS frontier queue overflow");
    if (host->done) break;
  }
  if (relabel) unpermute_u32(B.level, g->relab.new_of_old.as<uint32_t>(), level, n, s);
  double ms = region.stop();
  if (st) {
    std::memset(st, 0, sizeof(*st));
    st->iterations = host->level - 1;  // levels with a non-empty frontier beyond the source
    st->launches = 2 + slots * (hubs ? 4 : 2) + (relabel ? 1 : 0);
    st->edges_visited = host->edges;
    st->items = host->items;
    st->elapsed_ms = ms;
    st->main_kernel_ms = ktimer.total_ms();
    st->main_kernel_launches = ktimer.count();
  }
  GX_API_END
}

// Parents back to the caller's vertex ids: out[v] = old_of_new[p] for the
// parent p of v's degree-ordered id (the source's own id, or none).
__global__ void unpermute_parent_kernel(const uint32_t* __restrict__ pin, const uint32_t* __restrict__ new_of_old,
                                        const uint32_t* __restrict__ old_of_new, uint32_t* __restrict__ out,
                                        int64_t n) {
  for (int64_t v = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; v < n;
       v += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const uint32_t p = pin[new_of_old[v]];
    out[v] = p == kNoParent ? p : old_of_new[p];
  }
}

extern "C" gx_status gx_bfs_do(gx_graph* g, uint32_t src, uint32_t alpha, uint32_t beta, uint32_t* level,
                               uint32_t* parent, gx_stats* st) {
  GX_API_BEGIN
  check_graph(g);
  check_ptr(level, "level");
  check_vertex(g, src, "source");
  const int64_t n = g->n;
  hipStream_t s = g->stream;
  if (alpha == 0) alpha = 15;
  if (beta == 0) beta = 18;
  const int32_t* trow = g->row;
  const int32_t* tcol = g->col;
  if (!(g->flags & GX_GRAPH_SYMMETRIC)) {
    build_transpose(g);
    trow = g->trow();
    tcol = g->tcol();
  }
  const unsigned cap = static_cast<unsigned>(n);
  Bufs B{g->row, g->col, level, parent, {g->scratch<uint32_t>(WS_Q0, n), g->scratch<uint32_t>(WS_Q1, n)},
         g->scratch<uint32_t>(WS_Q2, n), g->scratch<BfsState>(WS_COUNTERS, 1), cap,
         g->scratch<uint32_t>(WS_HUBOFF, hub_off_words(n)), hub_degree(), nullptr, nullptr, n, g->m, nullptr, n, ~uint64_t(0), kNarrowEdgesNoHubs, kWideBlock};
  const int64_t words = (n + 31) / 32;
  uint32_t* bm[2] = {g->scratch<uint32_t>(WS_BITMAP0, words), g->scratch<uint32_t>(WS_BITMAP1, words)};
  const bool hubs = max_degree(g) > static_cast<int64_t>(B.hub);
  if (hubs) {
    B.narrow_max = kNarrowEdges;
    B.batch = kBatchMax;
  }
  // Symmetric graphs with hubs run on the degree-ordered copy of the CSR
  // (frontier.relabel): a bottom-up step scans each unvisited vertex's
  // neighbours hubs first, and the hubs are the first vertices reached, so
  // most scans stop at their first neighbour; levels and parents are mapped
  // back at the end.
  const bool relabel = (g->flags & GX_GRAPH_SYMMETRIC) && hubs && tune_effective("frontier.relabel", n, g->m) != 0;
  const uint32_t* src_map = nullptr;
  if (relabel) {
    build_relabeled(g);
    trow = B.row = g->relab.row.as<int32_t>();
    tcol = B.col = g->relab.col.as<int32_t>();
    B.level = g->scratch<uint32_t>(WS_V5, cap);
    B.parent = parent ? g->scratch<uint32_t>(WS_V4, cap) : nullptr;
    src_map = g->relab.new_of_old.as<uint32_t>();
    B.first = g->relab.first.as<uint32_t>();
    B.nonzero = g->relab.nonzero;
  }
  BfsState* host = static_cast<BfsState*>(g->host_pinned(sizeof(BfsState)));
  auto read_state = [&]() {
    GX_HIP(hipMemcpyAsync(host, B.S, sizeof(BfsState), hipMemcpyDeviceToHost, s));
    GX_HIP(hipStreamSynchronize(s));
    if (host->overflow) fail(GX_ERR_CAPACITY, "BFS frontier queue overflow");
  };
  RegionTimer region(s);
  KernelTimer ktimer(s);
  uint32_t launches = 2;
  bfs_init_kernel<<<sweep_grid(n), kBlock, 0, s>>>(B, n, src, src_map);
  narrow_kernel<<<1, kWideBlock, 0, s>>>(B);
  GX_LAUNCHED("bfs init");
  uint64_t pull_edges = 0, pull_items = 0;
  bool pulled = false;  // the frontier is what a pull phase left: push it
  read_state();
  while (!host->done) {
    // Edges out of the frontier against those that pushes have not walked.
    const int64_t scout = static_cast<int64_t>(host->scout);
    const int64_t edges_to_check = g->m - (static_cast<int64_t>(host->edges) - scout);
    if (!pulled && scout > edges_to_check / static_cast<int64_t>(alpha)) {
      // Pull phase: queue -> bitmap; pull while the frontier grows or stays
      // above n/beta.
      const unsigned q = host->q;
      uint32_t lvl = host->level - 1;  // the state has begun the level
      fill_kernel<uint32_t><<<sweep_grid(words), kBlock, 0, s>>>(bm[0], 0u, words);
      queue_to_bitmap_kernel<<<grid_for(host->count[q], kBlock, 4096), kBlock, 0, s>>>(B.q[q], &B.S->count[q], bm[0]);
      launches += 2;
      int b = 0;
      uint64_t work = static_cast<uint64_t>(scout), old_work;
      do {
        old_work = work;
        ++lvl;
        do_pull_begin_kernel<<<1, 64, 0, s>>>(B.S);
        ktimer.begin();
        bu_step_kernel<<<wide_grid(n), kWideBlock, 0, s>>>(trow, tcol, B.first, B.row, B.level, B.parent, bm[b],
                                                           bm[b ^ 1], B.S, n, B.nonzero, lvl);
        ktimer.end();
        GX_LAUNCHED("bu_step_kernel");
        launches += 2;
        read_state();
        work = static_cast<uint32_t>(host->app);
        pull_items += work;
        pull_edges += host->app >> 32;
        b ^= 1;
      } while (work > 0 && (work >= old_work || work > static_cast<uint64_t>(n) / beta));
      // Bitmap -> queue for the next push level.
      do_to_queue_begin_kernel<<<1, 64, 0, s>>>(B.S);
      bitmap_to_queue_kernel<<<wide_grid(words), kWideBlock, 0, s>>>(bm[b], words, B.q[0], &B.S->count[0], cap,
                                                              &B.S->overflow);
      do_pull_end_kernel<<<1, 64, 0, s>>>(B.S, lvl);
      GX_LAUNCHED("bitmap_to_queue_kernel");
      launches += 3;
      pulled = true;
    } else {
      ktimer.begin();
      enqueue_expand(B, hubs, s);
      ktimer.end();
      launches += hubs ? 3 : 1;
      pulled = false;
    }
    narrow_kernel<<<1, kWideBlock, 0, s>>>(B);
    GX_LAUNCHED("narrow_kernel");
    ++launches;
    read_state();
  }
  if (relabel) {
    unpermute_u32(B.level, g->relab.new_of_old.as<uint32_t>(), level, n, s);
    if (parent) {
      unpermute_parent_kernel<<<grid_for(n, kBlock, 8192), kBlock, 0, s>>>(
          B.parent, g->relab.new_of_old.as<uint32_t>(), g->relab.old_of_new.as<uint32_t>(), parent, n);
      GX_LAUNCHED("unpermute_parent_kernel");
    }
    launches += parent ? 2 : 1;
  }
  double ms = region.stop();
  if (st) {
    std::memset(st, 0, sizeof(*st));
    st->iterations = host->level;
    st->launches = launches;
    st->edges_visited = host->edges + pull_edges;
    st->items = host->items + pull_items;
    st->elapsed_ms = ms;
    st->main_kernel_ms = ktimer.total_ms();
    st->main_kernel_launches = ktimer.count();
  }
  GX_API_END
}
