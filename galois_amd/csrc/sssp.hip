// Single-source shortest paths by bucketed delta-stepping.
//
// Reference semantics: lonestar/analytics/cpu/sssp/SSSP.cpp:119-173
// (deltaStepAlgo): bucket index dist >> shift (BFS_SSSP.h:50-58, `-delta` is
// the shift), relaxation newDist = dist[src] + w with atomicMin
// (AtomicHelpers.h:60-67), push when it lowers the distance.  The GPU app
// (lonestar/analytics/gpu/sssp/sssp.cu:170-297) splits the work into a near
// list (dist within the current bucket) and a far pile.  Shortest distances
// are the unique fixpoint, so the output is bit-exact against the CPU path.
//
// Design (gfx950)
//  - near frontier: vertices whose new distance falls in the current bucket;
//    each round relaxes all of them with the load-balanced expansion of
//    frontier.hpp and atomicMin on the distance word; a vertex enters a
//    round's queue once (stamp word per vertex).  A vertex is expanded only
//    if its distance changed since it was last expanded (`done` word), the
//    GPU form of the reference's stale-item test (SSSP.cpp:138).
//  - far pile: vertices whose distance lies in a later bucket.  A vertex joins
//    it when it is first reached there and stays until a split takes it out
//    or finds it settled, so each is in the pile at most once and no mark is
//    needed (an atomic per improvement less; random atomics run at 27 G/s
//    on this GPU, a fifth of the gathers).  A
//    running minimum of the far buckets (every improvement into a later
//    bucket, and every item a split keeps) names the next bucket; when the
//    near frontier drains, one pass moves that bucket into the near frontier
//    and keeps the rest.  The running minimum can name a bucket whose items
//    have meanwhile moved nearer; that split then moves nothing and the next
//    one uses the exact minimum of the items it kept.
//  - A relax step of few items (relax_local) goes on with what its workgroups
//    improved into the near range for a few rounds before it ends: 153 steps
//    of 17 us become about 50 on a lattice of 2048 x 2048 (3.67 -> 2.17 ms).
//  - Merged buckets: a step covers the buckets [bucket, bucket + width).
//    width starts at 1 and doubles at an advance when the phase just ended
//    admitted fewer than kMergeLow items (up to the knob sssp.max_merge),
//    and halves when it admitted more than kMergeHigh: on road-like graphs
//    a delta-64 bucket holds a thin shell of a few thousand vertices, so
//    merging cuts the number of dependent steps, at the cost of a few
//    vertices expanded before their distance is final (they are expanded
//    again when it improves, as in any label-correcting order).  Power-law
//    graphs keep width 1 (their buckets hold millions of items).
//  - Hubs (degree above frontier.hub_degree) admitted in a relax step are
//    expanded over the whole grid in the same step.  With the knob
//    sssp.defer_hubs they instead join a pending list (once per list, mark
//    word per vertex) that is expanded in a step of its own when the near
//    frontier has drained, so a hub whose distance improves several times
//    inside a bucket is expanded once per drain rather than once per
//    improvement.  With sssp.hub_refine a step expands only the pending
//    hubs within a distance slice above the smallest pending hub distance
//    (2^(r - 1); while the knob is not set one distance at first, then as many
//    as the hubs per step call for) and keeps the rest pending, so hubs go out
//    nearly in distance order, almost all at their final distance, and a
//    hub's hundreds of thousands of edges are relaxed about once instead
//    of once per improvement (RMAT-26: 1.84 -> 1.10 relaxations per edge).
//    The hub selection joins a relax step whenever the smallest pending hub
//    distance is at or below the smallest distance in that step's near
//    queue (hubs above it wait; positive weights mean nothing left to
//    expand can lower the hubs taken), and otherwise runs in a step of its
//    own once the near frontier drains.  The extra steps pay on large
//    power-law graphs only, so the default enables it from 2^24 vertices
//    on.
//  - Shared words: a workgroup takes room in both queues with one atomic on
//    one packed word, lowers a minimum only when a read shows it would, and
//    counts edges and items in a pair of its own (RMAT-22 5.16 -> 4.20 ms
//    with these, the wavefronts' own queues and the hub order by edges).
//  - Wide steps are bound by the gathers in flight: the kernels keep to 64
//    registers, so that two workgroups share a CU, and the hub pass cuts hubs
//    into steps of a wavefront (256 edges; most hubs of an RMAT graph have
//    fewer than 1000), RMAT-22 4.07 -> 3.81 ms, one with 2 M vertices and all
//    weights in one bucket 1.60 -> 1.34.
//  - Locality: on graphs with hubs (knob frontier.relabel) the kernels run
//    on the degree-ordered copy of the CSR (gx_graph::relab): the hubs and
//    the vertices most often relaxed get the smallest ids, so their
//    distance words share a few megabytes that stay cached, instead of each
//    relaxation moving a line of a 268 MB array (RMAT-26).  The source is
//    mapped in and the distances mapped back at the end.
//  - The loop is driven on the device: every step is the same fixed kernel
//    sequence (step; work, which is either the relax, with the stale-item
//    filter fused in as the expansion's admission test, or the far split, as
//    the step's mode says; hub layout; hubs) whose kernels read the step's
//    mode from a device state word and return at once when it is not
//    theirs; the step kernel also closes the previous step.  On graphs
//    without hubs the two hub launches are left out.  Steps are captured
//    once into a HIP graph (kStepsPerGraph steps and a closing kernel) and
//    replayed until the state says done, so the host synchronises once per
//    graph replay instead of once per round.
#include <algorithm>

#include "frontier.hpp"
#include "gx_device.hpp"
#include "gx_internal.hpp"

using namespace gx;

namespace {

constexpr int kBlock = 256;
constexpr uint32_t kInf = GX_DIST_INFINITY;
// Graphs without hubs (maximum degree at or below the hub threshold, such as
// road-like grids) have small frontiers per step and many steps: half of the
// workgroups start faster and meet less at the step's counters (128: 2.88 ms on
// a lattice of 2048 x 2048, 256: 2.57, 512: 2.72).
constexpr int kGridNoHubs = 256;
constexpr int kHubLanes = 64;  // lanes per step of the hub pass
constexpr int kStepsPerGraph = 16;
constexpr int kHubSelectGrid = 128;
// Bucket merging thresholds (items per phase).  2^14 and 2^17: lattice of 2048 x
// 2048 with weights to 1000 the same, to 60000 5.4 ms against 4.2; 2^16 and
// 2^19: 2.64 ms against 2.17 and 3.8 against 4.2.
constexpr unsigned long long kMergeLow = 1ull << 15;
constexpr unsigned long long kMergeHigh = 1ull << 18;

// While sssp.hub_refine is not set, a hub step's slice of distances doubles when
// the step expanded few hubs and halves when it expanded many: a step costs 20 us
// however few hubs it has.  With weights to 60000 fixed slices of one distance took
// 90 ms on RMAT-22, these 8 (2^8 and 2^12 to 2^14 and 2^18 within 1% of each
// other).  A set knob's slices stay as they are.
constexpr unsigned kHubsFew = 1u << 10, kHubsMany = 1u << 14;

enum Mode : unsigned { kIdle = 0, kRelax = 1, kAdvance = 2, kHubs = 3 };

struct SsspState {
  unsigned near_count[2];  // near queues (double buffered by q)
  unsigned far_count[2];   // far piles (double buffered by far_sel)
  // Ends of the queues a step fills: near (low 32 bits) and far (high 32 bits),
  // so that a workgroup gets room in both with one atomic.
  unsigned long long app;
  unsigned hub_count;
  unsigned overflow;
  unsigned far_min;        // running minimum of the far buckets
  unsigned mode;
  unsigned done;
  unsigned q;              // near queue read this step
  unsigned far_sel;        // far pile appended to
  unsigned bucket;
  unsigned width;          // buckets merged into the current phase
  unsigned max_width;      // knob sssp.max_merge
  unsigned hub_gen;        // generation of the pending hub list
  unsigned hub_expand;     // hubs expanded this step (selected in a hub step, else 0)
  unsigned hq;             // pending hub list appended to (double buffered)
  unsigned hub_kept;       // pending hubs a hub step leaves for a later one
  uint32_t hub_min;        // smallest distance a pending hub had when it was listed
  uint32_t hub_min_next;   // the same over the hubs a hub step keeps
  uint32_t hub_limit;      // a hub step expands the pending hubs at or below this distance
  uint32_t hub_span;       // a hub step's slice of distances
  unsigned hub_adapt;      // hub_span follows the hubs of a step
  unsigned hub_step;       // this step selects and expands pending hubs
  uint32_t near_min;       // smallest distance in the near queue the step reads
  uint32_t near_min_next;  // the same for the near queue the step fills
  unsigned long long phase_start;  // items before the current phase
  unsigned long long queued;       // items of the near queues read so far
  unsigned round;
  unsigned phase;
  unsigned steps;
  unsigned long long edges;  // sums of the workgroups' counts at the end of a batch
  unsigned long long items;
  // Output of the current call, read by the captured step kernels.
  uint32_t* dist_out;
};

struct Bufs {
  const int32_t* row;
  const int32_t* col;
  const uint32_t* w;
  uint32_t* dist;
  uint32_t* stamp;
  uint32_t* done;
  uint32_t* hubmark;  // generation of the pending hub list a hub is in
  uint32_t* nearq[2];
  uint32_t* farq[2];
  uint32_t* hubq[2];  // pending hub lists (hq); without deferral hubq[0] holds the step's hubs
  uint32_t* hubx;     // hubs a hub step expands
  SsspState* S;
  // Edges relaxed and items expanded, per workgroup index: every kernel of the
  // run adds to its own workgroup's pair, and only the batch's end sums them.
  unsigned long long* tally;
  uint32_t shift;
  unsigned cap;
  uint32_t* hub_off;
  uint32_t hub;  // frontier.hub_degree
  uint32_t defer;  // sssp.defer_hubs: pending hub list expanded in hub steps
  // sssp.hub_refine r: a hub step expands the pending hubs within
  // hub_span = 2^(r - 1) of the smallest pending hub distance; 0 = all.
  uint32_t hub_span;
  int local_rounds;    // kLocalRounds or kLocalRoundsNoHubs
  unsigned local_max;  // most near items of a step with local rounds
  unsigned batch;      // most vertices a workgroup takes at a time
};

__global__ void sssp_init_kernel(uint32_t* __restrict__ dist, uint32_t* __restrict__ stamp,
                                 uint32_t* __restrict__ done,
                                 uint32_t* __restrict__ hubmark, int64_t n, uint32_t src) {
  int64_t v = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (; v < n; v += stride) {
    dist[v] = (v == src) ? 0u : kInf;
    stamp[v] = 0xffffffffu;
    done[v] = kInf;
    hubmark[v] = 0xffffffffu;
  }
}

__global__ void sssp_reset_kernel(SsspState* S, unsigned long long* tally, uint32_t* nearq0, uint32_t src,
                                  uint32_t* dist, unsigned max_width,
                                  uint32_t hub_span, unsigned hub_adapt) {
  for (int i = threadIdx.x; i < 2 * kWideGrid; i += blockDim.x) tally[i] = 0;
  if (threadIdx.x == 0) {
    S->dist_out = dist;
    S->near_count[0] = 1;
    S->near_count[1] = 0;
    S->far_count[0] = S->far_count[1] = 0;
    S->app = 0;
    S->hub_count = 0;
    S->overflow = 0;
    S->far_min = 0xffffffffu;
    S->mode = kIdle;
    S->done = 0;
    S->q = 0;
    S->far_sel = 0;
    S->bucket = 0;
    S->width = 1;
    S->max_width = max_width;
    S->hub_gen = 0;
    S->hub_expand = 0;
    S->hq = 0;
    S->hub_kept = 0;
    S->hub_min = S->hub_min_next = S->hub_limit = 0xffffffffu;
    S->hub_span = hub_span;
    S->hub_adapt = hub_adapt;
    S->hub_step = 0;
    S->near_min = 0;  // the source
    S->near_min_next = 0xffffffffu;
    S->phase_start = 0;
    S->queued = 0;
    S->round = 0;
    S->phase = 0;
    S->steps = 0;
    S->edges = 0;
    S->items = 0;
    nearq0[0] = src;
  }
}

// Closes a step: the queue it filled becomes the input; after a split the
// far piles swap; after a step that expanded hubs the pending list holds
// the hubs it kept, under a new generation.
__device__ __forceinline__ void close_step(SsspState* S) {
  if (S->hub_step) {
    S->hq ^= 1;
    if (S->hub_adapt) {
      if (S->hub_expand < kHubsFew && S->hub_span < (1u << 30)) S->hub_span *= 2;
      else if (S->hub_expand > kHubsMany && S->hub_span > 1) S->hub_span /= 2;
    }
    S->hub_count = S->hub_kept;  // kept hubs carry the new generation's mark
    S->hub_kept = 0;
    S->hub_expand = 0;
    S->hub_gen += 1;
    S->hub_min = S->hub_min_next;
    S->hub_step = 0;
  }
  if (S->mode == kAdvance) {
    S->far_count[S->far_sel] = 0;
    S->far_sel ^= 1;
  }
  if (S->mode != kIdle) {
    S->q ^= 1;
    S->near_count[S->q] = static_cast<unsigned>(S->app);
    S->far_count[S->far_sel] = static_cast<unsigned>(S->app >> 32);
    S->near_min = S->near_min_next;
    S->near_min_next = 0xffffffffu;
  }
  S->mode = kIdle;
}

// Starts the hub part of a step: pending hubs at or below `limit` are
// selected (hub_select_kernel) and expanded (hubs_kernel).
__device__ __forceinline__ void begin_hub_step(SsspState* S, uint32_t limit) {
  S->hub_step = 1;
  S->hub_expand = 0;  // counted by hub_select_kernel
  S->hub_kept = 0;
  S->hub_min_next = 0xffffffffu;
  S->hub_limit = limit;
}

// Closes the previous step, then chooses this step's mode and clears the
// counters it appends to: relax while the near frontier has items, then
// expand the pending hubs, then advance.  An advance takes the running far
// minimum as the new first bucket and sets the phase's width from the items
// of the last phase; with far items left but no live far bucket (minimum
// unset) every far item is settled and the run is done.  A phase's items are
// those expanded (the workgroups' counts: local rounds expand many that no
// queue has seen), with hubs those queued (tally null), which saves a step the
// read of the counts.
__global__ void __launch_bounds__(kWave) step_kernel(SsspState* S, const unsigned long long* __restrict__ tally,
                                                     uint32_t defer, uint32_t hub_span) {
  if (S->done) return;
  unsigned long long items = 0;
  if (tally) {  // kernel argument: the same for every lane
    for (int i = threadIdx.x; i < kWideGrid; i += kWave) items += tally[2 * i + 1];
    items = wave_sum(items);
  }
  if (threadIdx.x != 0) return;
  close_step(S);
  if (S->overflow) return;
  if (!tally) items = S->queued += S->near_count[S->q];
  S->round += 1;
  S->app = static_cast<unsigned long long>(S->far_count[S->far_sel]) << 32;
  if (!defer) S->hub_count = 0;  // hubs of a relax step are expanded in that step
  if (hub_span) hub_span = S->hub_span;
  const uint32_t span_limit =
      (hub_span == 0 || S->hub_min >= 0xffffffffu - hub_span) ? 0xffffffffu : S->hub_min + (hub_span - 1u);
  if (S->near_count[S->q] > 0) {
    S->mode = kRelax;
    // With hub slices, the pending hubs at or below every near distance are
    // expanded in the same step as the near frontier: nothing left to
    // expand can still lower them (weights are positive).
    if (defer && hub_span != 0 && S->hub_count > 0 && S->hub_min <= S->near_min)
      begin_hub_step(S, min(span_limit, S->near_min));
  } else if (defer && S->hub_count > 0) {
    S->mode = kHubs;
    begin_hub_step(S, span_limit);
  } else if (S->far_count[S->far_sel] > 0 && S->far_min != 0xffffffffu) {
    S->mode = kAdvance;
    const unsigned long long in_phase = items - S->phase_start;
    if (in_phase < kMergeLow && S->width < S->max_width)
      S->width = min(2 * S->width, S->max_width);
    else if (in_phase > kMergeHigh && S->width > 1)
      S->width >>= 1;
    S->phase_start = items;
    S->phase += 1;
    S->bucket = S->far_min;
    S->far_min = 0xffffffffu;
    S->app = 0;  // the kept far items fill the other pile
  } else {
    S->done = 1;
    return;
  }
  S->steps += 1;
}

// Last kernel of a captured batch (one workgroup of kBlock lanes): closes its
// last step and sums the workgroups' counts, so the state is whole when the
// host reads it.
__global__ void __launch_bounds__(kBlock) batch_end_kernel(SsspState* S, const unsigned long long* tally) {
  __shared__ unsigned long long s_sum[2][kBlock / kWave];
  unsigned long long e = 0, t = 0;
  for (int i = threadIdx.x; i < kWideGrid; i += kBlock) {
    e += tally[2 * i];
    t += tally[2 * i + 1];
  }
  e = wave_sum(e);
  t = wave_sum(t);
  if (lane_id() == 0) {
    s_sum[0][threadIdx.x / kWave] = e;
    s_sum[1][threadIdx.x / kWave] = t;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  S->edges = S->items = 0;
  for (int i = 0; i < kBlock / kWave; ++i) {
    S->edges += s_sum[0][i];
    S->items += s_sum[1][i];
  }
  close_step(S);
}

// Lowers *word to v.  Most workgroups bring nothing below what is there: a
// read at agent scope spares them the atomic.
__device__ __forceinline__ void lower(uint32_t* word, uint32_t v) {
  if (v < __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(word, v);
}

using Stage = uint32_t[kWideWaves][kWaveQCap];

// The two queues a step fills, staged per wavefront: nearer items go to nq,
// later ones to fq, room in both taken with one atomic.
struct PairQueue {
  WaveQueue<kWaveQCap> near, far;
  uint32_t* nq;
  uint32_t* fq;
  SsspState* S;
  unsigned cap;
  __device__ __forceinline__ PairQueue(SsspState* s, Stage& sn, Stage& sf, uint32_t* n, uint32_t* f, unsigned c)
      : near{sn[threadIdx.x / kWave]}, far{sf[threadIdx.x / kWave]}, nq(n), fq(f), S(s), cap(c) {}
  __device__ __forceinline__ unsigned long long counts() const {
    return near.count | (static_cast<unsigned long long>(far.count) << 32);
  }
  __device__ __forceinline__ void store(unsigned long long base) {
    near.store(static_cast<unsigned>(base), nq, cap, &S->overflow);
    far.store(static_cast<unsigned>(base >> 32), fq, cap, &S->overflow);
  }
  // After every step of at most `step` items a wavefront and queue.
  __device__ __forceinline__ void after_step(unsigned step) {
    if (!near.full(step) && !far.full(step)) return;
    unsigned long long base = 0;
    if (lane_id() == 0) base = atomicAdd(&S->app, counts());
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(base));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(base >> 32));
    store((static_cast<unsigned long long>(hi) << 32) | lo);
  }
  // Workgroup-uniform: what is left, for all wavefronts at once.
  __device__ __forceinline__ void finish() {
    __shared__ unsigned long long s_sum[kWideWaves + 1];
    unsigned long long total;
    const unsigned long long before = waves_exclusive_sum<kWideBlock>(counts(), s_sum, &total);
    if (threadIdx.x == 0) s_sum[kWideWaves] = total ? atomicAdd(&S->app, total) : 0ull;
    __syncthreads();
    store(s_sum[kWideWaves] + before);
  }
};

// Holds the output pointer read from the device state: the kernel-argument
// Bufs stays unmodified (a modified copy of it, with its runtime-indexed
// queue arrays, would be kept in scratch memory).
struct RelaxOp {
  Bufs B;
  uint32_t* dist;
  PairQueue q;
  uint32_t bucket_end, round, hub_gen;  // bucket_end: last bucket of the phase
  uint32_t far_min = 0xffffffffu;  // this lane's smallest far bucket improved into
  uint32_t hub_min = 0xffffffffu;  // this lane's smallest distance of a hub it listed
  uint32_t near_min = 0xffffffffu;  // this lane's smallest distance improved into the near range
  unsigned long long edges = 0, items = 0;
  // Stale-item filter (the reference's test at SSSP.cpp:138): a near item is
  // expanded only if its distance changed since it was last admitted.  A
  // hub passes into the pending list once per list generation (its edges
  // are counted when the list is expanded).
  __device__ __forceinline__ bool admit(uint32_t u) {
    const uint32_t d = dist[u];
    if (B.done[u] == d) return false;
    B.done[u] = d;
    const uint32_t deg = static_cast<uint32_t>(B.row[u + 1] - B.row[u]);
    if (deg > B.hub) {
      if (!B.defer) return true;
      if (atomicExch(&B.hubmark[u], hub_gen) == hub_gen) return false;
      hub_min = min(hub_min, d);
      return true;
    }
    edges += deg;
    items += 1;
    return true;
  }
  template <int U>
  __device__ __forceinline__ void run(const bool (&valid)[U], const uint32_t (&u)[U], const int32_t (&e)[U]) {
    bool to_near[U], to_far[U];
    uint32_t v[U], nd[U], dv[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
      v[k] = static_cast<uint32_t>(B.col[e[k]]);
      nd[k] = dist[u[k]] + B.w[e[k]];
    }
#pragma unroll
    for (int k = 0; k < U; ++k) dv[k] = dist[v[k]];
#pragma unroll
    for (int k = 0; k < U; ++k) {
      to_near[k] = to_far[k] = false;
      if (!valid[k] || nd[k] >= dv[k]) continue;
      const uint32_t old = atomicMin(&dist[v[k]], nd[k]);
      if (nd[k] >= old) continue;
      const uint32_t nb = nd[k] >> B.shift;
      if (nb > bucket_end) {
        far_min = min(far_min, nb);
        to_far[k] = old == kInf;  // reached before: it is in the far pile
      } else {
        near_min = min(near_min, nd[k]);
        to_near[k] = atomicExch(&B.stamp[v[k]], round) != round;
      }
    }
    q.near.push(to_near, v);
    q.far.push(to_far, v);
  }
  __device__ __forceinline__ void after_step() { q.after_step(kWideStep); }
  // End of a launch, workgroup-uniform: queues flushed, minima and counts
  // reduced over the workgroup; the counts go to the workgroup's own pair.
  __device__ __forceinline__ void finish() {
    q.finish();
    constexpr int kW = kWideBlock / kWave;
    __shared__ uint32_t s_min[3][kW];
    __shared__ unsigned long long s_sum[2][kW];
    const uint32_t fm = wave_min(far_min), hm = wave_min(hub_min), nm = wave_min(near_min);
    const unsigned long long ed = wave_sum(edges), it = wave_sum(items);
    const unsigned w = threadIdx.x / kWave;
    if (lane_id() == 0) {
      s_min[0][w] = fm;
      s_min[1][w] = hm;
      s_min[2][w] = nm;
      s_sum[0][w] = ed;
      s_sum[1][w] = it;
    }
    __syncthreads();
    if (w != 0) return;
    const unsigned i = lane_id() < kW ? lane_id() : 0u;  // a lane per wavefront
    const uint32_t f = wave_min(s_min[0][i]), h = wave_min(s_min[1][i]), nn = wave_min(s_min[2][i]);
    const unsigned long long e = wave_sum(lane_id() < kW ? s_sum[0][i] : 0ull),
                             t = wave_sum(lane_id() < kW ? s_sum[1][i] : 0ull);
    if (threadIdx.x == 0) {
      if (f != 0xffffffffu) lower(&B.S->far_min, f);
      if (h != 0xffffffffu) lower(&B.S->hub_min, h);
      if (nn != 0xffffffffu && B.hub_span) lower(&B.S->near_min_next, nn);  // read only with hub slices
      if (e | t) {
        B.tally[2 * blockIdx.x] += e;  // hub steps count edges in every workgroup, items in one
        B.tally[2 * blockIdx.x + 1] += t;
      }
    }
  }
};

__device__ __forceinline__ RelaxOp make_relax(const Bufs& B, Stage& sn, Stage& sf) {
  SsspState* S = B.S;
  const unsigned q = S->q, fs = S->far_sel;
  return RelaxOp{B, S->dist_out, PairQueue(S, sn, sf, B.nearq[q ^ 1], B.farq[fs], B.cap), S->bucket + (S->width - 1),
                 S->round, S->hub_gen};
}

// Relax operation over hub edges: counts every valid edge it relaxes.
template <class Op>
struct HubCount {
  Op& op;
  template <int U>
  __device__ __forceinline__ void run(const bool (&valid)[U], const uint32_t (&u)[U], const int32_t (&e)[U]) {
#pragma unroll
    for (int k = 0; k < U; ++k) op.edges += valid[k] ? 1ull : 0ull;
    op.run(valid, u, e);
  }
  __device__ __forceinline__ void after_step() { op.after_step(); }
};

// Relax step: expand the near items that pass the stale-item filter.
__device__ __forceinline__ void relax_step(const Bufs& B, Stage& sn, Stage& sf) {
  SsspState* S = B.S;
  RelaxOp op = make_relax(B, sn, sf);
  const unsigned q = S->q;
  expand_queue<kWideBlock, RelaxOp, true, kWideEdges>(B.row, B.nearq[q], S->near_count[q], B.hub, B.hubq[S->hq], &S->hub_count, B.cap,
                                      &S->overflow, op, 0, B.batch);
  op.finish();
}

// Relax step of a small near frontier: a workgroup takes one batch of it and
// goes on with what it improved into the near range itself, for up to
// kLocalRounds rounds, before the rest goes to the global queue.  Such a step
// is bound by its dependent trips to memory (about ten, 17 us, and 4 us to the
// next one) and not by its edges; a local round takes four: the rows of the
// listed vertices with their distances, the edges, the targets' distances, the
// atomic.  The list holds the distance a vertex was listed with, so that one
// listed twice is expanded once, at the smaller.  Rounds run ahead of what
// other workgroups find, which costs some expansions at distances that are not
// final yet.
// On graphs with hubs, whose shorter paths local rounds run ahead of, only the
// smallest steps (up to 2048 items; with three rounds instead of two unit weights
// on 4096 vertices take 328 us) of small graphs have them.  RMAT graphs, us
// without local rounds and with them, weights to 255 in buckets of 2^6 and 2^13,
// unit weights, weights to 60000 in buckets of 2^13:
//   0.10M edges  574 425   387 384   242 243   622 610
//   0.20M        635 499   449 463   259 252   694 677
//   0.43M        684 524   479 495   272 267   730 723
//   0.99M        841 827   647 640   315 289   1298 1283
//   1.82M        894 880   652 689   290 304   1143 1157
//   3.73M        969 991   691 751   338 350   1210 1250
constexpr unsigned kLocalMaxHubs = 1u << 11;
constexpr int64_t kLocalHubEdges = int64_t(1) << 20;
constexpr unsigned kLocalMax = 1u << 16;  // near items: at most one batch per workgroup
// Rounds: a lattice of 2048 x 2048 takes 3.54 ms with one, 2.84 with 2, 2.87
// with 8, 3.10 with 16, one of 300,000 vertices 1.52, 0.96, 0.59 and 0.56.
constexpr int kLocalRounds = 2, kLocalRoundsNoHubs = 8;
constexpr int kLocalEdges = 2;

static_assert(kLocalMax <= kGridNoHubs * kWideBlock && kLocalMaxHubs <= kWideGrid * kWideBlock, "one batch each");

// Lists of the workgroup, in the space of the near stage (used by then).
struct LocalLists {
  uint32_t v[2][kWideBlock], d[2][kWideBlock];
  int32_t start[kWideBlock];
  uint32_t off[kWideBlock];
};
static_assert(sizeof(LocalLists) <= sizeof(Stage), "fits the stage");

__device__ __forceinline__ void relax_local(const Bufs& B, Stage& sn, Stage& sf) {
  __shared__ uint32_t s_scan[kWideWaves + 1];
  __shared__ unsigned s_count;
  SsspState* S = B.S;
  RelaxOp op = make_relax(B, sn, sf);
  LocalLists& L = *reinterpret_cast<LocalLists*>(&sn[0][0]);
  const unsigned tid = threadIdx.x, qcount = S->near_count[S->q];
  const uint32_t* __restrict__ near = B.nearq[S->q];
  uint32_t* __restrict__ nout = op.q.nq;
  uint32_t* __restrict__ hubq = B.hubq[S->hq];
  // Wavefront-collective: v to the global near queue, once a step.
  auto to_queue = [&](bool pred, uint32_t v) {
    if (__ballot(pred) == 0) return;
    const bool won = pred && atomicExch(&B.stamp[v], op.round) != op.round;
    const uint64_t mask = __ballot(won);
    if (mask == 0) return;
    unsigned base = 0;
    if (lane_id() == 0)
      base = static_cast<unsigned>(atomicAdd(&S->app, static_cast<unsigned long long>(__popcll(mask))));
    base = __builtin_amdgcn_readfirstlane(base);
    if (won) {
      const unsigned p = base + lanes_below(mask);
      if (p < B.cap) nout[p] = v; else atomicOr(&S->overflow, 1u);
    }
  };
  const unsigned per = max(kBatchMin, (qcount + gridDim.x - 1) / gridDim.x);  // at most a vertex a lane (kLocalMax)
  const uint64_t base = static_cast<uint64_t>(blockIdx.x) * per;
  unsigned count = base < qcount ? min(per, static_cast<unsigned>(qcount - base)) : 0u;
  int cur = 0;
  for (int r = 0; count > 0 && r < B.local_rounds; ++r) {  // workgroup-uniform
    uint32_t v = 0, d = 0, deg = 0;
    int32_t start = 0;
    bool in = tid < count, hub = false;
    if (in) {
      v = r == 0 ? near[base + tid] : L.v[cur][tid];
      start = B.row[v];
      deg = static_cast<uint32_t>(B.row[v + 1] - start);
      if (r == 0) {
        d = op.dist[v];
        in = B.done[v] != d;
      } else {
        d = L.d[cur][tid];
        in = __hip_atomic_load(&op.dist[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == d;
      }
      hub = in && deg > B.hub;
      if (in && (r == 0 || !hub)) B.done[v] = d;
      if (in && !hub) {
        op.edges += deg;
        op.items += 1;
      } else {
        deg = 0;
      }
    }
    if (r == 0) {  // hubs go to the hub list, expanded in this step
      const uint64_t mask = __ballot(hub);
      if (mask) {
        unsigned at = 0;
        if (lane_id() == 0) at = atomicAdd(&S->hub_count, static_cast<unsigned>(__popcll(mask)));
        at = __builtin_amdgcn_readfirstlane(at);
        if (hub) {
          const unsigned p = at + lanes_below(mask);
          if (p < B.cap) hubq[p] = v; else atomicOr(&S->overflow, 1u);
        }
      }
    } else {
      to_queue(hub, v);
    }
    uint32_t total;
    const uint32_t off = block_exclusive_scan<kWideBlock>(deg, s_scan, &total);
    L.start[tid] = start;
    L.off[tid] = off;
    L.d[cur][tid] = d;
    if (tid == 0) s_count = 0;
    __syncthreads();
    for (uint32_t e0 = 0; e0 < total; e0 += kWideBlock * kLocalEdges) {
      bool valid[kLocalEdges], to_near[kLocalEdges], to_far[kLocalEdges];
      uint32_t t[kLocalEdges], nd[kLocalEdges], dv[kLocalEdges];
#pragma unroll
      for (int k = 0; k < kLocalEdges; ++k) {
        const uint32_t e = e0 + k * kWideBlock + tid;
        valid[k] = e < total;
        t[k] = nd[k] = 0;
        if (valid[k]) {
          int lo = 0, hi = static_cast<int>(count) - 1;
          while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (L.off[mid] <= e) lo = mid; else hi = mid - 1;
          }
          const int32_t edge = L.start[lo] + static_cast<int32_t>(e - L.off[lo]);
          t[k] = static_cast<uint32_t>(B.col[edge]);
          nd[k] = L.d[cur][lo] + B.w[edge];
        }
      }
#pragma unroll
      for (int k = 0; k < kLocalEdges; ++k) dv[k] = valid[k] ? op.dist[t[k]] : 0u;
      uint32_t old[kLocalEdges];
#pragma unroll
      for (int k = 0; k < kLocalEdges; ++k) old[k] = nd[k] < dv[k] ? atomicMin(&op.dist[t[k]], nd[k]) : 0u;
      unsigned mine = 0;  // near improvements of the wavefront in this step
#pragma unroll
      for (int k = 0; k < kLocalEdges; ++k) {
        const bool better = nd[k] < old[k];
        const uint32_t nb = nd[k] >> B.shift;
        to_near[k] = better && nb <= op.bucket_end;
        to_far[k] = better && nb > op.bucket_end;
        if (to_far[k]) op.far_min = min(op.far_min, nb);
        to_far[k] = to_far[k] && old[k] == kInf;  // reached before: it is in the far pile
        mine += static_cast<unsigned>(__popcll(__ballot(to_near[k])));
      }
      op.q.far.push(to_far, t);
      op.q.after_step(kWave * kLocalEdges);
      if (mine == 0) continue;  // wavefront-uniform
      unsigned at = 0;
      if (lane_id() == 0) at = atomicAdd(&s_count, mine);
      at = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
      for (int k = 0; k < kLocalEdges; ++k) {
        const uint64_t mask = __ballot(to_near[k]);
        const unsigned p = at + lanes_below(mask);
        if (to_near[k] && p < kWideBlock) {
          L.v[cur ^ 1][p] = t[k];
          L.d[cur ^ 1][p] = nd[k];
        }
        to_queue(to_near[k] && p >= kWideBlock, t[k]);  // no room in the list
        at += static_cast<unsigned>(__popcll(mask));
      }
    }
    __syncthreads();
    count = min(s_count, static_cast<unsigned>(kWideBlock));
    cur ^= 1;
  }
  // What is left goes to the next step; the lists' space is the near stage's again.
  const uint32_t rest[1] = {tid < count ? L.v[cur][tid] : 0u};
  const bool won[1] = {tid < count && atomicExch(&B.stamp[rest[0]], op.round) != op.round};
  __syncthreads();
  op.q.near.push(won, rest);
  op.finish();
}

// The hubs of a relax step (hub_count), or with deferral the pending hubs
// of a hub step (hub_expand, 0 outside hub steps), spread over the grid;
// hub_offsets ran over the same count.
__global__ void __launch_bounds__(kWideBlock) hubs_kernel(Bufs B) {
  SsspState* S = B.S;
  const unsigned hubs = B.defer ? (S->hub_step ? S->hub_expand : 0u) : (S->mode == kRelax ? S->hub_count : 0u);
  if (hubs == 0) return;
  __shared__ Stage sn, sf;
  RelaxOp op = make_relax(B, sn, sf);
  HubCount<RelaxOp> hc{op};
  expand_hubs<kWideBlock, HubCount<RelaxOp>, kHubLanes, kWideEdges>(B.row, B.defer ? B.hubx : B.hubq[0], hubs, B.cap, B.hub_off, hc);
  if (blockIdx.x == 0 && threadIdx.x == 0) op.items += min(hubs, B.cap);
  op.finish();
}

// Advance step: far items of the new bucket go to the near queue, later
// ones are kept (their buckets fold into the running far minimum), settled ones
// are dropped.
__device__ __forceinline__ void far_split_step(const Bufs& B, Stage& sn, Stage& sk) {
  SsspState* S = B.S;
  const uint32_t* __restrict__ dist = S->dist_out;
  const uint32_t next = S->bucket, last = S->bucket + (S->width - 1);
  const unsigned fs = S->far_sel, q = S->q;
  const unsigned cnt = S->far_count[fs];
  const uint32_t* farq = B.farq[fs];
  const uint32_t round = S->round;
  uint32_t kept_min = 0xffffffffu, near_min = 0xffffffffu;
  PairQueue out(S, sn, sk, B.nearq[q ^ 1], B.farq[fs ^ 1], B.cap);
  for (uint64_t b0 = static_cast<uint64_t>(blockIdx.x) * kWideBlock; b0 < cnt;
       b0 += static_cast<uint64_t>(gridDim.x) * kWideBlock) {
    const unsigned i = static_cast<unsigned>(b0) + threadIdx.x;
    bool to_near[1] = {false}, keep[1] = {false};
    uint32_t v[1] = {0};
    if (i < cnt) {
      v[0] = farq[i];
      const uint32_t dv = dist[v[0]], b = dv >> B.shift;
      if (b >= next && b <= last) {
        near_min = min(near_min, dv);
        B.stamp[v[0]] = round;
        to_near[0] = true;
      } else if (b > last) {
        keep[0] = true;
        kept_min = min(kept_min, b);
      }
    }
    out.near.push(to_near, v);
    out.far.push(keep, v);
    out.after_step(kWave);
  }
  out.finish();
  constexpr int kW = kWideBlock / kWave;
  __shared__ uint32_t s_min[2][kW];
  kept_min = wave_min(kept_min);
  near_min = wave_min(near_min);
  if (lane_id() == 0) {
    s_min[0][threadIdx.x / kWave] = kept_min;
    s_min[1][threadIdx.x / kWave] = near_min;
  }
  __syncthreads();
  if (threadIdx.x < kWave) {
    const unsigned i = lane_id() < kW ? lane_id() : 0u;
    kept_min = wave_min(s_min[0][i]);
    near_min = wave_min(s_min[1][i]);
  }
  if (threadIdx.x == 0) {
    if (kept_min != 0xffffffffu) lower(&S->far_min, kept_min);
    if (near_min != 0xffffffffu && B.hub_span) lower(&S->near_min_next, near_min);
  }
}

// Hub step, first part: the pending hubs at or below hub_limit go to the
// expand list; the others move to the other pending list under the next
// generation's mark (the generation advances when the step closes), so the
// admission filter does not list them twice, and their smallest distance
// becomes the next step's hub_min.
// The two lists are staged in LDS and moved out with one global atomic per
// flush, not one per wavefront: the pending list can hold millions of hubs,
// and every selecting step passes over it.
__global__ void __launch_bounds__(kWideBlock) hub_select_kernel(Bufs B) {
  SsspState* S = B.S;
  if (!S->hub_step) return;
  constexpr int kQCap = 4096;
  __shared__ LdsQueue<kQCap> qs, qk;
  lq_init(qs);
  lq_init(qk);
  const uint32_t* __restrict__ dist = S->dist_out;
  const unsigned cnt = min(S->hub_count, B.cap), hq = S->hq, gen = S->hub_gen + 1;
  const uint32_t limit = S->hub_limit;
  const uint32_t* pending = B.hubq[hq];
  uint32_t kept_min = 0xffffffffu;
  for (uint64_t b0 = static_cast<uint64_t>(blockIdx.x) * kWideBlock; b0 < cnt;
       b0 += static_cast<uint64_t>(gridDim.x) * kWideBlock) {  // workgroup-uniform
    const unsigned i = static_cast<unsigned>(b0) + threadIdx.x;
    bool sel = false, keep = false;
    uint32_t h = 0;
    if (i < cnt) {
      h = pending[i];
      const uint32_t d = dist[h];
      sel = d <= limit;
      keep = !sel;
      if (keep) {
        B.hubmark[h] = gen;
        kept_min = min(kept_min, d);
      }
    }
    lq_push(qs, sel, h);
    lq_push(qk, keep, h);
    lq_flush(qs, B.hubx, &S->hub_expand, B.cap, &S->overflow, false);
    lq_flush(qk, B.hubq[hq ^ 1], &S->hub_kept, B.cap, &S->overflow, false);
  }
  lq_flush(qs, B.hubx, &S->hub_expand, B.cap, &S->overflow, true);
  lq_flush(qk, B.hubq[hq ^ 1], &S->hub_kept, B.cap, &S->overflow, true);
  kept_min = wave_min(kept_min);
  if (lane_id() == 0 && kept_min != 0xffffffffu) lower(&S->hub_min_next, kept_min);
}

// The work of a step: a relax or an advance (the step's mode picks one; the
// two never share a step, so one launch serves both).  LOCAL: with local rounds
// (see local_max); left out elsewhere, where they would cost the wide steps
// half of the wavefronts a CU holds (78 registers against 64).
template <bool LOCAL>
__global__ void __launch_bounds__(kWideBlock, LOCAL ? 4 : 8) work_kernel(Bufs B) {
  const unsigned mode = B.S->mode;
  if (mode != kRelax && mode != kAdvance) return;
  __shared__ Stage s0, s1;
  if (mode == kAdvance) {
    far_split_step(B, s0, s1);
    return;
  }
  if constexpr (LOCAL) {
    if (B.S->near_count[B.S->q] <= B.local_max) {
      relax_local(B, s0, s1);
      return;
    }
  }
  relax_step(B, s0, s1);
}

// `hubs` false: no vertex exceeds the hub threshold, so the hub list stays
// empty and its two launches are left out of the step.
void enqueue_step(const Bufs& B, bool hubs, hipStream_t s) {
  step_kernel<<<1, kWave, 0, s>>>(B.S, hubs ? nullptr : B.tally, B.defer, B.hub_span);
  if (B.local_max > 0)
    work_kernel<true><<<hubs ? kWideGrid : kGridNoHubs, kWideBlock, 0, s>>>(B);
  else
    work_kernel<false><<<hubs ? kWideGrid : kGridNoHubs, kWideBlock, 0, s>>>(B);
  if (hubs) {
    if (B.defer) hub_select_kernel<<<kHubSelectGrid, kWideBlock, 0, s>>>(B);
    launch_hub_offsets<kHubLanes * kWideEdges>(B.row, B.defer ? B.hubx : B.hubq[0], B.defer ? &B.S->hub_expand : &B.S->hub_count,
                               B.cap, B.hub_off, s);
    hubs_kernel<<<kWideGrid, kWideBlock, 0, s>>>(B);
  }
  GX_LAUNCHED("sssp step");
}

}  // namespace

extern "C" gx_status gx_sssp_delta(gx_graph* g, uint32_t src, uint32_t shift, uint32_t* dist, gx_stats* st) {
  GX_API_BEGIN
  check_graph(g);
  check_ptr(dist, "dist");
  check_vertex(g, src, "source");
  GX_REQUIRE(g->flags & GX_GRAPH_WEIGHTED, "SSSP needs uint32 edge weights");
  GX_REQUIRE(shift < 32, "shift must be < 32");
  const int64_t n = g->n;
  hipStream_t s = g->stream;
  const unsigned cap = static_cast<unsigned>(std::max<int64_t>(n, 1));
  Bufs B;
  B.row = g->row;
  B.col = g->col;
  B.w = static_cast<const uint32_t*>(g->w);
  B.dist = dist;
  B.nearq[0] = g->scratch<uint32_t>(WS_Q0, cap);
  B.nearq[1] = g->scratch<uint32_t>(WS_Q1, cap);
  B.farq[0] = g->scratch<uint32_t>(WS_Q2, cap);
  B.farq[1] = g->scratch<uint32_t>(WS_Q3, cap);
  B.hubq[0] = g->scratch<uint32_t>(WS_V0, cap);
  B.hubq[1] = g->scratch<uint32_t>(WS_BITMAP0, cap);
  B.hubx = g->scratch<uint32_t>(WS_BITMAP1, cap);
  B.stamp = g->scratch<uint32_t>(WS_V1, n);
  B.done = g->scratch<uint32_t>(WS_V3, n);
  B.hubmark = g->scratch<uint32_t>(WS_V4, n);
  B.S = g->scratch<SsspState>(WS_COUNTERS, 1);
  B.tally = g->scratch<unsigned long long>(WS_REDUCE, 2 * kWideGrid);
  B.shift = shift;
  B.cap = cap;
  B.hub_off = g->scratch<uint32_t>(WS_HUBOFF, hub_off_words(cap));
  B.hub = hub_degree();
  const int64_t refine = tune_effective("sssp.hub_refine", n, g->m);
  B.defer = static_cast<uint32_t>(tune_effective("sssp.defer_hubs", n, g->m)) | (refine > 0 ? 1u : 0u);
  B.hub_span = refine > 0 ? 1u << std::min<int64_t>(refine - 1, 31) : 0u;
  const bool hubs = max_degree(g) > static_cast<int64_t>(B.hub);
  B.batch = hubs ? kBatchMax : kWideBlock;
  B.local_max = !hubs ? kLocalMax : g->m < kLocalHubEdges && !B.defer ? kLocalMaxHubs : 0u;
  B.local_rounds = hubs ? kLocalRounds : kLocalRoundsNoHubs;
  // Graphs with hubs run on the degree-ordered copy (frontier.relabel).
  const bool relabel = hubs && tune_effective("frontier.relabel", n, g->m) != 0;
  uint32_t run_src = src;
  if (relabel) {
    build_relabeled(g);
    B.row = g->relab.row.as<int32_t>();
    B.col = g->relab.col.as<int32_t>();
    B.w = g->relab.w.as<uint32_t>();
    B.dist = g->scratch<uint32_t>(WS_V5, n);
    run_src = read_scalar(g, g->relab.new_of_old.as<uint32_t>() + src);
  }
  SsspState* host = static_cast<SsspState*>(g->host_pinned(sizeof(SsspState)));

  RegionTimer region(s);
  KernelTimer ktimer(s);
  const unsigned max_width = static_cast<unsigned>(tune_effective("sssp.max_merge", n, g->m));
  sssp_init_kernel<<<grid_for(n, kBlock, 4096), kBlock, 0, s>>>(B.dist, B.stamp, B.done, B.hubmark, n,
                                                                 run_src);
  GX_LAUNCHED("sssp_init_kernel");
  sssp_reset_kernel<<<1, kBlock, 0, s>>>(B.S, B.tally, B.nearq[0], run_src, B.dist, max_width, B.hub_span,
                                      B.hub_span != 0 && !tune_is_set("sssp.hub_refine") ? 1u : 0u);
  GX_LAUNCHED("sssp_reset_kernel");
  uint64_t key = 0;
  for (const void* p : {(const void*)B.row, (const void*)B.col, (const void*)B.w,
                        (const void*)B.nearq[0], (const void*)B.nearq[1], (const void*)B.farq[0],
                        (const void*)B.farq[1], (const void*)B.hubq[0], (const void*)B.hubq[1], (const void*)B.hubx,
                        (const void*)B.stamp, (const void*)B.done, (const void*)B.hubmark, (const void*)B.S, (const void*)B.tally, (const void*)B.hub_off})
    key = mix_key(key, reinterpret_cast<uintptr_t>(p));
  key = mix_key(mix_key(mix_key(mix_key(mix_key(mix_key(key, shift), cap), B.hub), hubs ? 1u : 0u), B.defer),
                B.hub_span);
  uint32_t replays = 0;
  for (;;) {
    ktimer.begin();
    g->replay(g->sssp_batch, key, [&](hipStream_t cs) {
      for (int i = 0; i < kStepsPerGraph; ++i) enqueue_step(B, hubs, cs);
      batch_end_kernel<<<1, kBlock, 0, cs>>>(B.S, B.tally);
      GX_LAUNCHED("batch_end_kernel");
    });
    ktimer.end();
    ++replays;
    GX_HIP(hipMemcpyAsync(host, B.S, sizeof(SsspState), hipMemcpyDeviceToHost, s));
    GX_HIP(hipStreamSynchronize(s));
    if (host->overflow) fail(GX_ERR_CAPACITY, "SSSP queue overflow");
    if (host->done) break;
  }
  if (relabel) unpermute_u32(B.dist, g->relab.new_of_old.as<uint32_t>(), dist, n, s);
  double ms = region.stop();
  if (st) {
    std::memset(st, 0, sizeof(*st));
    st->iterations = host->steps;
    st->launches = 2 + replays * (kStepsPerGraph * (hubs ? (B.defer ? 5 : 4) : 2) + 1);
    st->edges_visited = host->edges;
    st->items = host->items;
    st->elapsed_ms = ms;
    st->main_kernel_ms = ktimer.total_ms();
    st->main_kernel_launches = ktimer.count();
  }
  GX_API_END
}
