// k-core decomposition (symmetric graphs) by synchronous cascade peeling.
//
// Reference semantics: lonestar/analytics/cpu/k-core/kcore.cpp:86-95
// (degreeCounting: currentDegree = degree), :103-115 (initial dead worklist:
// currentDegree < k), :124-159 (syncCascadeKCore: every dead vertex
// decrements each neighbour with atomicSubtract; a neighbour whose old value
// was exactly k dies and joins the next worklist), :201-217 (alive:
// currentDegree >= k).  The D-IrGL GPU form is KCoreStep1/2
// (lonestar/analytics/distributed/k-core/kcore_push_cuda.py:10-87).  Every
// dead vertex is processed exactly once and decrements all its neighbours, so
// the final degree array equals the number of alive neighbours: bit-exact
// whatever the schedule.
//
// Design (gfx950): the dead frontier is expanded with the load-balanced
// workgroup expansion of frontier.hpp (hubs spread over the grid); each
// decrement is one atomicSub on the degree word, and the `old == k` winner
// appends the neighbour to the next frontier through the wavefront's LDS
// queue.  The first round's decrements take most of the call: random atomics
// run at 27 G/s on this GPU, those that meet on a line or a word much slower,
// so that the words are permuted and the hottest counted in LDS (kPage, kHotCap
// below: RMAT-22 at k = 10, peel 473 -> 233 us).  The passes over all vertices
// count per workgroup (init 53 -> 28 us, membership 171 -> 20 us).  The call:
// 899 -> 410 us.
#include <algorithm>

#include "frontier.hpp"
#include "gx_device.hpp"
#include "gx_internal.hpp"

using namespace gx;

namespace {

constexpr int kBlock = 256;

struct KcoreCounters {
  unsigned count[2];
  unsigned hub_count;
  unsigned overflow;
  unsigned in;      // dead frontier read this round (q[in]); the next is q[in ^ 1]
  unsigned active;  // this round has a frontier
  unsigned done;
  unsigned rounds;
  unsigned long long items;
  unsigned long long alive;
  unsigned hot_count;
};
__global__ void kcore_reset_kernel(KcoreCounters* c) {
  if (threadIdx.x == 0) {
    c->count[0] = c->count[1] = 0;
    c->hub_count = 0;
    c->overflow = 0;
    c->in = 0;
    c->active = 0;
    c->done = 0;
    c->rounds = 0;
    c->items = 0;
    c->alive = 0;
    c->hot_count = 0;
  }
}

constexpr int kQCap = 4096;  // kcore_init_kernel
constexpr int kHubLanes = 64;  // lanes per step of the hub pass
// In the first round (every vertex below k dies at once) many decrements land
// on the few vertices of highest degree, and atomics on one word take 12 ns
// each, one after another; on RMAT graphs the hubs' ids are powers of two
// apart, so that their words queue up on the same memory channels.  The init
// pass therefore lists up to kHotCap vertices with at least 1/8192 of the
// adjacency entries (and kHotDegree), and every workgroup counts their
// decrements in an LDS table and applies each counter with one atomicSub at
// the end of the launch; the atomic that takes a word from k or above to below
// k finds the death, so every vertex still dies exactly once.  Frontiers of
// fewer than kHotMin vertices do without: no word can take more decrements
// than that (25 us), and the table costs a few.
constexpr uint32_t kHotCap = 512;
constexpr uint32_t kHotDegree = 256;
constexpr uint32_t kHotMin = 2048;
constexpr int kHotBits = 11;  // table slots: at most a quarter in use
constexpr int kHotProbe = 4;  // a vertex that finds no slot among these is not counted
constexpr uint32_t kNoVertex = 0xffffffffu;

// On the degree-ordered copy the hottest vertices are the first ids: every word
// of the table then is the counter of its own index (RMAT-26, k = 10, with the
// words in order: 3.2 ms, with the list and permuted words 4.27).
struct HotTable {
  uint32_t id[1 << kHotBits];
  uint32_t count[1 << kHotBits];
};
constexpr uint32_t kFirstHot = 2u << kHotBits;
__device__ __forceinline__ uint32_t hot_slot(uint32_t v, int probe) {
  return (((v * 2654435769u) >> (32 - kHotBits)) + probe) & ((1u << kHotBits) - 1);
}

struct KcoreState {
  KcoreCounters c;
  uint32_t hot[kHotCap];
};

// Atomics on one cache line queue up as those on one word do.  Neighbouring ids
// are often alike (ids of RMAT graphs with few set bits are hubs), so with hubs the degree words are
// permuted within pages of kPage words: 4.4 M decrements of an RMAT
// distribution over 2^22 words take 499 us in id order, 225 us permuted
// (uniform ones 168 us).  Pages keep the passes over all vertices sequential.
// A graph without hubs keeps its order (and the lines its neighbours share), and
// so does the degree-ordered copy, whose hottest ids are all counted in LDS and
// whose degrees are read back in runs of neighbouring words (RMAT-26: the last
// pass 534 us, permuted 1020, the peel 2.47 ms either way).
constexpr uint32_t kPage = 4096;
constexpr uint32_t kPageMul = 1597;  // odd: a permutation of the page
__device__ __forceinline__ uint32_t degree_pos(uint32_t v, uint32_t mul) {
  return (v & ~(kPage - 1)) | ((v * mul) & (kPage - 1));
}
constexpr int kRoundsPerGraph = 4;
constexpr int kRoundsFirst = 2;  // first replay: many graphs need one round (plus the empty one)

// degree[v] = out-degree; vertices below k form the first dead frontier
// (staged in LDS, one global append per workgroup flush).  Vertices without
// edges are dead from the start but decrement no one, so they are left out
// of it (on RMAT graphs they are a large share of the vertices).
__global__ void __launch_bounds__(kWideBlock) kcore_init_kernel(const int32_t* __restrict__ row,
                                                            uint32_t* __restrict__ degree, int64_t n, uint32_t k,
                                                            uint32_t* __restrict__ q, KcoreState* st,
                                                            unsigned cap, uint32_t hot_min, uint32_t mul) {
  KcoreCounters* c = &st->c;
  __shared__ LdsQueue<kQCap> sq;
  lq_init(sq);
  for (int64_t p = blockIdx.x * static_cast<int64_t>(kPage); p < n; p += gridDim.x * static_cast<int64_t>(kPage)) {
    for (uint32_t i = threadIdx.x; i < kPage; i += kWideBlock) {
      const int64_t v = p + i;
      bool dead = false;
      if (v < n) {
        const uint32_t d = static_cast<uint32_t>(row[v + 1] - row[v]);
        degree[degree_pos(static_cast<uint32_t>(v), mul)] = d;
        dead = d < k && d > 0;
        if (d >= hot_min && __hip_atomic_load(&c->hot_count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < kHotCap) {
          const unsigned at = atomicAdd(&c->hot_count, 1u);
          if (at < kHotCap) st->hot[at] = static_cast<uint32_t>(v);
        }
      }
      lq_push(sq, dead, static_cast<uint32_t>(v));
      lq_flush(sq, q, &c->count[0], cap, &c->overflow, false);
    }
  }
  lq_flush(sq, q, &c->count[0], cap, &c->overflow, true);
}

// Plain pointers, the output queue picked from the device state in the
// kernel (the kernel arguments are never modified or copied).
struct PeelOp {
  const int32_t* col;
  uint32_t* degree;
  uint32_t* qout;
  KcoreCounters* c;
  WaveQueue<kWaveQCap> wq;
  uint32_t k;
  unsigned out;
  unsigned cap;
  uint32_t hub;   // frontier.hub_degree
  uint32_t mul;   // degree_pos
  HotTable* hot;  // nullptr: every decrement goes to the degree word
  bool first_hot;
  // Whether v has a counter, which then takes its decrement.
  __device__ __forceinline__ bool count_hot(uint32_t v) {
    if (!hot) return false;
    if (first_hot) {
      if (v < kFirstHot) atomicAdd(&hot->id[0] + v, 1u);
      return v < kFirstHot;
    }
    for (int p = 0; p < kHotProbe; ++p) {
      const uint32_t slot = hot_slot(v, p);
      const uint32_t id = hot->id[slot];
      if (id == v) {
        atomicAdd(&hot->count[slot], 1u);
        return true;
      }
      if (id == kNoVertex) return false;
    }
    return false;
  }
  template <int U>
  __device__ __forceinline__ void run(const bool (&valid)[U], const uint32_t (&)[U], const int32_t (&e)[U]) {
    bool dies[U];
    uint32_t v[U];
#pragma unroll
    for (int k = 0; k < U; ++k) v[k] = static_cast<uint32_t>(col[e[k]]);
#pragma unroll
    for (int k = 0; k < U; ++k) {
      dies[k] = false;
      if (valid[k]) {
        if (!count_hot(v[k])) dies[k] = atomicSub(&degree[degree_pos(v[k], mul)], 1u) == this->k;
      }
    }
    wq.push(dies, v);
  }
  __device__ __forceinline__ void after_step() {
    if (!wq.full(kWideStep)) return;
    unsigned base = 0;
    if (lane_id() == 0) base = atomicAdd(&c->count[out], wq.count);
    wq.store(__builtin_amdgcn_readfirstlane(base), qout, cap, &c->overflow);
  }
  // Workgroup-uniform: what is left, for all wavefronts with one atomic.
  __device__ __forceinline__ void finish() {
    __shared__ unsigned long long s_sum[kWideWaves + 1];
    unsigned long long total;
    const unsigned long long before = waves_exclusive_sum<kWideBlock>(wq.count, s_sum, &total);
    if (threadIdx.x == 0) s_sum[kWideWaves] = total ? atomicAdd(&c->count[out], static_cast<unsigned>(total)) : 0u;
    __syncthreads();
    wq.store(static_cast<unsigned>(s_sum[kWideWaves] + before), qout, cap, &c->overflow);
  }
};

struct KcoreBufs {
  const int32_t* row;
  const int32_t* col;
  uint32_t* degree;
  uint32_t* q0;
  uint32_t* q1;
  uint32_t* hubq;
  uint32_t* hub_off;
  KcoreCounters* c;
  const uint32_t* hot;  // listed vertices (hot_count of them)
  uint32_t k;
  unsigned cap;
  uint32_t hub;
  uint32_t mul;
  unsigned batch;  // most vertices a workgroup takes at a time
  bool first_hot;  // the hottest are the first ids
};

__device__ __forceinline__ PeelOp make_peel(const KcoreBufs& B, uint32_t (&stage)[kWideWaves][kWaveQCap],
                                            HotTable* hot) {
  const unsigned out = B.c->in ^ 1u;
  return PeelOp{B.col, B.degree, out ? B.q1 : B.q0, B.c, {stage[threadIdx.x / kWave]}, B.k, out, B.cap, B.hub,
                B.mul, hot, B.first_hot};
}

// Workgroup-uniform.  The table of the listed vertices, or nullptr when there
// are none or the frontier is small.
__device__ __forceinline__ HotTable* hot_load(HotTable& T, const KcoreBufs& B, unsigned frontier) {
  const unsigned nhot = min(B.c->hot_count, kHotCap);
  if (nhot == 0 || frontier < kHotMin) return nullptr;
  if (B.first_hot) {
    for (uint32_t i = threadIdx.x; i < kFirstHot; i += kWideBlock) (&T.id[0])[i] = 0;
    __syncthreads();
    return &T;
  }
  for (uint32_t i = threadIdx.x; i < (1u << kHotBits); i += kWideBlock) {
    T.id[i] = kNoVertex;
    T.count[i] = 0;
  }
  __syncthreads();
  if (threadIdx.x < nhot) {
    const uint32_t v = B.hot[threadIdx.x];
    for (int p = 0; p < kHotProbe; ++p)
      if (atomicCAS(&T.id[hot_slot(v, p)], kNoVertex, v) == kNoVertex) break;
  }
  __syncthreads();
  return &T;
}

// Workgroup-uniform.  Applies the workgroup's counted decrements.
__device__ __forceinline__ void hot_apply(PeelOp& op) {
  if (!op.hot) return;
  __syncthreads();
  const uint32_t slots = op.first_hot ? kFirstHot : 1u << kHotBits;
  for (uint32_t i = threadIdx.x; i < slots; i += kWideBlock) {
    const uint32_t cnt = op.first_hot ? (&op.hot->id[0])[i] : op.hot->count[i];
    bool dies[1] = {false};
    const uint32_t id[1] = {op.first_hot ? i : op.hot->id[i]};
    if (cnt) {
      const uint32_t old = atomicSub(&op.degree[degree_pos(id[0], op.mul)], cnt);
      dies[0] = old >= op.k && old - cnt < op.k;
    }
    op.wq.push(dies, id);
    op.after_step();
  }
}

__global__ void __launch_bounds__(kWideBlock) kcore_peel_kernel(KcoreBufs B) {
  KcoreCounters* c = B.c;
  if (!c->active) return;
  __shared__ uint32_t stage[kWideWaves][kWaveQCap];
  __shared__ HotTable hot;
  const unsigned in = c->in, count = c->count[in];
  PeelOp op = make_peel(B, stage, hot_load(hot, B, count));
  expand_queue<kWideBlock, PeelOp, false, kWideEdges>(B.row, in ? B.q1 : B.q0, count, B.hub, B.hubq, &c->hub_count,
                                                      B.cap, &c->overflow, op, 0, B.batch);
  hot_apply(op);
  op.finish();
}

__global__ void __launch_bounds__(kWideBlock) kcore_hubs_kernel(KcoreBufs B) {
  KcoreCounters* c = B.c;
  if (!c->active || c->hub_count == 0) return;
  __shared__ uint32_t stage[kWideWaves][kWaveQCap];
  __shared__ HotTable hot;
  PeelOp op = make_peel(B, stage, hot_load(hot, B, c->hub_count));
  expand_hubs<kWideBlock, PeelOp, kHubLanes, kWideEdges>(B.row, B.hubq, c->hub_count, B.cap, B.hub_off, op);
  hot_apply(op);
  op.finish();
}

// Round bracket, driven by the device state: a round runs while the dead
// frontier is nonempty; the end swaps the frontiers.
__device__ __forceinline__ void round_begin(KcoreCounters* c) {
  if (c->done || c->overflow || c->count[c->in] == 0) {
    c->active = 0;
    c->done = 1;
    return;
  }
  c->active = 1;
  c->count[c->in ^ 1] = 0;
  c->hub_count = 0;
  c->items += c->count[c->in];
  c->rounds += 1;
}

__device__ __forceinline__ void round_end(KcoreCounters* c) {
  if (!c->active) return;
  c->in ^= 1;
  c->active = 0;
}

__global__ void kcore_round_begin_kernel(KcoreCounters* c) {
  if (threadIdx.x == 0) round_begin(c);
}

__global__ void kcore_round_end_kernel(KcoreCounters* c) {
  if (threadIdx.x == 0) round_end(c);
}

// End of one round and begin of the next in one launch.
__global__ void kcore_round_turn_kernel(KcoreCounters* c) {
  if (threadIdx.x != 0) return;
  round_end(c);
  round_begin(c);
}

// The degrees in the caller's order (work may be degree itself: then in place),
// membership and its count.
__global__ void __launch_bounds__(kWideBlock) kcore_finish_kernel(const uint32_t* work, uint32_t mul,
                                                                  const uint32_t* __restrict__ new_of_old,
                                                                  uint32_t* degree, uint8_t* __restrict__ alive,
                                                                  int64_t n, uint32_t k, KcoreCounters* c) {
  if (!c->done) return;  // rounds are left: launched again after the next replay
  int64_t v = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  unsigned long long cnt = 0;
  for (; v < n; v += stride) {
    const uint32_t d = work[degree_pos(new_of_old ? new_of_old[v] : static_cast<uint32_t>(v), mul)];
    if (work != degree) degree[v] = d;
    const bool a = d >= k;
    if (alive) alive[v] = a ? 1 : 0;
    cnt += a ? 1ull : 0ull;
  }
  // One atomic per workgroup, few workgroups: with one per wavefront 65,536
  // of them met at one word (RMAT-22: 171 us, 10 us this way).
  __shared__ unsigned long long s_cnt[kWideBlock / kWave];
  cnt = wave_sum(cnt);
  if (lane_id() == 0) s_cnt[threadIdx.x / kWave] = cnt;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t = 0;
    for (int i = 0; i < kWideBlock / kWave; ++i) t += s_cnt[i];
    if (t) atomicAdd(&c->alive, t);
  }
}

}  // namespace

extern "C" gx_status gx_kcore(gx_graph* g, uint32_t k, uint32_t* degree, uint8_t* alive, uint64_t* alive_count,
                              gx_stats* st) {
  GX_API_BEGIN
  check_graph(g);
  check_ptr(degree, "degree");
  GX_REQUIRE(g->flags & GX_GRAPH_SYMMETRIC, "k-core needs a symmetric graph");
  const int64_t n = g->n;
  hipStream_t s = g->stream;
  const unsigned cap = static_cast<unsigned>(std::max<int64_t>(n, 1));
  uint32_t* q[2] = {g->scratch<uint32_t>(WS_Q0, cap), g->scratch<uint32_t>(WS_Q1, cap)};
  uint32_t* hubq = g->scratch<uint32_t>(WS_Q2, cap);
  uint32_t* hub_off = g->scratch<uint32_t>(WS_HUBOFF, hub_off_words(cap));
  KcoreState* state = g->scratch<KcoreState>(WS_COUNTERS, 1);
  KcoreCounters* c = &state->c;
  KcoreCounters* host = static_cast<KcoreCounters*>(g->host_pinned(sizeof(KcoreCounters)));
  RegionTimer region(s);
  KernelTimer ktimer(s);
  uint32_t launches = 2;
  // Rounds are driven on the device: rounds (begin, peel, hub layout, hubs,
  // end) captured in HIP graphs, kRoundsFirst for the first replay and
  // kRoundsPerGraph for the next ones, replayed until the state says done,
  // and the membership pass runs after
  // the replay that ends with it, so the host synchronises once per replay.
  KcoreBufs B{g->row, g->col, degree, q[0], q[1], hubq, hub_off, c, state->hot, k, cap, hub_degree(), 1u, kWideBlock, false};
  // No vertex above the hub threshold: the hub list stays empty and its two
  // launches are left out of each round.
  const bool hubs = max_degree(g) > static_cast<int64_t>(B.hub);
  // Graphs with hubs peel on the degree-ordered copy of the CSR
  // (frontier.relabel): the decrements mostly land on the hubs, whose degree
  // words then share a few cached megabytes; the membership pass maps the
  // degrees back.
  const bool relabel = hubs && tune_effective("frontier.relabel", n, g->m) != 0;
  if (relabel) {
    build_relabeled(g);
    B.row = g->relab.row.as<int32_t>();
    B.col = g->relab.col.as<int32_t>();
  }
  if (hubs) {
    B.degree = g->scratch<uint32_t>(WS_V5, (static_cast<size_t>(cap) + kPage - 1) / kPage * kPage);
    if (!relabel) B.mul = kPageMul;
    B.batch = kBatchMax;
    B.first_hot = relabel;
  }
  const uint32_t hot_min = static_cast<uint32_t>(std::max<int64_t>(kHotDegree, g->m >> 13));
  kcore_reset_kernel<<<1, 64, 0, s>>>(c);
  kcore_init_kernel<<<grid_for(n, kPage, kWideGrid), kWideBlock, 0, s>>>(B.row, B.degree, n, k, q[0], state, cap,
                                                                            hot_min, B.mul);
  GX_LAUNCHED("kcore_init_kernel");
  uint64_t key = 0;
  for (const void* p : {(const void*)B.row, (const void*)B.col, (const void*)B.degree, (const void*)B.q0,
                        (const void*)B.q1, (const void*)B.hubq, (const void*)B.hub_off, (const void*)B.c})
    key = mix_key(key, reinterpret_cast<uintptr_t>(p));
  key = mix_key(mix_key(mix_key(mix_key(key, k), cap), B.hub), hubs ? 1u : 0u);
  uint32_t replays = 0, slots = 0;
  for (;;) {
    const int nr = replays == 0 ? kRoundsFirst : kRoundsPerGraph;
    ktimer.begin();
    g->replay(replays == 0 ? g->kcore_head : g->kcore_batch, key, [&](hipStream_t cs) {
      kcore_round_begin_kernel<<<1, 64, 0, cs>>>(c);
      for (int i = 0; i < nr; ++i) {
        kcore_peel_kernel<<<kWideGrid, kWideBlock, 0, cs>>>(B);
        if (hubs) {
          launch_hub_offsets<kHubLanes * kWideEdges>(B.row, B.hubq, &c->hub_count, cap, B.hub_off, cs);
          kcore_hubs_kernel<<<kWideGrid, kWideBlock, 0, cs>>>(B);
        }
        if (i + 1 < nr)
          kcore_round_turn_kernel<<<1, 64, 0, cs>>>(c);
        else
          kcore_round_end_kernel<<<1, 64, 0, cs>>>(c);
      }
      GX_LAUNCHED("kcore rounds");
    });
    ktimer.end();
    ++replays;
    slots += static_cast<uint32_t>(nr);
    kcore_finish_kernel<<<grid_for(n, kWideBlock, kWideGrid), kWideBlock, 0, s>>>(
        B.degree, B.mul, relabel ? g->relab.new_of_old.as<uint32_t>() : nullptr, degree, alive, n, k, c);
    GX_LAUNCHED("kcore_finish_kernel");
    GX_HIP(hipMemcpyAsync(host, c, sizeof(KcoreCounters), hipMemcpyDeviceToHost, s));
    GX_HIP(hipStreamSynchronize(s));
    if (host->overflow) fail(GX_ERR_CAPACITY, "k-core worklist overflow");
    if (host->done) break;
  }
  launches += slots * (hubs ? 4 : 2) + 2 * replays;
  const uint32_t rounds = host->rounds;
  const uint64_t items = host->items;
  double ms = region.stop();
  if (alive_count) *alive_count = host->alive;
  if (st) {
    std::memset(st, 0, sizeof(*st));
    st->iterations = rounds;
    st->launches = launches;
    st->items = items;
    st->elapsed_ms = ms;
    st->main_kernel_ms = ktimer.total_ms();
    st->main_kernel_launches = ktimer.count();
  }
  GX_API_END
}
