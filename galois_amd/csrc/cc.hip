// Connected components (symmetric graphs) with a lock-free union-find.
//
// Reference semantics: the union-find of libgalois/include/galois/UnionFind.h
// (merge :108-122 links the root with the higher address into the lower
// one; compress :66-82) driven over every edge with src < dst by
// lonestar/analytics/cpu/connected-components/ConnectedComponents.cpp
// (EdgeTiledAsync :523-613, Async :341-383).  Because a root is only ever
// linked below a smaller root, each tree's root is the minimum vertex id of
// its set, and after full compression label[v] = min id of v's component —
// the canonical labelling that LabelProp (:183-230) also produces.  The GPU
// app's hook/jump scheme (lonestar/analytics/gpu/connected-components/
// cc.cu:244-357) leaves non-minimum roots; this kernel set does not.
//
// Design (gfx950): the sampling scheme of the reference's Afforest variant
// (ConnectedComponents.cpp:654-759) on a lock-free GPU union-find:
//  1. every vertex starts below its first neighbour when that has the smaller
//     id (a strictly descending forest, no atomics), one pass links the first
//     two neighbours that this left out, then compress;
//  2. estimate the largest component from 1024 hashed samples of roots;
//  3. hook the remaining edges of every vertex outside that component (load
//     balanced with frontier.hpp over a compacted vertex list; hubs spread
//     over the grid).  Edges of vertices inside it need no hooking: the graph
//     is symmetric, so their other endpoint hooks the edge if it matters;
//  4. compress again, unless no vertex was left to hook.
// find() uses path halving on cached loads and stores (see find_root); linking
// is one atomicCAS of the higher root onto the lower one, so roots stay
// component minima and the labels are the canonical min labels.
#include <algorithm>
#include <mutex>

#include "frontier.hpp"
#include "gx_device.hpp"
#include "gx_internal.hpp"

using namespace gx;

namespace {

constexpr int kBlock = 256;

// Relaxed loads and stores that the nearest cache may serve.  A word only ever
// changes from its own id to a smaller id of the same set (by an atomicCAS)
// and from one proper ancestor to another (by path halving), so a stale value
// is still an ancestor: a find that ends early at a stale root is corrected in
// unite(), which reads the root's word at agent scope before it links it.  At
// agent scope every hop would miss the L1.
__device__ __forceinline__ uint32_t ld(const uint32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}
__device__ __forceinline__ void st(uint32_t* p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// Root of x (as far as the cached values show) with path halving: every
// visited node is re-pointed to its grandparent.  Only non-roots are rewritten
// and always to an ancestor, so the writes are benign under concurrent linking.
__device__ __forceinline__ uint32_t find_root(uint32_t* parent, uint32_t x) {
  uint32_t p = ld(&parent[x]);
  while (p != x) {
    const uint32_t gp = ld(&parent[p]);
    if (gp != p) st(&parent[x], gp);
    x = gp;
    p = ld(&parent[x]);
  }
  return x;
}

// Every round ends the loop or moves a to a smaller id: what the root's word
// holds, when not a itself, is below a.  The plain read before the CAS and the
// store after a miss are what makes linking fast where many vertices meet in
// one large tree: its root is linked once, and without them every later vertex
// that still sees the old root issues a CAS that fails, one after another at
// one address.  3,000,001 vertices, 81M edges, shuffled ids: 2.2-3.6 ms a call
// with CAS alone, 0.19 ms with the read (a staged linking of every 4096th,
// 256th, 16th vertex first: 0.30 ms and 0.23 ms); 2048 x 2048 lattice 1.82 ->
// 0.40 ms, RMAT-22 in generator order 0.36 -> 0.18 ms.
__device__ __forceinline__ void unite(uint32_t* parent, uint32_t a, uint32_t b) {
  for (;;) {
    a = find_root(parent, a);
    b = find_root(parent, b);
    if (a == b) return;
    if (a < b) {
      const uint32_t t = a;
      a = b;
      b = t;
    }
    // a is the higher root: link it below b.
    uint32_t cur = __hip_atomic_load(&parent[a], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (cur == a) cur = atomicCAS(&parent[a], a, b);
    if (cur == a) return;
    st(&parent[a], cur);  // linked meanwhile: an ancestor, for the next find that passes here
    a = cur;
  }
}

// Counters of a call: [0] hubs, [1] overflow, [2] rest, [3] largest.  Every
// vertex starts below its first neighbour if that is smaller.
__global__ void cc_init_kernel(const int32_t* __restrict__ row, const int32_t* __restrict__ col,
                               uint32_t* __restrict__ parent, int64_t n, unsigned* __restrict__ ctr) {
  int64_t v = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (v < 4) ctr[v] = 0;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (; v < n; v += stride) {
    const int32_t b = row[v];
    const uint32_t self = static_cast<uint32_t>(v);
    parent[v] = row[v + 1] > b ? min(self, static_cast<uint32_t>(col[b])) : self;
  }
}

// Links v with its first two neighbours, where cc_init_kernel has not.
__global__ void cc_sample_kernel(const int32_t* __restrict__ row, const int32_t* __restrict__ col,
                                 uint32_t* __restrict__ parent, int64_t n) {
  for (int64_t v = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; v < n;
       v += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int32_t b = row[v], d = row[v + 1] - b;
    if (d < 1) continue;
    const uint32_t self = static_cast<uint32_t>(v), c0 = static_cast<uint32_t>(col[b]);
    if (c0 > self) unite(parent, self, c0);
    if (d > 1) unite(parent, self, static_cast<uint32_t>(col[b + 1]));
  }
}

// Roots of 1024 hashed sample vertices, one per lane of a single workgroup;
// the most frequent one (the smallest of several) is taken as the largest
// component.  Counted in an LDS hash table of twice as many slots: a vertex's
// count is final when its table entry is.  A comparison of all pairs by 256
// lanes took 71 us, this 8 us, most of it the two dependent loads.
constexpr int kSamples = 1024;
__global__ void __launch_bounds__(kSamples) cc_largest_kernel(uint32_t* __restrict__ parent, int64_t n,
                                                              uint32_t* __restrict__ out) {
  constexpr uint32_t kSlots = 2 * kSamples, kFree = 0xffffffffu;
  __shared__ uint32_t keys[kSlots];
  __shared__ unsigned cnt[kSlots];
  __shared__ unsigned long long best;
  for (uint32_t i = threadIdx.x; i < kSlots; i += kSamples) {
    keys[i] = kFree;
    cnt[i] = 0;
  }
  if (threadIdx.x == 0) best = 0;
  __syncthreads();
  const uint64_t v = (mix64(0x43434343u + static_cast<uint64_t>(threadIdx.x)) >> 11) % static_cast<uint64_t>(n);
  const uint32_t root = find_root(parent, static_cast<uint32_t>(v));
  uint32_t slot = (root * 2654435769u) >> 21;  // 11 bits; at most half of the slots fill, so a free one is found
  for (;;) {
    const uint32_t k = atomicCAS(&keys[slot], kFree, root);
    if (k == kFree || k == root) break;
    slot = (slot + 1) & (kSlots - 1);
  }
  atomicAdd(&cnt[slot], 1u);
  __syncthreads();
  // Largest count, then smallest root.
  atomicMax(&best, (static_cast<unsigned long long>(cnt[slot]) << 32) | (0xffffffffu - root));
  __syncthreads();
  if (threadIdx.x == 0) *out = 0xffffffffu - static_cast<uint32_t>(best);
}

constexpr int kQCap = 2048;

// Vertices outside the largest component that still have unhooked edges
// (label: the roots of the compress pass; nothing was linked since).
__global__ void __launch_bounds__(kBlock) cc_rest_list_kernel(const int32_t* __restrict__ row,
                                                              const uint32_t* __restrict__ label, int64_t n,
                                                              const uint32_t* __restrict__ largest,
                                                              uint32_t* __restrict__ q, unsigned* count,
                                                              unsigned cap, unsigned* overflow) {
  __shared__ LdsQueue<kQCap> sq;
  lq_init(sq);
  const uint32_t c = *largest;
  for (int64_t b = blockIdx.x * static_cast<int64_t>(blockDim.x); b < n;
       b += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t v = b + threadIdx.x;
    bool keep = false;
    if (v < n && row[v + 1] - row[v] > 2) keep = label[v] != c;
    lq_push(sq, keep, static_cast<uint32_t>(v));
    lq_flush(sq, q, count, cap, overflow, false);
  }
  lq_flush(sq, q, count, cap, overflow, true);
}

struct HookOp {
  const int32_t* row;
  const int32_t* col;
  uint32_t* parent;
  __device__ __forceinline__ void after_step() {}
  __device__ __forceinline__ void operator()(bool valid, uint32_t u, int32_t e) {
    if (!valid || e - row[u] < 2) return;  // the first two edges were sampled
    unite(parent, u, static_cast<uint32_t>(col[e]));
  }
};

__global__ void __launch_bounds__(kBlock) cc_hook_kernel(const int32_t* __restrict__ row, HookOp op,
                                                         const uint32_t* __restrict__ q, const unsigned* count,
                                                         uint32_t* __restrict__ hubq, unsigned* hub_count,
                                                         unsigned cap, unsigned* overflow, uint32_t hub) {
  expand_queue<kBlock>(row, q, *count, hub, hubq, hub_count, cap, overflow, op);
}

__global__ void __launch_bounds__(kBlock) cc_hubs_kernel(const int32_t* __restrict__ row, HookOp op,
                                                         const uint32_t* __restrict__ hubq,
                                                         const unsigned* hub_count, unsigned cap,
                                                         const uint32_t* __restrict__ hub_off) {
  expand_hubs<kBlock>(row, hubq, *hub_count, cap, hub_off, op);
}

// rest: null, or the count of hooked vertices (with none, label is already final).
__global__ void cc_compress_kernel(uint32_t* __restrict__ parent, uint32_t* __restrict__ label, int64_t n,
                                   const unsigned* __restrict__ rest) {
  if (rest && *rest == 0) return;
  int64_t v = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (; v < n; v += stride) label[v] = find_root(parent, static_cast<uint32_t>(v));
}

// The launches of one call.  ctr: four counters; parent, rest, hubq: n words;
// hub_off: hub_off_words(cap) words.
constexpr uint32_t kCcLaunches = 9;
void enqueue_cc(const gx_graph* g, uint32_t* parent, uint32_t* rest, uint32_t* hubq, uint32_t* hub_off, unsigned* ctr,
                unsigned cap, uint32_t* label, hipStream_t s, KernelTimer* timer) {
  const int64_t n = g->n;
  const unsigned vgrid = grid_for(n, kBlock, 4096);
  cc_init_kernel<<<vgrid, kBlock, 0, s>>>(g->row, g->col, parent, n, ctr);
  GX_LAUNCHED("cc_init_kernel");
  if (timer) timer->begin();
  cc_sample_kernel<<<vgrid, kBlock, 0, s>>>(g->row, g->col, parent, n);
  cc_compress_kernel<<<vgrid, kBlock, 0, s>>>(parent, label, n, nullptr);
  cc_largest_kernel<<<1, kSamples, 0, s>>>(parent, n, &ctr[3]);
  cc_rest_list_kernel<<<vgrid, kBlock, 0, s>>>(g->row, label, n, &ctr[3], rest, &ctr[2], cap, &ctr[1]);
  HookOp op{g->row, g->col, parent};
  cc_hook_kernel<<<256 * 8, kBlock, 0, s>>>(g->row, op, rest, &ctr[2], hubq, &ctr[0], cap, &ctr[1], hub_degree());
  GX_LAUNCHED("cc_hook_kernel");
  launch_hub_offsets<kBlock>(g->row, hubq, &ctr[0], cap, hub_off, s);
  cc_hubs_kernel<<<256 * 8, kBlock, 0, s>>>(g->row, op, hubq, &ctr[0], cap, hub_off);
  if (timer) timer->end();
  GX_LAUNCHED("cc_hubs_kernel");
  cc_compress_kernel<<<vgrid, kBlock, 0, s>>>(parent, label, n, &ctr[2]);
  GX_LAUNCHED("cc_compress_kernel");
}

}  // namespace

extern "C" gx_status gx_cc(gx_graph* g, uint32_t* label, gx_stats* stp) {
  GX_API_BEGIN
  check_graph(g);
  check_ptr(label, "label");
  GX_REQUIRE(g->flags & GX_GRAPH_SYMMETRIC, "connected components needs a symmetric graph");
  const int64_t n = g->n;
  hipStream_t s = g->stream;
  const unsigned cap = static_cast<unsigned>(std::max<int64_t>(n, 1));
  uint32_t* parent = g->scratch<uint32_t>(WS_V0, cap);
  uint32_t* rest = g->scratch<uint32_t>(WS_Q1, cap);
  uint32_t* hubq = g->scratch<uint32_t>(WS_Q2, cap);
  uint32_t* hub_off = g->scratch<uint32_t>(WS_HUBOFF, hub_off_words(cap));
  unsigned* ctr = g->scratch<unsigned>(WS_COUNTERS, 4);  // [0] hubs, [1] overflow, [2] rest, [3] largest
  RegionTimer region(s);
  KernelTimer ktimer(s);
  if (n > 0) {
    enqueue_cc(g, parent, rest, hubq, hub_off, ctr, cap, label, s, &ktimer);
    unsigned hc[2];
    read_bytes(g, hc, ctr, sizeof(hc));
    if (hc[1]) fail(GX_ERR_CAPACITY, "CC vertex list overflow");
  }
  double ms = region.stop();
  if (stp) {
    std::memset(stp, 0, sizeof(*stp));
    stp->iterations = 1;
    stp->launches = n > 0 ? kCcLaunches : 0;
    stp->edges_visited = static_cast<uint64_t>(g->m);
    stp->items = static_cast<uint64_t>(n);
    stp->elapsed_ms = ms;
    stp->main_kernel_ms = ktimer.total_ms();
    stp->main_kernel_launches = ktimer.count();
  }
  GX_API_END
}

// ------------------------------------------------------------ no allocation
// gx_cc_noalloc runs the kernels of gx_cc with their scratch (union-find
// parents, the vertex list, the hub list and its offsets, four counters) in
// one file-scope device array instead of the graph's workspace, so a call
// allocates nothing.  Each device holds its own copy of the array from module
// load until the process ends; its address on the current device is resolved
// once per device (gx_init, or the first call on that device) and kept.
namespace {

constexpr int64_t kNoAllocMaxVertices = int64_t(1) << 22;
constexpr int64_t align256(int64_t b) { return (b + 255) & ~int64_t(255); }
// Byte offsets of the scratch parts for n vertices: counters, parents, vertex
// list, hub list, hub offsets.
struct NoAllocParts {
  int64_t parent, rest, hubq, hub_off, end;
};
constexpr NoAllocParts noalloc_parts(int64_t n) {
  const int64_t w = align256(4 * n);
  return NoAllocParts{256, 256 + w, 256 + 2 * w, 256 + 3 * w, 256 + 3 * w + align256(4 * hub_off_words(n))};
}
constexpr int64_t kNoAllocScratchBytes = noalloc_parts(kNoAllocMaxVertices).end;

__device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
unsigned char* g_scratch_ptr[kMaxDevices] = {};

}  // namespace

namespace gx {
unsigned char* noalloc_scratch() {
  int dev = 0;
  GX_HIP(hipGetDevice(&dev));
  GX_REQUIRE(dev >= 0 && dev < kMaxDevices, "device index beyond the no-allocation table");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    GX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    GX_REQUIRE(p != nullptr, "no device address for the no-allocation scratch");
    g_scratch_ptr[dev] = static_cast<unsigned char*>(p);
  }
  return g_scratch_ptr[dev];
}
}  // namespace gx

extern "C" gx_status gx_cc_noalloc(gx_graph* g, uint32_t* label) {
  GX_API_BEGIN
  check_graph(g);
  check_ptr(label, "label");
  GX_REQUIRE(g->flags & GX_GRAPH_SYMMETRIC, "connected components needs a symmetric graph");
  const int64_t n = g->n;
  if (n > kNoAllocMaxVertices)
    fail(GX_ERR_CAPACITY, "gx_cc_noalloc: the graph has " + std::to_string(n) +
                              " vertices; its static scratch holds at most " + std::to_string(kNoAllocMaxVertices));
  if (n == 0) return GX_OK;
  hipStream_t s = g->stream;
  unsigned char* base = noalloc_scratch();  // this device's address of `scratch`
  const NoAllocParts P = noalloc_parts(n);
  unsigned* ctr = reinterpret_cast<unsigned*>(base);  // [0] hubs, [1] overflow, [2] rest, [3] largest
  uint32_t* parent = reinterpret_cast<uint32_t*>(base + P.parent);
  uint32_t* rest = reinterpret_cast<uint32_t*>(base + P.rest);
  uint32_t* hubq = reinterpret_cast<uint32_t*>(base + P.hubq);
  uint32_t* hub_off = reinterpret_cast<uint32_t*>(base + P.hub_off);
  const unsigned cap = static_cast<unsigned>(n);  // lists hold at most n vertices: no overflow
  enqueue_cc(g, parent, rest, hubq, hub_off, ctr, cap, label, s, nullptr);
  GX_HIP(hipStreamSynchronize(s));
  GX_API_END
}
