// Layout and work tables of the propagation-blocked PageRank sweep
// (pr_blocking.hpp), built once per graph from the CSR and the degree order.
//
//  1. key_kernel: one 64-bit key per edge, (run, source in chunk, destination
//     in bin) in degree-order ids, run = chunk of the source * bins + bin of
//     the destination; a radix sort over the used bits puts the edges in
//     layout order (deterministic: the graph has no duplicate edges).
//  2. mark_kernel: dst16 with the group flag, the flag array for the group
//     numbering, and the edge and group counts per run (one atomic per run of
//     equal keys in a wavefront).
//  3. exclusive scans: group number of every edge's group start, start of
//     every run in edges and in groups; bin_major_kernel moves dst16 into
//     bin-major run order (the runs of one bin, from every chunk, in one
//     stretch, long runs first, then mid, then short: each of phase 2's
//     three passes over a bin reads one contiguous part); group_kernel
//     writes gsrc16 (groups stay in run-major order, as phase 1 writes them).
//  4. run_classes_kernel and two scans over (bin, class, chunk) and (class,
//     bin, chunk): where every run's edges and jobs start; jobs_kernel writes
//     the phase-2 jobs (start in bin-major dst16, length, group base).
//  5. host: phase-1 pieces per chunk (in groups) and tasks (bins, heavy bins
//     sliced), sorted longest first.
// The tables have bins^2 entries (16.7 M for 2^26 vertices); made on the host,
// with the job lists in a vector per bin, they took 150 ms of the 470 ms of a
// first solve of RMAT-26.
//
// Edges within a run are in (source, destination) order: neighbouring edges
// of a group have distinct, ascending destinations, so a wavefront's adds
// mostly hit different LDS words.
#include <algorithm>
#include <vector>

#include "pr_blocking.hpp"

namespace gx {
namespace pb {
namespace {

constexpr int kBuildBlock = 256;

// Per wavefront: lanes whose key differs from the previous lane's start a
// run; returns the run heads as a mask and the length of the caller's run
// (valid on head lanes).
__device__ __forceinline__ uint64_t run_heads(bool valid, uint32_t key, unsigned lane, unsigned nvalid,
                                              unsigned& len) {
  const uint32_t prev = __shfl_up(key, 1);
  const bool head = valid && (lane == 0 || prev != key);
  const uint64_t heads = __ballot(head);
  const uint64_t above = lane == 63 ? 0ull : (heads >> (lane + 1)) << (lane + 1);
  const unsigned next = above ? static_cast<unsigned>(__builtin_ctzll(above)) : nvalid;
  len = next - lane;
  return heads;
}

__global__ void __launch_bounds__(kBuildBlock) key_kernel(const uint32_t* __restrict__ esrc,
                                                          const int32_t* __restrict__ col,
                                                          const uint32_t* __restrict__ rank, int64_t m, uint32_t nb,
                                                          uint64_t* __restrict__ keys) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kBuildBlock;
  for (int64_t e = blockIdx.x * static_cast<int64_t>(kBuildBlock) + threadIdx.x; e < m; e += stride) {
    const uint32_t u = rank[esrc[e]], v = rank[col[e]];
    const uint64_t run = static_cast<uint64_t>(u >> kShift) * nb + (v >> kShift);
    keys[e] = (run << (2 * kShift)) | (static_cast<uint64_t>(u & (kSpan - 1)) << kShift) | (v & (kSpan - 1));
  }
}

// Sorted keys -> dst16 (+ group flag), flag[e] (0/1), edges and groups per run.
__global__ void __launch_bounds__(kBuildBlock) mark_kernel(const uint64_t* __restrict__ keys, int64_t m,
                                                           uint16_t* __restrict__ dst16, uint32_t* __restrict__ flag,
                                                           uint32_t* __restrict__ cnt, uint32_t* __restrict__ gcnt) {
  const unsigned lane = lane_id();
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kBuildBlock;
  for (int64_t e0 = blockIdx.x * static_cast<int64_t>(kBuildBlock) + (threadIdx.x & ~(kWave - 1)); e0 < m;
       e0 += stride) {
    const int64_t e = e0 + lane;
    const bool valid = e < m;
    const unsigned nvalid = static_cast<unsigned>(m - e0 < kWave ? m - e0 : kWave);
    const uint64_t k = valid ? keys[e] : 0ull;
    const bool first = valid && (e == 0 || (keys[e - 1] >> kShift) != (k >> kShift));
    const uint32_t run = valid ? static_cast<uint32_t>(k >> (2 * kShift)) : 0xffffffffu;
    if (valid) {
      dst16[e] = static_cast<uint16_t>((k & (kSpan - 1)) | (first ? kFirst : 0u));
      flag[e] = first ? 1u : 0u;
    }
    unsigned len;
    const uint64_t heads = run_heads(valid, run, lane, nvalid, len);
    const uint64_t f = __ballot(first);
    if ((heads >> lane) & 1ull) {
      const uint64_t span = (len >= 64 ? ~0ull : ((uint64_t(1) << len) - 1)) << lane;
      atomicAdd(&cnt[run], len);
      atomicAdd(&gcnt[run], static_cast<uint32_t>(__popcll(f & span)));
    }
  }
}

// gsrc16[group] = source in chunk, for every edge that opens a group.
__global__ void __launch_bounds__(kBuildBlock) group_kernel(const uint64_t* __restrict__ keys,
                                                            const uint32_t* __restrict__ flag,
                                                            const uint32_t* __restrict__ gpos, int64_t m,
                                                            uint16_t* __restrict__ gsrc16) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kBuildBlock;
  for (int64_t e = blockIdx.x * static_cast<int64_t>(kBuildBlock) + threadIdx.x; e < m; e += stride)
    if (flag[e]) gsrc16[gpos[e]] = static_cast<uint16_t>((keys[e] >> kShift) & (kSpan - 1));
}

// Job class of the first job of a run of len edges: long, mid or short.
__device__ __forceinline__ int run_class(uint32_t len) { return len > kMid ? 0 : (len > kShort ? 1 : 2); }

// Per run (chunk, bin): its edges at (bin, class of its first job, chunk), and
// its jobs at (class, bin, chunk); 0 in the other classes.
__global__ void __launch_bounds__(kBuildBlock) run_classes_kernel(const uint32_t* __restrict__ cstart, int64_t nb,
                                                                  uint32_t* __restrict__ edges,
                                                                  uint32_t* __restrict__ jobs) {
  const int64_t nkeys = nb * nb, stride = static_cast<int64_t>(gridDim.x) * kBuildBlock;
  for (int64_t i = blockIdx.x * static_cast<int64_t>(kBuildBlock) + threadIdx.x; i < nkeys; i += stride) {
    const int64_t b = i / nb, c = i - b * nb;  // chunks vary fastest: the writes are sequential
    const uint32_t len = cstart[c * nb + b + 1] - cstart[c * nb + b];
    const uint32_t tail = len % kJob;
    const int first = run_class(len), last = run_class(tail);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      edges[(b * 3 + k) * nb + c] = k == first ? len : 0u;
      jobs[(k * nb + b) * nb + c] = (k == 0 ? len / kJob : 0u) + (tail > 0 && k == last ? 1u : 0u);
    }
  }
}

// Where run r of len edges starts in bin-major order.
__device__ __forceinline__ uint32_t run_start(const uint32_t* __restrict__ estart, int64_t nb, uint32_t r,
                                              uint32_t len) {
  const int64_t c = r / nb, b = r - c * nb;
  return estart[(b * 3 + run_class(len)) * nb + c];
}

// dst16 from run-major (chunk, bin) order into bin-major order: phase 2 reads
// the runs of one bin, from every chunk, as one stretch of dst16, and inside
// it the runs whose first job is long, then mid, then short, so that each of
// its three passes over the bin (one per job class) reads a contiguous part.
// Edge e of run r moves from cstart[r] + i to the run's start + i.
__global__ void __launch_bounds__(kBuildBlock) bin_major_kernel(const uint64_t* __restrict__ keys, int64_t m,
                                                                int64_t nb, const uint32_t* __restrict__ cstart,
                                                                const uint32_t* __restrict__ estart,
                                                                const uint16_t* __restrict__ in,
                                                                uint16_t* __restrict__ out) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kBuildBlock;
  for (int64_t e = blockIdx.x * static_cast<int64_t>(kBuildBlock) + threadIdx.x; e < m; e += stride) {
    const uint32_t r = static_cast<uint32_t>(keys[e] >> (2 * kShift));
    const uint32_t c0 = cstart[r];
    out[run_start(estart, nb, r, cstart[r + 1] - c0) + (static_cast<uint32_t>(e) - c0)] = in[e];
  }
}

// The jobs of every run: full ones, then the tail, at the run's place in the
// list of their class.  A lane takes a run; the full jobs of long runs are
// written by the wavefront together.
__global__ void __launch_bounds__(kBuildBlock) jobs_kernel(const uint32_t* __restrict__ cstart, int64_t nb,
                                                           const uint32_t* __restrict__ estart,
                                                           const uint32_t* __restrict__ jstart,
                                                           const uint32_t* __restrict__ gpos, Job* __restrict__ jobs) {
  const int64_t nkeys = nb * nb, stride = static_cast<int64_t>(gridDim.x) * kBuildBlock;
  const unsigned lane = lane_id();
  for (int64_t i0 = blockIdx.x * static_cast<int64_t>(kBuildBlock) + (threadIdx.x & ~(kWave - 1)); i0 < nkeys;
       i0 += stride) {
    const int64_t i = i0 + lane;
    uint32_t from = 0, to = 0, len = 0, at = 0;  // run-major start, bin-major start, edges, first full job
    if (i < nkeys) {
      const int64_t b = i / nb, c = i - b * nb;
      from = cstart[c * nb + b];
      len = cstart[c * nb + b + 1] - from;
      if (len > 0) {
        to = estart[(b * 3 + run_class(len)) * nb + c];
        at = jstart[b * nb + c];
        const uint32_t full = len / kJob, tail = len % kJob;
        if (tail > 0) {
          const int k = run_class(tail);
          const uint32_t p = k == 0 ? at + full : jstart[(k * nb + b) * nb + c];
          jobs[p] = Job{to + full * kJob, tail, gpos[from + full * kJob] - 1u};
        }
      }
    }
    uint64_t runs = __ballot(len >= kJob);
    while (runs) {
      const int r = __ffsll(static_cast<unsigned long long>(runs)) - 1;
      runs &= runs - 1;
      const uint32_t full = static_cast<uint32_t>(__builtin_amdgcn_readlane(len, r)) / kJob;
      const uint32_t f0 = __builtin_amdgcn_readlane(from, r), t0 = __builtin_amdgcn_readlane(to, r);
      const uint32_t a0 = __builtin_amdgcn_readlane(at, r);
      for (uint32_t j = lane; j < full; j += kWave) jobs[a0 + j] = Job{t0 + j * kJob, kJob, gpos[f0 + j * kJob] - 1u};
    }
  }
}

// out[i] = in[i * step] for i in [0, count).
__global__ void strided_kernel(const uint32_t* __restrict__ in, int64_t step, int64_t count,
                               uint32_t* __restrict__ out) {
  for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < count;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x)
    out[i] = in[i * step];
}

// One workgroup per bin: its jobs lie in its stretch of dst16 and hold as many
// edges as it has; raises *bad otherwise.
__global__ void __launch_bounds__(kBuildBlock) check_jobs_kernel(const Job* __restrict__ jobs, int64_t nb,
                                                                 const uint32_t* __restrict__ first,
                                                                 const uint32_t* __restrict__ bin_edge,
                                                                 uint32_t* __restrict__ bad) {
  __shared__ unsigned long long s_sum[kBuildBlock / kWave];
  for (int64_t b = blockIdx.x; b < nb; b += gridDim.x) {
    const uint32_t e0 = bin_edge[b], e1 = bin_edge[b + 1];
    unsigned long long sum = 0;
    bool ok = true;
    for (int k = 0; k < 3; ++k)
      for (uint32_t j = first[k * nb + b] + threadIdx.x; j < first[k * nb + b + 1]; j += kBuildBlock) {
        const Job J = jobs[j];
        ok = ok && J.len > 0 && J.len <= kJob && J.start >= e0 && J.start < e1 && J.len <= e1 - J.start;
        sum += J.len;
      }
    sum = wave_sum(sum);
    if (lane_id() == 0) s_sum[threadIdx.x / kWave] = sum;
    __syncthreads();
    unsigned long long all = 0;
    for (int w = 0; w < kBuildBlock / kWave; ++w) all += s_sum[w];
    if (!ok || all != e1 - e0) *bad = 1u;
    __syncthreads();
  }
}

// Number of vertices with out-edges: out-degrees are non-increasing in
// degree order, so it is the first index whose out-degree is 0 (one thread,
// binary search).
__global__ void nonzero_kernel(const uint32_t* __restrict__ outdeg, int64_t n, int64_t* __restrict__ out) {
  if (blockIdx.x != 0 || threadIdx.x != 0) return;
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    const int64_t mid = lo + ((hi - lo) >> 1);
    if (outdeg[mid] > 0) lo = mid + 1; else hi = mid;
  }
  *out = lo;
}

}  // namespace

void build_layout(gx_graph* g) {
  DegreeOrder& D = g->degree_order;
  PbLayout& L = D.pb;
  if (L.ready) return;
  const int64_t n = g->n, m = g->m;
  GX_REQUIRE(D.ready, "propagation blocking needs the degree order");
  GX_REQUIRE(supported(n, m), "graph too large or empty for the propagation-blocked sweep");
  hipStream_t s = g->stream;
  const int64_t nb = (n + kSpan - 1) / kSpan;
  const int64_t nkeys = nb * nb;
  auto scalar = [s](const uint32_t* d) {
    uint32_t v = 0;
    GX_HIP(hipMemcpyAsync(&v, d, 4, hipMemcpyDeviceToHost, s));
    GX_HIP(hipStreamSynchronize(s));
    return v;
  };

  int64_t ngroups = 0;
  // First job of every (class, bin), and one past the last; first edge of
  // every bin in bin-major order; first group of every chunk.
  std::vector<uint32_t> first(3 * nb + 1), bin_edge(nb + 1), chunk_group(nb + 1);
  {
    // One working allocation of 18 bytes an edge and 64 a run: the keys' two
    // buffers, of which the one that the sort leaves free takes the flags and
    // their scan, the run-major dst16, the tables.  Large allocations are what a
    // first solve waits for: some ten of them, 40 bytes an edge, could take a
    // second or more where the device's memory had been in use (first solve of
    // RMAT-26 on an idle device 322 -> 311 ms).
    DevBuf arena;
    size_t used = 0;
    auto carve = [&used](size_t bytes) {
      const size_t at = used;
      used += (bytes + 255) & ~size_t(255);
      return at;
    };
    const size_t o_a = carve(m * 8 + 64), o_b = carve(m * 8 + 64), o_d16 = carve(m * 2);
    const size_t o_cnt = carve((nkeys + 1) * 4), o_gcnt = carve((nkeys + 1) * 4), o_cur = carve((nkeys + 1) * 4),
                 o_gcur = carve((nkeys + 1) * 4);
    const size_t o_ecount = carve((3 * nkeys + 1) * 4), o_jcount = carve((3 * nkeys + 1) * 4),
                 o_estart = carve((3 * nkeys + 1) * 4), o_jstart = carve((3 * nkeys + 1) * 4);
    const size_t o_small = carve((5 * nb + 4) * 4);
    arena.ensure(used);
    char* base = arena.as<char>();
    auto words = [base](size_t o) { return reinterpret_cast<uint32_t*>(base + o); };
    uint64_t* keys = reinterpret_cast<uint64_t*>(base + o_a);
    uint64_t* other = reinterpret_cast<uint64_t*>(base + o_b);
    uint32_t* esrc = words(o_b);  // done with before the sort
    edge_sources(g->row, n, m, esrc, s);
    key_kernel<<<grid_for(m, kBuildBlock, 1 << 16), kBuildBlock, 0, s>>>(esrc, g->col, D.new_of_old.as<uint32_t>(), m,
                                                                         static_cast<uint32_t>(nb), keys);
    GX_LAUNCHED("pb key_kernel");
    int run_bits = 0;
    while ((int64_t(1) << run_bits) < nkeys) ++run_bits;
    const uint64_t* sorted = radix_sort_pair_u64(keys, other, m, 2 * kShift + run_bits, s);
    uint32_t* flag = sorted == keys ? words(o_b) : words(o_a);
    uint32_t* gpos = flag + m + 1;  // exclusive scan of the group flags
    uint32_t *cnt = words(o_cnt), *gcnt = words(o_gcnt), *cur = words(o_cur), *gcur = words(o_gcur);
    uint32_t *ecount = words(o_ecount), *jcount = words(o_jcount), *estart = words(o_estart),
             *jstart = words(o_jstart);
    uint16_t* d16 = reinterpret_cast<uint16_t*>(base + o_d16);  // run-major; L.dst16 gets it bin-major below
    GX_HIP(hipMemsetAsync(cnt, 0, (nkeys + 1) * 4, s));
    GX_HIP(hipMemsetAsync(gcnt, 0, (nkeys + 1) * 4, s));
    GX_HIP(hipMemsetAsync(flag + m, 0, 4, s));
    mark_kernel<<<grid_for(m, kBuildBlock, 1 << 16), kBuildBlock, 0, s>>>(
        sorted, m, d16, flag, cnt, gcnt);
    GX_LAUNCHED("pb mark_kernel");
    exclusive_scan_u32(cnt, cur, nkeys + 1, s);
    exclusive_scan_u32(gcnt, gcur, nkeys + 1, s);
    exclusive_scan_u32(flag, gpos, m + 1, s);
    const uint32_t edges = scalar(cur + nkeys), groups = scalar(gcur + nkeys), total = scalar(gpos + m);
    ngroups = total;
    GX_REQUIRE(edges == static_cast<uint32_t>(m), "propagation-blocking layout: edge count mismatch");
    GX_REQUIRE(groups == total && ngroups >= 1 && ngroups <= m,
               "propagation-blocking layout: group count mismatch");
    const unsigned kgrid = grid_for(nkeys, kBuildBlock, 1 << 16);
    GX_HIP(hipMemsetAsync(ecount + 3 * nkeys, 0, 4, s));
    GX_HIP(hipMemsetAsync(jcount + 3 * nkeys, 0, 4, s));
    run_classes_kernel<<<kgrid, kBuildBlock, 0, s>>>(cur, nb, ecount, jcount);
    GX_LAUNCHED("pb run_classes_kernel");
    exclusive_scan_u32(ecount, estart, 3 * nkeys + 1, s);
    exclusive_scan_u32(jcount, jstart, 3 * nkeys + 1, s);
    uint32_t* d_first = words(o_small);  // the three small tables, then the check's flag
    uint32_t* d_bin = d_first + 3 * nb + 1;
    uint32_t* d_chunk = d_bin + nb + 1;
    uint32_t* d_bad = d_chunk + nb + 1;
    const unsigned sgrid = grid_for(3 * nb + 1, kBuildBlock, 256);
    strided_kernel<<<sgrid, kBuildBlock, 0, s>>>(jstart, nb, 3 * nb + 1, d_first);
    strided_kernel<<<sgrid, kBuildBlock, 0, s>>>(estart, 3 * nb, nb + 1, d_bin);
    strided_kernel<<<sgrid, kBuildBlock, 0, s>>>(gcur, nb, nb + 1, d_chunk);
    GX_LAUNCHED("pb strided_kernel");
    GX_HIP(hipMemsetAsync(d_bad, 0, 4, s));
    GX_HIP(hipStreamSynchronize(s));
    GX_HIP(hipMemcpy(first.data(), d_first, first.size() * 4, hipMemcpyDeviceToHost));
    GX_HIP(hipMemcpy(bin_edge.data(), d_bin, bin_edge.size() * 4, hipMemcpyDeviceToHost));
    GX_HIP(hipMemcpy(chunk_group.data(), d_chunk, chunk_group.size() * 4, hipMemcpyDeviceToHost));
    GX_REQUIRE(bin_edge[nb] == static_cast<uint32_t>(m), "propagation-blocking layout: bin-major offsets");
    L.dst16.ensure(m * 2);
    bin_major_kernel<<<grid_for(m, kBuildBlock, 1 << 16), kBuildBlock, 0, s>>>(
        sorted, m, nb, cur, estart, d16, L.dst16.as<uint16_t>());
    GX_LAUNCHED("pb bin_major_kernel");
    L.jobs.ensure(std::max<size_t>(first[3 * nb], 1) * sizeof(Job));
    jobs_kernel<<<kgrid, kBuildBlock, 0, s>>>(cur, nb, estart, jstart,
                                              gpos, L.jobs.as<Job>());
    GX_LAUNCHED("pb jobs_kernel");
    check_jobs_kernel<<<static_cast<unsigned>(std::min<int64_t>(nb, 4096)), kBuildBlock, 0, s>>>(
        L.jobs.as<Job>(), nb, d_first, d_bin, d_bad);
    GX_LAUNCHED("pb check_jobs_kernel");
    L.gsrc16.ensure(ngroups * 2);
    group_kernel<<<grid_for(m, kBuildBlock, 1 << 16), kBuildBlock, 0, s>>>(
        sorted, flag, gpos, m, L.gsrc16.as<uint16_t>());
    GX_LAUNCHED("pb group_kernel");
    GX_HIP(hipStreamSynchronize(s));
    GX_REQUIRE(scalar(d_bad) == 0, "propagation-blocking layout: jobs do not cover their bin");
  }

  // Phase-1 pieces: the groups of every nonempty chunk in slices of
  // kPieceEntries.
  std::vector<Piece> pieces;
  for (int64_t c = 0; c < nb; ++c) {
    const uint32_t a = chunk_group[c], b = chunk_group[c + 1];
    for (uint64_t p = a; p < b; p += kPieceEntries)
      pieces.push_back(Piece{static_cast<uint32_t>(c), static_cast<uint32_t>(p),
                             static_cast<uint32_t>(std::min<uint64_t>(b, p + kPieceEntries)), 0u});
  }

  // Tasks: a bin with at most `task_entries` edges (knob "pr.task_edges")
  // is one task; a heavier bin is cut into slices of about that many (long,
  // then mid, then short jobs) that share a global accumulator slot.  The
  // default, m / 1024 within [2^19, 2^20] (pr_task_edges_default), grows the
  // tasks of graphs with more than 2^29 edges only, which still get about
  // four tasks per CU.  A slice closes at the first job that reaches the
  // limit, so it holds up to kJob - 1 edges more.
  // Smaller graphs are cut finer unless the knob is set: a task is one
  // workgroup's, and the default leaves a graph of 16 M edges fewer than a
  // hundred.  m / 160, at least 2^13: RMAT with 30,000 vertices 1.95 -> 0.93 ms
  // a solve, 100,000 3.56 -> 1.6, 1 M 4.77 -> 3.3, 4 M 6.47 -> 6.2; half and
  // twice as long slices are slower at one end or the other, and from 84 M
  // edges on the default is the shorter one.
  constexpr int64_t kTasks = 160, kTaskMin = 1 << 13;
  const int64_t task_limit = tune_effective("pr.task_edges", n, m);
  const uint64_t task_entries = static_cast<uint64_t>(
      tune_is_set("pr.task_edges") ? task_limit : std::min(task_limit, std::max(m / kTasks, kTaskMin)));
  std::vector<std::pair<uint64_t, Task>> tasks;
  std::vector<Multi> multi;
  // Jobs of class cls and bin b: [first_of(cls, b), first_of(cls, b + 1)) of
  // the class's list.
  auto first_of = [&](int cls, int64_t b) { return first[cls * nb + b] - first[cls * nb]; };
  std::vector<Job> heavy;  // the jobs of one class of a bin that is cut
  for (int64_t b = 0; b < nb; ++b) {
    const uint64_t entries = bin_edge[b + 1] - bin_edge[b];
    Task t{};
    t.bin = static_cast<uint32_t>(b);
    if (entries <= task_entries) {
      t.slot = kSingle;
      for (int cls = 0; cls < 3; ++cls) {
        t.job0[cls] = first_of(cls, b);
        t.job1[cls] = first_of(cls, b + 1);
      }
      tasks.push_back({entries, t});
      continue;
    }
    t.slot = static_cast<uint32_t>(multi.size());
    multi.push_back(Multi{static_cast<uint32_t>(b), t.slot});
    // A slice starts at job j of class cls: earlier classes are done, later
    // ones start at the bin's first job; every range is empty until filled.
    auto reset = [&](int cls, uint32_t j) {
      for (int k = 0; k < 3; ++k)
        t.job0[k] = t.job1[k] = k < cls ? first_of(k, b + 1) : (k == cls ? j : first_of(k, b));
    };
    reset(0, first_of(0, b));
    uint64_t acc = 0, sum = 0;
    for (int cls = 0; cls < 3; ++cls) {
      const uint32_t j0 = first_of(cls, b), j1 = first_of(cls, b + 1);
      heavy.resize(j1 - j0);
      if (j1 > j0)
        GX_HIP(hipMemcpy(heavy.data(), L.jobs.as<Job>() + first[cls * nb + b], heavy.size() * sizeof(Job),
                         hipMemcpyDeviceToHost));
      for (uint32_t j = j0; j < j1; ++j) {
        t.job1[cls] = j + 1;
        acc += heavy[j - j0].len;
        sum += heavy[j - j0].len;
        if (acc >= task_entries) {
          tasks.push_back({acc, t});
          acc = 0;
          reset(cls, j + 1);
        }
      }
    }
    if (acc > 0) tasks.push_back({acc, t});
    GX_REQUIRE(sum == entries, "propagation-blocking layout: task size mismatch");
  }
  std::stable_sort(tasks.begin(), tasks.end(),
                   [](const std::pair<uint64_t, Task>& a, const std::pair<uint64_t, Task>& b) {
                     return a.first > b.first;
                   });

  // The tables must cover every edge exactly once, every job range must lie
  // in its bin's and every bin must be finalised once, before any launch.
  {
    uint64_t covered = 0, pieced = 0;
    std::vector<uint8_t> fin(nb, 0);
    for (const auto& pt : tasks) {
      const Task& t = pt.second;
      for (int cls = 0; cls < 3; ++cls)
        GX_REQUIRE(t.job0[cls] <= t.job1[cls] && t.job0[cls] >= first_of(cls, t.bin) &&
                       t.job1[cls] <= first_of(cls, t.bin + 1),
                   "propagation-blocking layout: bad job range");
      covered += pt.first;
      if (t.slot == kSingle) fin[t.bin] += 1;
      else GX_REQUIRE(t.slot < multi.size() && multi[t.slot].bin == t.bin, "propagation-blocking layout: bad slot");
    }
    for (const Multi& mu : multi) fin[mu.bin] += 1;
    for (int64_t b = 0; b < nb; ++b) GX_REQUIRE(fin[b] == 1, "propagation-blocking layout: bin not finalised once");
    for (const Piece& pc : pieces) {
      GX_REQUIRE(pc.p0 < pc.p1 && pc.p1 <= static_cast<uint64_t>(ngroups) && pc.chunk < nb,
                 "propagation-blocking layout: bad piece");
      pieced += pc.p1 - pc.p0;
    }
    GX_REQUIRE(covered == static_cast<uint64_t>(m) && pieced == static_cast<uint64_t>(ngroups),
               "propagation-blocking layout: edges not covered exactly once");
  }

  // Upload.
  std::vector<Task> tv(tasks.size());
  for (size_t i = 0; i < tasks.size(); ++i) tv[i] = tasks[i].second;
  L.pieces.ensure(std::max<size_t>(pieces.size(), 1) * sizeof(Piece));
  L.tasks.ensure(tv.size() * sizeof(Task));
  L.multi.ensure(std::max<size_t>(multi.size(), 1) * sizeof(Multi));
  GX_HIP(hipMemcpy(L.pieces.p, pieces.data(), pieces.size() * sizeof(Piece), hipMemcpyHostToDevice));
  GX_HIP(hipMemcpy(L.tasks.p, tv.data(), tv.size() * sizeof(Task), hipMemcpyHostToDevice));
  if (!multi.empty())
    GX_HIP(hipMemcpy(L.multi.p, multi.data(), multi.size() * sizeof(Multi), hipMemcpyHostToDevice));
  for (int cls = 0; cls < 3; ++cls) L.njobs[cls] = first[(cls + 1) * nb] - first[cls * nb];
  L.gacc.ensure(std::max<size_t>(multi.size(), 1) * kSpan * sizeof(unsigned long long));
  GX_HIP(hipMemsetAsync(L.gacc.p, 0, std::max<size_t>(multi.size(), 1) * kSpan * sizeof(unsigned long long), s));
  L.vals.ensure(ngroups * sizeof(float));
  GX_HIP(hipStreamSynchronize(s));
  L.ngroups = ngroups;
  L.nbins = nb;
  L.npieces = static_cast<int64_t>(pieces.size());
  L.ntasks = static_cast<int64_t>(tv.size());
  L.nmulti = static_cast<int64_t>(multi.size());
  L.task_limit = task_limit;
  L.task_entries = static_cast<int64_t>(task_entries);
  {
    DevBuf nz;
    nz.ensure(8);
    nonzero_kernel<<<1, 64, 0, s>>>(D.outdeg.as<uint32_t>(), n, nz.as<int64_t>());
    GX_LAUNCHED("pb nonzero_kernel");
    GX_HIP(hipMemcpy(&L.nonzero, nz.p, 8, hipMemcpyDeviceToHost));
  }
  L.ready = true;
}

}  // namespace pb
}  // namespace gx
