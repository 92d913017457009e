// Layout of the blocked row sums (blocksum.hpp), built once per graph.
//
//  1. The edges, in row order, are sorted stably by chunk (a radix sort of a
//     few bits, the edge id riding in the key's upper half): (chunk, row) order.
//  2. Each chunk starts on a tile; every position gets its in-chunk index with
//     the group-end flag, its row and (weighted) its edge id.
//  3. Group ends counted per tile and scanned; every group gets its row.
//  4. Bins: blocks of rows, halved while they hold many groups, so that no
//     wavefront of phase 2 sums much more than the others.
//  5. Run starts marked and scanned, the runs sorted stably by bin.
#include <algorithm>
#include <vector>

#include "blocksum.hpp"

namespace gx {
namespace bs {
namespace {

constexpr int kB = 256;
constexpr double kAvgRun = 16.0;
constexpr int64_t kMinBins = 1024;  // bins that keep phase 2 busy: a wavefront each
constexpr uint32_t kNone = 0xffffffffu;
// 16: at 64 and 256 a graph without hubs keeps its error (1.06e-16 against 0.67e-16)
// and the solves take as long.
constexpr uint32_t kPairRow = 16, kHalveRow = 64;
constexpr uint32_t kFirst = 1u << 31;  // grow: first group of a wavefront's range

unsigned grid(int64_t n) { return grid_for(n, kB, 16384); }

__global__ void key_kernel(const int32_t* __restrict__ col, int64_t m, int shift, uint64_t* __restrict__ key) {
  for (int64_t e = blockIdx.x * static_cast<int64_t>(kB) + threadIdx.x; e < m; e += static_cast<int64_t>(gridDim.x) * kB)
    key[e] = (static_cast<uint64_t>(e) << 32) | (static_cast<uint32_t>(col[e]) >> shift);
}

// First position whose low word is >= c, for c in [0, count].
__global__ void bounds_kernel(const uint64_t* __restrict__ key, int64_t len, int64_t count, uint32_t* __restrict__ off) {
  for (int64_t c = blockIdx.x * static_cast<int64_t>(kB) + threadIdx.x; c <= count;
       c += static_cast<int64_t>(gridDim.x) * kB) {
    int64_t lo = 0, hi = len;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (static_cast<uint32_t>(key[mid]) < static_cast<uint32_t>(c)) lo = mid + 1; else hi = mid;
    }
    off[c] = static_cast<uint32_t>(lo);
  }
}

template <class T>
__global__ void set_kernel(T* __restrict__ p, T v, int64_t n) {
  for (int64_t i = blockIdx.x * static_cast<int64_t>(kB) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * kB)
    p[i] = v;
}

__global__ void place_kernel(const uint64_t* __restrict__ key, const int32_t* __restrict__ col,
                             const int32_t* __restrict__ perm, const uint32_t* __restrict__ esrc, int64_t m, int shift,
                             const uint32_t* __restrict__ off, const uint32_t* __restrict__ tile0,
                             uint16_t* __restrict__ idx16, uint32_t* __restrict__ prow, uint32_t* __restrict__ eid) {
  for (int64_t i = blockIdx.x * static_cast<int64_t>(kB) + threadIdx.x; i < m; i += static_cast<int64_t>(gridDim.x) * kB) {
    const uint64_t k = key[i];
    const uint32_t c = static_cast<uint32_t>(k), e = static_cast<uint32_t>(k >> 32);
    const uint32_t rel = static_cast<uint32_t>(i) - off[c], row = esrc[e];
    const int64_t p = static_cast<int64_t>(tile0[c]) * kTile + rel;
    const bool end = static_cast<uint32_t>(i) + 1 == off[c + 1] || (rel + 1) % (kRangeTiles * kTile) == 0 ||
                     esrc[static_cast<uint32_t>(key[i + 1] >> 32)] != row;
    idx16[p] = static_cast<uint16_t>((static_cast<uint32_t>(col[e]) & ((1u << shift) - 1)) | (end ? kEnd : 0u));
    prow[p] = row;
    if (eid) eid[p] = perm ? static_cast<uint32_t>(perm[e]) : e;
  }
}

// One wavefront per tile: group ends of the tile.
__global__ void tile_count_kernel(const uint16_t* __restrict__ idx16, int64_t ntiles, uint32_t* __restrict__ cnt) {
  const int64_t nw = static_cast<int64_t>(gridDim.x) * (kB / kWave);
  for (int64_t T = blockIdx.x * static_cast<int64_t>(kB / kWave) + threadIdx.x / kWave; T <= ntiles; T += nw) {
    uint32_t c = 0;
    if (T < ntiles)
      for (int i = 0; i < kItems; ++i) c += __popcll(__ballot((idx16[T * kTile + i * kWave + lane_id()] & kEnd) != 0));
    if (lane_id() == 0) cnt[T] = c;
  }
}

// One wavefront per tile: the rows of its groups; the first group of a range is
// marked.  range_first: first tile of each tile's range is (T - its chunk's
// first tile) % kRangeTiles == 0.
__global__ void group_kernel(const uint16_t* __restrict__ idx16, const uint32_t* __restrict__ prow, int64_t ntiles,
                             const uint32_t* __restrict__ tile_grp, const uint8_t* __restrict__ range_first,
                             uint32_t* __restrict__ grow) {
  const int64_t nw = static_cast<int64_t>(gridDim.x) * (kB / kWave);
  for (int64_t T = blockIdx.x * static_cast<int64_t>(kB / kWave) + threadIdx.x / kWave; T < ntiles; T += nw) {
    uint32_t g = tile_grp[T];
    // The first group that ends in a range need not end in its first tile.
    bool first = false;
    for (int64_t t = T;; --t) {
      if (range_first[t]) {
        first = tile_grp[t] == g;
        break;
      }
    }
    for (int i = 0; i < kItems; ++i) {
      const int64_t p = T * kTile + i * kWave + lane_id();
      const bool end = (idx16[p] & kEnd) != 0;
      const uint64_t mask = __ballot(end);
      const unsigned before = lanes_below(mask);
      if (end) grow[g + before] = prow[p] | (first && before == 0 ? kFirst : 0u);
      if (mask) first = false;
      g += static_cast<uint32_t>(__popcll(mask));
    }
  }
}

struct Bins {
  const uint32_t* block_bin;  // first bin of every block of 2^block_shift rows
  const uint8_t* block_shift; // log2 of the rows of its bins
  int shift;                  // log2 of the rows of a block
};
__device__ __forceinline__ uint32_t bin_of(const Bins& B, uint32_t row) {
  const uint32_t b = row >> B.shift;
  return B.block_bin[b] + ((row & ((1u << B.shift) - 1)) >> B.block_shift[b]);
}

__global__ void run_flag_kernel(const uint32_t* __restrict__ grow, int64_t ng, Bins B, uint32_t* __restrict__ flag) {
  for (int64_t g = blockIdx.x * static_cast<int64_t>(kB) + threadIdx.x; g <= ng; g += static_cast<int64_t>(gridDim.x) * kB) {
    if (g == ng) {
      flag[g] = 0;
      continue;
    }
    const uint32_t w = grow[g];
    flag[g] = g == 0 || (w & kFirst) || bin_of(B, w & ~kFirst) != bin_of(B, grow[g - 1] & ~kFirst) ? 1u : 0u;
  }
}

// pos: scanned flags of run_flag_kernel (group g is in run pos[g + 1] - 1);
// cut: 1 on the first group of every run and every kWave groups on.
__global__ void run_first_kernel(const uint32_t* __restrict__ pos, int64_t ng, uint32_t* __restrict__ run_g0) {
  for (int64_t g = blockIdx.x * static_cast<int64_t>(kB) + threadIdx.x; g < ng; g += static_cast<int64_t>(gridDim.x) * kB)
    if (pos[g + 1] != pos[g]) run_g0[pos[g]] = static_cast<uint32_t>(g);
}
__global__ void run_cut_kernel(const uint32_t* __restrict__ pos, const uint32_t* __restrict__ run_g0, int64_t ng,
                               uint32_t* __restrict__ cut) {
  for (int64_t g = blockIdx.x * static_cast<int64_t>(kB) + threadIdx.x; g <= ng; g += static_cast<int64_t>(gridDim.x) * kB)
    cut[g] = g < ng && (static_cast<uint32_t>(g) - run_g0[pos[g + 1] - 1]) % kWave == 0 ? 1u : 0u;
}

__global__ void run_key_kernel(const uint32_t* __restrict__ grow, int64_t ng, Bins B, const uint32_t* __restrict__ pos,
                               const uint32_t* __restrict__ bin_row, uint64_t* __restrict__ key,
                               uint32_t* __restrict__ run_g0, uint16_t* __restrict__ row16) {
  for (int64_t g = blockIdx.x * static_cast<int64_t>(kB) + threadIdx.x; g < ng; g += static_cast<int64_t>(gridDim.x) * kB) {
    const uint32_t row = grow[g] & ~kFirst, b = bin_of(B, row), p = pos[g];
    row16[g] = static_cast<uint16_t>(row - bin_row[b]);
    if (pos[g + 1] != p) {
      key[p] = (static_cast<uint64_t>(p) << 32) | b;
      run_g0[p] = static_cast<uint32_t>(g);
    }
  }
}

__global__ void run_table_kernel(const uint64_t* __restrict__ key, const uint32_t* __restrict__ run_g0, int64_t nruns,
                                 uint32_t ng, uint2* __restrict__ runs) {
  for (int64_t k = blockIdx.x * static_cast<int64_t>(kB) + threadIdx.x; k < nruns;
       k += static_cast<int64_t>(gridDim.x) * kB) {
    const uint32_t r = static_cast<uint32_t>(key[k] >> 32);
    const uint32_t a = run_g0[r], e = r + 1 < nruns ? run_g0[r + 1] : ng;
    runs[k] = make_uint2(a, e - a);
  }
}

__global__ void weights_kernel(const uint32_t* __restrict__ eid, const float* __restrict__ w, int64_t len,
                               float* __restrict__ wt) {
  for (int64_t p = blockIdx.x * static_cast<int64_t>(kB) + threadIdx.x; p < len; p += static_cast<int64_t>(gridDim.x) * kB) {
    const uint32_t e = eid[p];
    wt[p] = e == kNone ? 0.0f : w[e];
  }
}

// Per block of 2^shift rows: its edges, and those of its longest row.  One
// wavefront per block.
__global__ void block_edges_kernel(const int32_t* __restrict__ rowoff, int64_t n, int shift, int64_t nblocks,
                                   uint2* __restrict__ out) {
  const int64_t nw = static_cast<int64_t>(gridDim.x) * (kB / kWave);
  for (int64_t b = blockIdx.x * static_cast<int64_t>(kB / kWave) + threadIdx.x / kWave; b < nblocks; b += nw) {
    const int64_t r0 = b << shift, r1 = std::min<int64_t>(n, (b + 1) << shift);
    uint32_t longest = 0;
    for (int64_t r = r0 + lane_id(); r < r1; r += kWave)
      longest = max(longest, static_cast<uint32_t>(rowoff[r + 1] - rowoff[r]));
    longest = wave_max(longest);
    if (lane_id() == 0) out[b] = make_uint2(static_cast<uint32_t>(rowoff[r1] - rowoff[r0]), longest);
  }
}

int bits_for(uint64_t v) {  // bits that hold 0 .. v - 1
  int b = 1;
  while ((uint64_t(1) << b) < v) ++b;
  return b;
}

}  // namespace

// From 7 * 2^19 edges and 2^15 rows on.  Forward and adjoint in FP32 (FP64), ms, row
// sweep against blocks, and the first call on a graph, which builds both layouts:
//   n       m      again                     first
//   160000  2.56M  3.65 3.76 (3.97 4.00)     5.3 8.0 (6.2 9.0)
//   200000  3.20M  4.81 3.83 (5.36 4.46)     7.3 8.1 (8.4 8.9)
//   230000  3.68M  5.81 4.31 (5.99 4.96)     8.7 8.9 (9.2 10.1)
//   270000  4.32M  6.26 4.55 (6.27 5.26)     9.4 9.3 (10.1 10.3)
//    65536  13.1M  11.3 5.7                  14.3 11.3
//   1000000 12.0M  14.0 9.2                  17.4 16.4
//    16384  4.10M  4.44 3.52                 7.1 8.2
//    32768  3.28M  4.24 3.27                 6.1 7.4
//     8192  3.28M  4.02 4.39                 5.9 8.5
bool pays(int64_t n, int64_t m) {
  return m >= (int64_t(7) << 19) && n >= (int64_t(1) << 15) && m < (int64_t(1) << 31);
}

void layout_weights(const Plan& P, const float* w, float* wt, hipStream_t s) {
  weights_kernel<<<grid(P.ntiles * kTile), kB, 0, s>>>(P.eid, w, P.ntiles * kTile, wt);
  GX_LAUNCHED("bs::weights_kernel");
}

Plan build(gx_graph* g, const int32_t* rowoff, const int32_t* col, const int32_t* perm, int64_t n, int64_t m,
           int shift, bool weighted, BlockSums& L) {
  auto up = [](size_t b) { return (b + 255) & ~size_t(255); };
  auto view = [&]() {
    const size_t len = static_cast<size_t>(L.ntiles) * kTile;
    char* e = L.edges.as<char>();
    char* r = L.groups.as<char>();
    Plan P{};
    P.idx16 = reinterpret_cast<uint16_t*>(e);
    P.eid = reinterpret_cast<uint32_t*>(e += up(len * 2));
    P.tile_grp = reinterpret_cast<uint32_t*>(e += up(L.weighted ? len * 4 : 0));
    P.pieces = reinterpret_cast<Piece*>(e + up((L.ntiles + 1) * 4));
    P.runs = reinterpret_cast<uint2*>(r);
    P.bins = reinterpret_cast<Bin*>(r += up(L.nruns * sizeof(uint2)));
    P.row16 = reinterpret_cast<uint16_t*>(r + up(L.nbins * sizeof(Bin)));
    P.npieces = L.npieces;
    P.ntiles = L.ntiles;
    P.ngroups = L.ngroups;
    P.nruns = L.nruns;
    P.nbins = L.nbins;
    P.lds_sums = L.lds_sums;
    return P;
  };
  if (L.ready && L.shift == shift) return view();
  L.ready = false;
  L.weighted = weighted;
  GX_REQUIRE(n > 0 && m > 0, "blocked row sums over an empty graph");
  hipStream_t s = g->stream;
  const int64_t nchunks = (n + (int64_t(1) << shift) - 1) >> shift;
  // Working memory, allocated and freed once (both wait, 0.1 ms and more each; with
  // the layout's parts, the scans' and the sorts' scratch one by one, the first FP64
  // solve of 700,000 vertices, 13.8M edges, took 8.0 ms, 7.0 this way): five areas
  // used again as the steps go on.  No more groups and runs than edges; every chunk
  // pads its last tile.
  const int64_t most_tiles = (m + kTile - 1) / kTile + nchunks;
  const size_t area_a = (m + 2) * 8, area_b = (m + 2) * 8, area_c = (m + 2) * 4, area_d = most_tiles * kTile * 8,
               area_e = (m + 2) * 4;
  const int64_t most_blocks = n / 16 + 1, most_bins = n / 16 + most_blocks + 1;
  const size_t tables = 2 * (nchunks + 1) * 4 + most_tiles + 13 * most_blocks + 8 * (most_bins + 1) + 16 * 256;
  const size_t scratch = std::max(sort_words(m), scan_words(m + 2)) * 4;
  DevBuf work;
  work.ensure(up(area_a) + up(area_b) + up(area_c) + up(area_d) + up(area_e) + up(scratch) + tables);
  char* top = work.as<char>();
  auto take = [&](size_t b) {
    char* p = top;
    top += up(b);
    GX_REQUIRE(top <= work.as<char>() + work.bytes, "blocked row sums: working memory");
    return p;
  };
  char* const wa = take(area_a);
  char* const wb = take(area_b);
  char* const wc = take(area_c);
  char* const wd = take(area_d);
  char* const we = take(area_e);
  uint32_t* const tmp = reinterpret_cast<uint32_t*>(take(scratch));
  // 1. (chunk, row) order.
  uint64_t* k0 = reinterpret_cast<uint64_t*>(wa);
  uint32_t* esrc = reinterpret_cast<uint32_t*>(wc);
  uint32_t* prow = reinterpret_cast<uint32_t*>(wd);
  uint32_t* off = reinterpret_cast<uint32_t*>(take((nchunks + 1) * 4));
  uint32_t* tile0 = reinterpret_cast<uint32_t*>(take((nchunks + 1) * 4));
  key_kernel<<<grid(m), kB, 0, s>>>(col, m, shift, k0);
  GX_LAUNCHED("bs::key_kernel");
  const uint64_t* key = radix_sort_pair_u64(k0, reinterpret_cast<uint64_t*>(wb), m, bits_for(nchunks), s, tmp);
  edge_sources(rowoff, n, m, esrc, s, tmp);
  bounds_kernel<<<grid(nchunks + 1), kB, 0, s>>>(key, m, nchunks, off);
  GX_LAUNCHED("bs::bounds_kernel");
  std::vector<uint32_t> hoff(nchunks + 1), htile(nchunks + 1);
  read_bytes(g, hoff.data(), off, hoff.size() * 4);
  // 2. Tiles and pieces.  A piece has at least a range for every wavefront of
  // its workgroup and at most 32 (64K edges, against which the staging of the
  // chunk costs little), and about a thousand pieces spread a graph over the
  // CUs.
  constexpr int64_t waves = kGatherBlock / kWave;
  const uint32_t kPieceTiles = static_cast<uint32_t>(
      kRangeTiles * std::min<int64_t>(32, std::max<int64_t>(waves, m / (int64_t(1024) * kRangeTiles * kTile))));
  std::vector<Piece> pieces;
  uint32_t nt = 0;
  for (int64_t c = 0; c < nchunks; ++c) {
    htile[c] = nt;
    const uint32_t t = (hoff[c + 1] - hoff[c] + kTile - 1) / kTile;
    for (uint32_t a = 0; a < t; a += kPieceTiles)
      pieces.push_back(Piece{static_cast<uint32_t>(c), nt + a, nt + std::min(t, a + kPieceTiles), 0});
    nt += t;
  }
  htile[nchunks] = nt;
  std::vector<uint8_t> hfirst(nt);
  for (int64_t c = 0; c < nchunks; ++c)
    for (uint32_t t = htile[c]; t < htile[c + 1]; ++t) hfirst[t] = (t - htile[c]) % kRangeTiles == 0;
  // Largest first: the pieces' sizes differ where a chunk ends.
  std::stable_sort(pieces.begin(), pieces.end(),
                   [](const Piece& a, const Piece& b) { return a.tile1 - a.tile0 > b.tile1 - b.tile0; });
  L.npieces = static_cast<int64_t>(pieces.size());
  L.ntiles = nt;
  const int64_t len = static_cast<int64_t>(nt) * kTile;
  L.edges.ensure(up(len * 2) + up(weighted ? len * 4 : 0) + up((static_cast<size_t>(nt) + 1) * 4) +
                 up(pieces.size() * sizeof(Piece)));
  Plan P = view();
  auto* const idx16 = const_cast<uint16_t*>(P.idx16);
  auto* const eid = weighted ? const_cast<uint32_t*>(P.eid) : nullptr;
  auto* const tile_grp = const_cast<uint32_t*>(P.tile_grp);
  uint8_t* first = reinterpret_cast<uint8_t*>(take(hfirst.size()));
  GX_HIP(hipMemcpyAsync(const_cast<Piece*>(P.pieces), pieces.data(), pieces.size() * sizeof(Piece), hipMemcpyHostToDevice, s));
  GX_HIP(hipMemcpyAsync(tile0, htile.data(), htile.size() * 4, hipMemcpyHostToDevice, s));
  GX_HIP(hipMemcpyAsync(first, hfirst.data(), hfirst.size(), hipMemcpyHostToDevice, s));
  set_kernel<uint16_t><<<grid(len), kB, 0, s>>>(idx16, uint16_t(0), len);
  if (weighted) set_kernel<uint32_t><<<grid(len), kB, 0, s>>>(eid, kNone, len);
  place_kernel<<<grid(m), kB, 0, s>>>(key, col, perm, esrc, m, shift, off, tile0, idx16, prow, eid);
  GX_LAUNCHED("bs::place_kernel");
  // 3. Groups.
  tile_count_kernel<<<grid((nt + 1) * int64_t(kWave)), kB, 0, s>>>(idx16, nt, tile_grp);
  GX_LAUNCHED("bs::tile_count_kernel");
  exclusive_scan_u32(tile_grp, tile_grp, nt + 1, s, tmp);
  uint32_t ng = 0;
  read_bytes(g, &ng, tile_grp + nt, 4);
  L.ngroups = ng;
  uint32_t* grow = reinterpret_cast<uint32_t*>(wc);  // the edges' rows are not needed any more
  group_kernel<<<grid(nt * int64_t(kWave)), kB, 0, s>>>(idx16, prow, nt, tile_grp, first, grow);
  GX_LAUNCHED("bs::group_kernel");
  // 4. Bins: rows per block so that a run holds about 16 groups (a quarter of
  // a wavefront's lanes), between 512 and 4096 (4 and 32 KB of LDS sums); where that
  // makes fewer than kMinBins bins, as few as 16 while the runs are as long (32768
  // vertices, 10.0M edges, FP64: 3.10 ms a solve with 64 bins, 1.47 with 512,
  // 1.14 with 1024).  FP64
  // vectors have two sums a row in bins with rows of more than kPairRow edges, 8 to
  // 32 KB up to 2048 rows.  With 64 KB for 4096 rows too few wavefronts fit a CU
  // (RMAT-26 245 ms a solve -> 551), and with 2048 the runs are half as long (418),
  // so blocks of 4096 rows have them only where they are halved, which one with a
  // row of more than kHalveRow edges is.
  auto avg_run = [&](int shift) {
    return static_cast<double>(ng) * static_cast<double>(int64_t(1) << shift) / (static_cast<double>(nchunks) * n);
  };
  int bshift = 9;
  while (bshift < 12 && avg_run(bshift) < kAvgRun) ++bshift;
  while (bshift > 4 && (n >> bshift) < kMinBins && avg_run(bshift - 1) >= kAvgRun) --bshift;
  const int64_t nblocks = (n + (int64_t(1) << bshift) - 1) >> bshift;
  uint2* bedges = reinterpret_cast<uint2*>(take(nblocks * 8));
  block_edges_kernel<<<grid(nblocks * kWave), kB, 0, s>>>(rowoff, n, bshift, nblocks, bedges);
  GX_LAUNCHED("bs::block_edges_kernel");
  std::vector<uint2> hedges(nblocks);
  std::vector<uint32_t> hbin(nblocks), brows;
  std::vector<uint8_t> hshift(nblocks);
  read_bytes(g, hedges.data(), bedges, nblocks * 8);
  const bool f64 = shift == Shape<double>::kShift;
  const int lds_sums = f64 && bshift < 12 ? 2 << bshift : 1 << bshift;
  std::vector<uint32_t> brow;
  // A block is halved until its groups (at most its edges, and a row's at most
  // the chunks) are within three times the average or 16 rows are left.
  const double most = 3.0 * std::max(1.0, static_cast<double>(ng) / static_cast<double>(nblocks));
  for (int64_t b = 0; b < nblocks; ++b) {
    int sh = bshift;
    double w = std::min<double>(hedges[b].x, static_cast<double>(nchunks) * (int64_t(1) << bshift));
    while (sh > 4 && (w > most || (f64 && hedges[b].y > kHalveRow && (2 << sh) > lds_sums))) {
      w /= 2;
      --sh;
    }
    hbin[b] = static_cast<uint32_t>(brow.size());
    hshift[b] = static_cast<uint8_t>(sh);
    const int64_t r0 = b << bshift, r1 = std::min<int64_t>(n, (b + 1) << bshift);
    const uint32_t pair = f64 && hedges[b].y > kPairRow && (2 << sh) <= lds_sums ? kPair : 0u;
    for (int64_t r = r0; r < r1; r += int64_t(1) << sh) {
      brow.push_back(static_cast<uint32_t>(r));
      brows.push_back(static_cast<uint32_t>(std::min<int64_t>(r1 - r, int64_t(1) << sh)) | pair);
    }
  }
  L.nbins = static_cast<int64_t>(brow.size());
  brow.push_back(static_cast<uint32_t>(n));
  L.lds_sums = lds_sums;
  uint32_t* drow = reinterpret_cast<uint32_t*>(take(brow.size() * 4));
  uint32_t* dbin = reinterpret_cast<uint32_t*>(take(nblocks * 4));
  uint8_t* dshift = reinterpret_cast<uint8_t*>(take(nblocks));
  GX_HIP(hipMemcpyAsync(drow, brow.data(), brow.size() * 4, hipMemcpyHostToDevice, s));
  GX_HIP(hipMemcpyAsync(dbin, hbin.data(), nblocks * 4, hipMemcpyHostToDevice, s));
  GX_HIP(hipMemcpyAsync(dshift, hshift.data(), nblocks, hipMemcpyHostToDevice, s));
  const Bins B{dbin, dshift, bshift};
  // 5. Runs, first as they lie, then cut.
  uint32_t* pos = reinterpret_cast<uint32_t*>(wa);  // ng + 1
  uint32_t* cut = pos + ng + 1;                       // ng + 1
  uint32_t* rg0 = reinterpret_cast<uint32_t*>(we);
  run_flag_kernel<<<grid(ng + int64_t(1)), kB, 0, s>>>(grow, ng, B, pos);
  GX_LAUNCHED("bs::run_flag_kernel");
  exclusive_scan_u32(pos, pos, ng + int64_t(1), s, tmp);
  run_first_kernel<<<grid(ng), kB, 0, s>>>(pos, ng, rg0);
  run_cut_kernel<<<grid(ng + int64_t(1)), kB, 0, s>>>(pos, rg0, ng, cut);
  GX_LAUNCHED("bs::run_cut_kernel");
  exclusive_scan_u32(cut, cut, ng + int64_t(1), s, tmp);
  uint32_t nr = 0;
  read_bytes(g, &nr, cut + ng, 4);
  L.nruns = nr;
  uint64_t* rkey = reinterpret_cast<uint64_t*>(wb);
  L.groups.ensure(up(static_cast<size_t>(nr) * sizeof(uint2)) + up(L.nbins * sizeof(Bin)) +
                  up(static_cast<size_t>(ng) * 2));
  P = view();
  uint32_t* boff = reinterpret_cast<uint32_t*>(take((L.nbins + 1) * 4));
  run_key_kernel<<<grid(ng), kB, 0, s>>>(grow, ng, B, cut, drow, rkey, rg0,
                                      const_cast<uint16_t*>(P.row16));
  GX_LAUNCHED("bs::run_key_kernel");
  const uint64_t* rsorted = radix_sort_pair_u64(rkey, reinterpret_cast<uint64_t*>(wd), nr, bits_for(L.nbins), s, tmp);
  bounds_kernel<<<grid(L.nbins + 1), kB, 0, s>>>(rsorted, nr, L.nbins, boff);
  run_table_kernel<<<grid(nr), kB, 0, s>>>(rsorted, rg0, nr, ng, const_cast<uint2*>(P.runs));
  GX_LAUNCHED("bs::run_table_kernel");
  std::vector<uint32_t> hoffs(L.nbins + 1);
  read_bytes(g, hoffs.data(), boff, hoffs.size() * 4);
  std::vector<Bin> bins(L.nbins);
  for (int64_t b = 0; b < L.nbins; ++b) bins[b] = Bin{brow[b], brows[b], hoffs[b], hoffs[b + 1]};
  std::stable_sort(bins.begin(), bins.end(), [](const Bin& a, const Bin& b) { return a.run1 - a.run0 > b.run1 - b.run0; });
  GX_HIP(hipMemcpyAsync(const_cast<Bin*>(P.bins), bins.data(), bins.size() * sizeof(Bin), hipMemcpyHostToDevice, s));
  GX_HIP(hipStreamSynchronize(s));  // the host tables above are read by then
  L.shift = shift;
  L.ready = true;
  return view();
}

}  // namespace bs
}  // namespace gx
