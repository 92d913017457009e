// Plan tables of the row sweep (rowsweep.hpp), built once per row-offset array
// and cached in the graph.
#include <algorithm>

#include "rowsweep.hpp"

namespace gx {
namespace rs {
namespace {

__global__ void full_flag_kernel(const int32_t* __restrict__ rowoff, int64_t n, uint32_t* __restrict__ flag) {
  for (int64_t r = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; r <= n;
       r += static_cast<int64_t>(gridDim.x) * blockDim.x)
    flag[r] = r < n && rowoff[r + 1] > rowoff[r] ? 1u : 0u;
}

// pos: rows with edges before each row (n + 1 entries).
__global__ void rid_kernel(const uint32_t* __restrict__ pos, int64_t n, uint32_t* __restrict__ rid) {
  const uint32_t full = pos[n];
  for (int64_t r = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; r < n;
       r += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const uint32_t p = pos[r];
    rid[pos[r + 1] > p ? p : full + static_cast<uint32_t>(r) - p] = static_cast<uint32_t>(r);
  }
}

// Index in rid of the row that holds edge e (e < m).
__device__ __forceinline__ uint32_t row_index(const int32_t* __restrict__ rowoff, const uint32_t* __restrict__ rid,
                                              uint32_t full, int64_t e) {
  uint32_t lo = 0, hi = full - 1;  // last row with rowoff <= e
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo + 1) / 2;
    if (rowoff[rid[mid]] <= e) lo = mid; else hi = mid - 1;
  }
  return lo;
}

__global__ void tile_row_kernel(const int32_t* __restrict__ rowoff, const uint32_t* __restrict__ rid, uint32_t full,
                                int64_t m, int64_t ntiles, uint32_t* __restrict__ tile_row) {
  for (int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t <= ntiles;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x)
    tile_row[t] = t * kTile < m ? row_index(rowoff, rid, full, t * kTile) : full;
}

__global__ void lane_info_kernel(const int32_t* __restrict__ rowoff, const uint32_t* __restrict__ rid, uint32_t full,
                                 int64_t m, int64_t ntiles, const uint32_t* __restrict__ tile_row,
                                 uint32_t* __restrict__ info) {
  for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < ntiles * kWave;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t e0 = i * kItems;
    uint32_t word = 0;
    if (e0 < m) {
      uint32_t k = row_index(rowoff, rid, full, e0);
      word = (k - tile_row[i / kWave]) << 8;
      int64_t end = rowoff[rid[k] + 1];
      for (int u = 0; u < kItems && e0 + u < m; ++u) {
        if (e0 + u + 1 != end) continue;
        word |= 1u << u;
        if (++k < full) end = rowoff[rid[k] + 1];
      }
    }
    info[i] = word;
  }
}

// Per chunk: the row that began in an earlier chunk and ends in this one
// (kNoRow: none), and the chunk it began in.
__global__ void spans_kernel(RowPlan P, uint32_t* __restrict__ row, uint32_t* __restrict__ first) {
  const int64_t chunk_edges = static_cast<int64_t>(P.kt) * kTile;
  for (int64_t c = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; c < P.nchunks;
       c += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const uint32_t r = P.rid[P.tile_row[c * P.kt]];
    const int32_t rb = P.rowoff[r], re = P.rowoff[r + 1];
    const bool spans = rb < c * chunk_edges && re <= (c + 1) * chunk_edges;
    row[c] = spans ? r : kNoRow;
    first[c] = static_cast<uint32_t>(rb / chunk_edges);
  }
}

}  // namespace

// Layout of cache.buf (words): rid[n] | tile_row[ntiles + 1] |
// lane_info[64 * ntiles] | span_row[nchunks] | span_first[nchunks].
RowPlan build_plan(gx_graph* g, const int32_t* rowoff, const int32_t* col, int64_t n, int64_t m, PullPlan& cache) {
  GX_REQUIRE(n > 0, "row sweep over an empty graph");
  const int64_t ntiles = (m + kTile - 1) / kTile;
  const int kt = tiles_per_chunk(ntiles);
  const int64_t nchunks = (ntiles + kt - 1) / kt;
  auto view = [&]() {
    RowPlan P{};
    P.rowoff = rowoff;
    P.col = col;
    P.n = n;
    P.len = m;
    P.rid = cache.buf.as<uint32_t>();
    P.full = cache.full;
    P.tile_row = P.rid + n;
    P.lane_info = P.tile_row + ntiles + 1;
    P.ntiles = ntiles;
    P.kt = kt;
    P.nchunks = nchunks;
    P.span_row = P.lane_info + ntiles * kWave;
    P.span_first = P.span_row + nchunks;
    return P;
  };
  if (cache.ready) return view();
  hipStream_t s = g->stream;
  cache.buf.ensure((n + ntiles + 1 + ntiles * kWave + 2 * nchunks) * sizeof(uint32_t));
  uint32_t* rid = cache.buf.as<uint32_t>();
  uint32_t* tile_row = rid + n;
  DevBuf pos;
  pos.ensure((n + 1) * sizeof(uint32_t));
  full_flag_kernel<<<grid_for(n + 1, kBlock, 8192), kBlock, 0, s>>>(rowoff, n, pos.as<uint32_t>());
  GX_LAUNCHED("full_flag_kernel");
  exclusive_scan_u32(pos.as<uint32_t>(), pos.as<uint32_t>(), n + 1, s);
  rid_kernel<<<grid_for(n, kBlock, 8192), kBlock, 0, s>>>(pos.as<uint32_t>(), n, rid);
  GX_LAUNCHED("rid_kernel");
  uint32_t full = 0;
  read_bytes(g, &full, pos.as<uint32_t>() + n, sizeof(full));
  cache.full = full;
  tile_row_kernel<<<grid_for(ntiles + 1, kBlock, 8192), kBlock, 0, s>>>(rowoff, rid, full, m, ntiles, tile_row);
  GX_LAUNCHED("tile_row_kernel");
  if (ntiles > 0) {
    lane_info_kernel<<<grid_for(ntiles * kWave, kBlock, 16384), kBlock, 0, s>>>(rowoff, rid, full, m, ntiles, tile_row,
                                                                                tile_row + ntiles + 1);
    GX_LAUNCHED("lane_info_kernel");
    uint32_t* span_row = tile_row + ntiles + 1 + ntiles * kWave;
    spans_kernel<<<grid_for(nchunks, kBlock, 8192), kBlock, 0, s>>>(view(), span_row, span_row + nchunks);
    GX_LAUNCHED("spans_kernel");
  }
  GX_HIP(hipStreamSynchronize(s));
  cache.ready = true;
  return view();
}

}  // namespace rs
}  // namespace gx
