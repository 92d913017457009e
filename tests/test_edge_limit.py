"""Edge ids are int32 and a graph may hold up to 2^31 - 1 edges, so that the
last lists end where an id plus a wavefront's lanes no longer fits.  The loops
that walk such a list (the pulled BFS levels, the chunks of the batched sweeps)
are restated here with the helpers they use, in a host build of the header;
no GPU."""
from __future__ import annotations

import shutil
import subprocess
import tempfile
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

SRC = r'''
#include <cstdint>
#include <cstdio>
#include <vector>
#include "gx_device.hpp"
using gx::chunk_len; using gx::list_edge;
constexpr int32_t kLast = INT32_MAX;  // one past the last edge of the largest graph

// Every edge of [begin, end) seen at least once and none outside: at most
// `again` positions more than there are edges.
struct Seen {
  int32_t begin, end;
  std::vector<int> hits;
  long bad = 0;
  Seen(int32_t b, int32_t e) : begin(b), end(e), hits(static_cast<size_t>(e - b), 0) {}
  void at(int32_t e) { if (e < begin || e >= end) ++bad; else ++hits[e - begin]; }
  bool ok() const {
    for (int h : hits) if (!h) return false;
    return bad == 0;
  }
};

int main() {
  long wrong = 0;
  for (int32_t back : {0, 1, 5, 31, 32, 63, 64, 65, 300}) {
    for (int32_t len : {1, 2, 3, 4, 5, 31, 32, 33, 63, 64, 65, 95, 96, 97, 128, 255, 256, 257, 1000}) {
      const int32_t end = kLast - back, begin = end - len;
      const uint32_t n = static_cast<uint32_t>(end - begin);
      // A lane's own neighbours, four at a time, then the wavefront's.
      Seen scan(begin, end);
      const uint32_t serial = n < 32 ? n : 32;
      for (uint32_t i = 0; i < serial; i += 4)
        for (int k = 0; k < 4; ++k) scan.at(list_edge(begin, i + k, n));
      for (uint32_t j = 32; j < n; j += 64)
        for (uint32_t lane = 0; lane < 64; ++lane) scan.at(list_edge(begin, j + lane, n));
      if (!scan.ok()) ++wrong;
      // The list cut into chunks, every chunk walked 64 edges at a time.
      for (int chunk : {64, 256, 4096}) {
        Seen walk(begin, end);
        for (int64_t x = begin; x < end; x += chunk) {
          const int32_t b = static_cast<int32_t>(x);
          const uint32_t c = chunk_len(b, end, chunk);
          if (c == 0 || c > static_cast<uint32_t>(chunk)) ++wrong;
          for (uint32_t j0 = 0; j0 < c; j0 += 64)
            for (uint32_t lane = 0; lane < 64; ++lane)
              if (j0 + lane < c) walk.at(b + static_cast<int32_t>(j0 + lane));
        }
        if (!walk.ok()) ++wrong;
        for (int h : walk.hits) if (h != 1) ++wrong;
      }
    }
  }
  // One list of every edge: the position after the last step still fits.
  const uint32_t all = static_cast<uint32_t>(kLast);
  const uint32_t last_step = 32 + (all - 33) / 64 * 64;
  if (last_step + 64 < last_step || list_edge(0, last_step + 63, all) != kLast - 1) ++wrong;
  if (chunk_len(0, kLast, 4096) != 4096u || chunk_len(kLast - 1, kLast, 256) != 1u) ++wrong;
  std::printf("%ld\n", wrong);
  return 0;
}
'''


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc not available")
def test_lists_at_the_edge_limit_are_walked_inside_their_bounds():
    with tempfile.TemporaryDirectory() as td:
        src, exe = Path(td) / "limit.hip", Path(td) / "limit"
        src.write_text(SRC)
        subprocess.run([HIPCC, "-O1", "-std=c++17", "-w", "--offload-arch=gfx950", "-Xclang", "-target-feature",
                        "-Xclang", "-packed-fp32-ops", "-I", str(ROOT / "include"), "-I",
                        str(ROOT / "galois_amd" / "csrc"), str(src), "-o", str(exe)],
                       check=True, capture_output=True, timeout=300)
        out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120, check=True).stdout.split()
    assert out == ["0"], out
