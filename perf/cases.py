"""Timed cases of the lonestar analytics on one GPU: what a program that holds a
graph in device memory asks of it, from a call on four thousand vertices, where
launches and waits are all there is, to a PageRank solve on RMAT-26.

Graphs are made here with torch on the GPU from the seed alone and handed over
with `Graph.from_device`, as a program with its own data does: RMAT graphs
(a/b/c/d = .57/.19/.19/.05, self-loops and duplicate edges removed) of any
vertex count, with the generator's ids (small ids are the hubs) or shuffled
ones, road-like lattices, and disjoint unions of uneven graphs.  A case's
`kind` is the entry point it calls.

  bfs           level-synchronous BFS, levels
  bfs_do        direction-optimising BFS, levels
  sssp          delta-stepping, uint32 weights, distances
  sssp_batched  distances from up to 64 sources in one call
  cc            minimum labels of the connected components
  kcore         degrees, membership and size of the k-core
  pagerank      normalised PageRank, FP32 or FP64
  adjoint       differentiable PageRank through torch.autograd: forward, then
                the gradients of the edge weights and of the teleport vector
  bc            betweenness centrality, sources batched 64 to a wavefront
"""
from __future__ import annotations

import math

import numpy as np
import torch

import galois_amd as gx

A, B, C = 0.57, 0.19, 0.19
CHUNK = 1 << 26  # edges drawn at a time: bounds the generator's memory

# The analytics take a source vertex, a core size or a tolerance; the sizes are
# those of this repository's benchmark and tests, or ragged ones near them.
LISTED = [
    # A query on a small graph, one of thousands in a service: nothing but latency.
    dict(name="bfs_4k", kind="bfs", graph="rmat", n=4096, ef=16, symmetric=True, shuffled=False),
    # The benchmark's first workload: a graph that fits in the caches.
    dict(name="bfs_rmat18", kind="bfs", graph="rmat", n=1 << 18, ef=16, symmetric=True, shuffled=False),
    # Hop counts on a large social graph whose ids say nothing of the degrees.
    dict(name="bfs_do_rmat24", kind="bfs_do", graph="rmat", n=1 << 24, ef=16, symmetric=True, shuffled=True),
    # Shortest paths on a power-law graph and on a road network: the two ends
    # of delta-stepping, few wide steps and many narrow ones.
    dict(name="sssp_rmat22", kind="sssp", graph="rmat", n=1 << 22, ef=16, symmetric=True, shuffled=False, wlo=1,
         whi=255, shift=6),
    dict(name="sssp_grid2048", kind="sssp", graph="grid", n=2048 * 2048, symmetric=True, wlo=1, whi=1000, shift=6),
    # Distances from a set of landmarks, one call for all of them.
    dict(name="sssp_batched_rmat20", kind="sssp_batched", graph="rmat", n=1 << 20, ef=16, symmetric=True,
         shuffled=False, wlo=1, whi=255, shift=6, sources=64),
    # Clustering and pruning of a graph read from a file: an odd vertex count.
    dict(name="cc_3m", kind="cc", graph="rmat", n=3000001, ef=16, symmetric=True, shuffled=True),
    dict(name="kcore_rmat22", kind="kcore", graph="rmat", n=1 << 22, ef=16, symmetric=True, shuffled=False, k=10),
    # Ranking: the headline solve, and a smaller one in FP64.
    dict(name="pagerank_rmat26", kind="pagerank", graph="rmat", n=1 << 26, ef=16, symmetric=False, shuffled=False,
         precision="fp32"),
    dict(name="pagerank_f64_1500k", kind="pagerank", graph="rmat", n=1500007, ef=16, symmetric=False, shuffled=True,
         precision="fp64"),
    # A training step that learns edge weights through the ranks.
    dict(name="adjoint_rmat22", kind="adjoint", graph="rmat", n=1 << 22, ef=16, symmetric=False, shuffled=False,
         precision="fp32"),
    # Centrality estimated from a batch of sampled sources.
    dict(name="bc_rmat20", kind="bc", graph="rmat", n=1 << 20, ef=16, symmetric=True, shuffled=False, parts=1,
         sources=64),
]

# Vertex counts that draw() spans, per kind (over the logarithm).
RANGE = {"bfs": (1 << 10, 1 << 22), "bfs_do": (1 << 12, 1 << 24), "sssp": (1 << 10, 1 << 22),
         "sssp_batched": (1 << 10, 1 << 20), "cc": (1 << 10, 1 << 23), "kcore": (1 << 10, 1 << 22),
         "pagerank": (1 << 10, 1 << 24), "adjoint": (1 << 10, 1 << 21), "bc": (1 << 10, 1 << 19)}


def listed():
    return [dict(c) for c in LISTED]


def draw(rng):
    kind = rng.choice(sorted(RANGE))
    lo, hi = RANGE[kind]
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    c = dict(kind=kind, graph="rmat", n=n, ef=rng.randint(6, 24), symmetric=True, shuffled=rng.random() < 0.5)
    if kind in ("bfs", "bfs_do", "sssp", "cc") and rng.random() < 0.35:
        c["graph"] = "grid"
        del c["ef"], c["shuffled"]
    elif kind in ("bfs", "bfs_do", "sssp", "pagerank", "adjoint", "sssp_batched"):
        c["symmetric"] = kind not in ("pagerank", "adjoint") and rng.random() < 0.7
    if kind in ("sssp", "sssp_batched"):
        c.update(wlo=1, whi=rng.choice([1, 20, 255, 1000, 60000]), shift=rng.choice([4, 6, 8, 13]))
    if kind in ("sssp_batched", "bc"):
        c["sources"] = rng.choice([1, 7, 33, 64])
    if kind == "bc":
        c["parts"] = rng.choice([1, 1, 3, 16])
    if kind == "kcore":
        c["k"] = rng.randint(2, 40)
    if kind in ("pagerank", "adjoint"):
        c["precision"] = rng.choice(["fp32", "fp64"])
    return c


# ------------------------------------------------------------------- graphs
def _rmat_keys(n, edges, gen):
    """u * n + v of `edges` RMAT edges (fewer: those outside a ragged n are left out)."""
    levels = max(1, (n - 1).bit_length())
    out = []
    for first in range(0, edges, CHUNK):
        k = min(CHUNK, edges - first)
        u = torch.zeros(k, dtype=torch.int32, device="cuda")
        v = torch.zeros(k, dtype=torch.int32, device="cuda")
        for _ in range(levels):
            r = torch.rand(k, generator=gen, device="cuda")
            hi = r >= A + B
            u.mul_(2).add_(hi)
            v.mul_(2).add_(((r >= A) & ~hi) | (r >= A + B + C))
        keep = u != v
        if n & (n - 1):
            keep &= (u < n) & (v < n)
        out.append((u[keep], v[keep]))
    return out


def _csr(keys, n):
    """CSR (int32 row, int32 col) of the distinct ascending keys u * n + v."""
    row = torch.searchsorted(keys, torch.arange(n + 1, device="cuda", dtype=torch.int64) * n).to(torch.int32)
    return row, torch.remainder(keys, n).to(torch.int32)


def _distinct(parts):
    keys = torch.cat(parts) if len(parts) > 1 else parts[0]
    parts.clear()
    return torch.unique(keys)


def _rmat(n, ef, symmetric, shuffled, gen, count=0):
    """CSR of an RMAT graph; count > 0: of so many of its edges, chosen at random."""
    perm = torch.randperm(n, generator=gen, device="cuda") if shuffled else None
    keys = []
    for u, v in _rmat_keys(n, ef * n, gen):
        u, v = (perm[u], perm[v]) if shuffled else (u.to(torch.int64), v.to(torch.int64))
        keys.append(u * n + v)
        if symmetric:
            keys.append(v * n + u)
    keys = _distinct(keys)
    if 0 < count < keys.numel():
        keys = keys[torch.randperm(keys.numel(), generator=gen, device="cuda")[:count].sort()[0]]
    return _csr(keys, n)


def _grid(n, gen):
    """Lattice of about n vertices, 5% of its edges dropped, 1% random shortcuts."""
    side = max(2, math.isqrt(n))
    n = side * side
    ids = torch.arange(n, device="cuda", dtype=torch.int64).view(side, side)
    u = torch.cat([ids[:, :-1].reshape(-1), ids[:-1, :].reshape(-1)])
    v = torch.cat([ids[:, 1:].reshape(-1), ids[1:, :].reshape(-1)])
    keep = torch.rand(u.numel(), generator=gen, device="cuda") >= 0.05
    extra = torch.randint(n, (2, max(1, u.numel() // 100)), generator=gen, device="cuda")
    extra = extra[:, extra[0] != extra[1]]
    u, v = torch.cat([u[keep], extra[0]]), torch.cat([v[keep], extra[1]])
    return n, *_csr(_distinct([u * n + v, v * n + u]), n)


def _graph(case, gen):
    """(row, col) on the GPU, and the first vertex of each part and the end."""
    n = case["n"]
    if case["graph"] == "grid":
        n, row, col = _grid(n, gen)
        return row, col, [0, n]
    parts = case.get("parts", 1)
    if case["kind"] == "adjoint":  # a fixed number of weights: more edges are drawn than are kept
        more = 4.0 if n < 1 << 16 else 2.5
        row, col = _rmat(n, math.ceil(more * case["ef"]), case["symmetric"], case["shuffled"], gen, case["ef"] * n)
        return row, col, [0, n]
    if parts == 1:
        row, col = _rmat(n, case["ef"], case["symmetric"], case["shuffled"], gen)
        return row, col, [0, n]
    # Uneven parts: geometric sizes that add up to n.
    share = np.exp(np.linspace(0.0, 3.0, parts))
    sizes = [max(8, int(n * s / share.sum())) for s in share]
    rows, cols, first, edges = [torch.zeros(1, dtype=torch.int32, device="cuda")], [], [0], 0
    for s in sizes:
        r, c = _rmat(s, case["ef"], case["symmetric"], case["shuffled"], gen)
        rows.append(r[1:] + edges)
        cols.append(c + first[-1])
        first.append(first[-1] + s)
        edges += c.numel()
    return torch.cat(rows), torch.cat(cols), first


def _sources_of_edges(row, col):
    return torch.repeat_interleave(torch.arange(row.numel() - 1, device="cuda"), (row[1:] - row[:-1]).to(torch.int64))


def _pair_weights(row, col, lo, hi):
    """The same weight in [lo, hi] for both directions of an edge."""
    u, v = _sources_of_edges(row, col), col.to(torch.int64)
    h = torch.minimum(u, v) * 0x9E3779B97F4A7C1 + torch.maximum(u, v) * 0x85EBCA77C2B2AE3
    h = (h ^ (h >> 29)) * 0xBF58476D1CE4E5
    h = (h ^ (h >> 32)) & 0x7FFFFFFF
    return (h % (hi - lo + 1) + lo).to(torch.int32)


def _pick(col, count, gen, lo=0, hi=None):
    """Vertices that have edges, the busier the likelier, as host integers."""
    at = torch.randint(lo, col.numel() if hi is None else hi, (count,), generator=gen, device="cuda")
    return col[at].cpu().numpy().astype(np.uint32)


def _inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    row, col, first = _graph(case, gen)
    s = {"case": case, "row": row, "col": col}
    n, m = row.numel() - 1, col.numel()
    if "whi" in case:
        s["w"] = _pair_weights(row, col, case["wlo"], case["whi"])
    if case["kind"] in ("bfs", "bfs_do", "sssp"):
        s["source"] = int(_pick(col, 1, gen)[0])
    if case["kind"] in ("sssp_batched", "bc"):
        ends = row[torch.tensor(first, device="cuda")].tolist()
        if len(first) == 2:
            s["sources"] = _pick(col, case["sources"], gen)
        else:  # a few sources in every part
            s["sources"] = np.concatenate([_pick(col, 4, gen, a, b) for a, b in zip(ends, ends[1:]) if b > a])
    if case["kind"] == "adjoint":
        s["weights"] = torch.empty(m, device="cuda").log_normal_(generator=gen).requires_grad_()
        t = torch.rand(n, generator=gen, device="cuda") + 0.5
        s["teleport"] = (t / t.sum()).requires_grad_()
        s["grad"] = torch.randn(n, generator=gen, device="cuda") / n  # of a mean over the vertices
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    s["graph"] = gx.Graph.from_device(s["row"], s["col"], s.get("w"), symmetric=case["symmetric"])
    if s["col"].numel() > 1 << 27:
        torch.cuda.empty_cache()  # the generator's buffers, many times the graph
    return s


def run(s):
    c, g = s["case"], s["graph"]
    kind = c["kind"]
    if kind == "bfs":
        return gx.bfs(g, s["source"])[0]
    if kind == "bfs_do":
        return gx.bfs_do(g, s["source"])[0]
    if kind == "sssp":
        return gx.sssp(g, s["source"], c["shift"])[0]
    if kind == "sssp_batched":
        return gx.sssp_batched(g, s["sources"], c["shift"])[0]
    if kind == "cc":
        return gx.connected_components(g)[0]
    if kind == "kcore":
        return gx.kcore(g, c["k"])[:3]
    if kind == "pagerank":
        return gx.pagerank(g, precision=c["precision"])[0]
    if kind == "bc":
        return gx.betweenness_centrality_batched(g, s["sources"])[0]
    x = gx.differentiable_pagerank(g, s["weights"], s["teleport"], precision=c["precision"])
    gw, gt = torch.autograd.grad(x, (s["weights"], s["teleport"]), s["grad"].to(x.dtype))
    return x.detach(), gw, gt


def work(case):
    """Bytes: the graph's arrays and the caller's read once and the results
    written once; the solves that iterate read the graph again in every
    iteration (it does not fit in a cache), each wavefront's worth of sources
    likewise once.  About 0.9 of the edges drawn remain after duplicates (all of
    the adjoint's are kept)."""
    n, kind = case["n"], case["kind"]
    m = 4 * n if case["graph"] == "grid" else int(0.9 * case["ef"] * n) * (2 if case["symmetric"] else 1)
    graph = 4 * m + 4 * n
    k = case.get("sources", 1)
    if kind in ("bfs", "bfs_do", "cc"):
        return {"bytes": graph + 4 * n, "flops": 0}
    if kind == "sssp":
        return {"bytes": graph + 4 * m + 4 * n, "flops": 0}
    if kind == "sssp_batched":
        return {"bytes": graph + 4 * m + 4 * n * k, "flops": 0}
    if kind == "kcore":
        return {"bytes": graph + 5 * n, "flops": 0}
    real = 8 if case.get("precision") == "fp64" else 4
    if kind == "pagerank":
        it = 31
        return {"bytes": it * (graph + 3 * real * n), "flops": it * 2 * m}
    if kind == "adjoint":
        m = case["ef"] * n
        it = 60  # both solves
        return {"bytes": it * (graph + 4 * m + 3 * real * n) + real * (m + 2 * n), "flops": it * 3 * m}
    return {"bytes": 2 * graph + (12 * k + 8) * n, "flops": 2 * m * k}


# ------------------------------------------------- the same in 64 bits, in torch
def _matrix(row, col, val):
    n = row.numel() - 1
    return torch.sparse_csr_tensor(row, col, val, size=(n, n), check_invariants=False)


def _transposed(row, col, val):
    """The same entries by column (val: one per entry)."""
    n = row.numel() - 1
    order = torch.argsort(col, stable=True)
    src = _sources_of_edges(row, col)[order].to(torch.int32)
    return _matrix(torch.searchsorted(col[order], torch.arange(n + 1, device="cuda", dtype=torch.int32)).to(torch.int32),
                   src, val[order])


def _fixed_point(step, x, tol, iters):
    for _ in range(iters):
        new = step(x)
        done = float((new - x).abs().sum()) < tol
        x = new
        if done:
            break
    return x


def _bc64(row, col, sources):
    """Brandes over all sources at once: one column per source."""
    n, k = row.numel() - 1, len(sources)
    ones = torch.ones(col.numel(), dtype=torch.float64, device="cuda")
    out, into = _matrix(row, col, ones), _transposed(row, col, ones)
    level = torch.full((n, k), -1, dtype=torch.int16, device="cuda")
    sigma = torch.zeros((n, k), dtype=torch.float64, device="cuda")
    at = torch.tensor(sources.astype(np.int64), device="cuda"), torch.arange(k, device="cuda")
    level[at], sigma[at] = 0, 1.0
    depth = 0
    while True:
        paths = into @ (sigma * (level == depth))
        new = (level < 0) & (paths > 0)
        if not bool(new.any()):
            break
        depth += 1
        level[new] = depth
        sigma += paths * new
    delta = torch.zeros_like(sigma)
    for d in range(depth - 1, 0, -1):
        below = torch.where(level == d + 1, (1 + delta) / sigma, 0.0)
        delta += sigma * (out @ below) * (level == d)
    return delta.sum(1)


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("pagerank", "adjoint", "bc"):
        return None  # whole numbers
    s = _inputs(case, seed)
    row, col, n, m = s["row"], s["col"], s["row"].numel() - 1, s["col"].numel()
    if kind == "bc":
        return _bc64(row, col, s["sources"]) if m * len(s["sources"]) <= 1 << 31 else None
    alpha = 0.85
    start = torch.full((n,), 1.0 / n, dtype=torch.float64, device="cuda")
    if kind == "pagerank":
        deg = (row[1:] - row[:-1]).double()
        none = deg == 0
        into = _transposed(row, col, torch.ones(m, dtype=torch.float64, device="cuda"))
        share = torch.where(none, 0.0, 1.0 / deg)
        return _fixed_point(lambda x: alpha * (into @ (x * share) + (x * none).sum() / n) + (1 - alpha) / n, start, 1e-9, 100)
    w, t, c = (s[k].detach().double() for k in ("weights", "teleport", "grad"))
    src, dst = _sources_of_edges(row, col), col.to(torch.int64)
    total = _matrix(row, col, w) @ torch.ones_like(c)
    none = total == 0
    val = w / total[src]
    P, into = _matrix(row, col, val), _transposed(row, col, val)
    x = _fixed_point(lambda x: alpha * (into @ x + (x * none).sum() / n) + (1 - alpha) * t, start, 1e-13, 300)
    below = lambda lam: P @ lam + none * (lam.sum() / n)  # noqa: E731
    lam = _fixed_point(lambda v: c + alpha * below(v), c, 1e-13, 300)
    gw = alpha * x[src] * (lam[dst] - below(lam)[src]) / total[src]
    return x, gw, (1 - alpha) * lam
