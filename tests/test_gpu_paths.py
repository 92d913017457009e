"""Kernel and dispatch edges on the GPU: sizes at tile and size-rule borders,
adjacency orders other than ascending, against the oracle (whole numbers are
compared for equality)."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def u32(t):
    return t.cpu().numpy().view(np.uint32)


def random_csr(n, m, seed, symmetric=True, order="ascending", shuffle_hubs=False):
    """CSR of about m random edges (both directions when symmetric), adjacency
    lists ascending, descending or in random order."""
    rng = np.random.default_rng(seed)
    u = rng.integers(0, n, m)
    v = rng.integers(0, n, m)
    if shuffle_hubs:  # a few vertices meet a large share of the edges
        hubs = rng.integers(0, n, 4)
        k = m // 3
        u[:k] = hubs[rng.integers(0, 4, k)]
    keep = u != v
    u, v = u[keep], v[keep]
    if symmetric:
        u, v = np.concatenate([u, v]), np.concatenate([v, u])
    key = np.unique(u.astype(np.int64) * n + v)
    u, v = key // n, key % n
    if order == "descending":
        o = np.lexsort((-v, u))
    elif order == "random":
        o = np.lexsort((rng.random(len(u)), u))
    else:
        o = np.arange(len(u))
    u, v = u[o], v[o]
    row = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(u, minlength=n), out=row[1:])
    return row, v.astype(np.int32)


@pytest.mark.parametrize("n,m,order", [(1, 0, "ascending"), (2, 1, "ascending"), (63, 40, "descending"),
                                       (1000, 700, "random"), (1025, 400, "descending"), (70001, 69000, "random"),
                                       (70001, 700000, "descending"), (300007, 150000, "ascending")])
def test_cc_orders_and_components(gx, oracle, n, m, order):
    """Minimum labels whatever neighbours come first: the first two decide the
    sampled links, and with many components the rest is hooked afterwards."""
    row, col = random_csr(n, m, n + m, order=order, shuffle_hubs=n > 10000)
    print(f"cc n={n} m={len(col)} {order}", flush=True)
    G = gx.Graph.from_csr(row, col, symmetric=True)
    exp = oracle.cc(row, col)
    for _ in range(3):  # scratch of an earlier call
        assert np.array_equal(u32(gx.connected_components(G)[0]), exp)


def weighted_csr(n, m, seed, hub_rows=0):
    """Directed CSR with float32 weights; the first hub_rows rows hold half of
    the edges, so that rows span several tiles and chunks of tiles."""
    rng = np.random.default_rng(seed)
    u = rng.integers(0, n, m)
    if hub_rows:
        u[:m // 2] = rng.integers(0, hub_rows, m // 2)
    v = rng.integers(0, n, m)
    key = np.unique(u.astype(np.int64) * n + v)
    u, v = key // n, key % n
    row = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(u, minlength=n), out=row[1:])
    w = rng.lognormal(size=len(u)).astype(np.float32)
    return row, v.astype(np.int32), w


def weighted_reference(row, col, w, t, c, alpha=0.85, tol=1e-15, iters=300):
    """Forward vector, weight gradients and teleport gradients in FP64 (numpy
    sums pairwise: the oracle adds 200,000 dangling terms one after another,
    which alone is 1.2e-12 off)."""
    import scipy.sparse as sp
    n = len(row) - 1
    A = sp.csr_matrix((w.astype(np.float64), col, row), shape=(n, n))
    s = np.asarray(A.sum(1)).ravel()
    none = s == 0
    inv = np.divide(1.0, s, out=np.zeros(n), where=~none)
    At = sp.csr_matrix(A.T)

    def fixed_point(step, x):
        for _ in range(iters):
            new = step(x)
            done = np.abs(new - x).sum() < tol
            x = new
            if done:
                break
        return x

    t, c = t.astype(np.float64), c.astype(np.float64)
    x = fixed_point(lambda x: alpha * (At @ (x * inv) + x[none].sum() / n) + (1 - alpha) * t, np.full(n, 1.0 / n))
    below = lambda lam: (A @ lam) * inv + none * (lam.sum() / n)  # noqa: E731
    lam = fixed_point(lambda v: c + alpha * below(v), c)
    src = np.repeat(np.arange(n), np.diff(row))
    # The terms whose difference a weight's gradient is, for its error's scale.
    terms = (alpha * np.abs(x[src]) * np.abs(lam).max() * inv[src]).max()
    return x, alpha * x[src] * (lam[col] - below(lam)[src]) * inv[src], (1 - alpha) * lam, terms


# (vertices, edges drawn, hub rows): one edge; one tile less one, full and plus
# one edge; rows over several tiles; one row over every chunk; mostly empty rows.
SWEEPS = [(2, 1, 0), (600, 511, 0), (600, 513, 0), (5000, 20000, 3), (3000, 9000, 1), (200003, 60000, 2),
          (40001, 700000, 1)]


# The blocked sums' side of the size rule: few chunks and many, rows with edges in
# every chunk and over many of a wavefront's ranges, mostly empty rows, a last
# chunk of one vertex.
BLOCKS = [(32768, 2300000, 0), (65537, 2600000, 2), (1 << 20, 2200000, 1), (300001, 5000000, 3)]


@pytest.mark.parametrize("n,m,hubs", SWEEPS + BLOCKS)
def test_row_sweep_shapes(gx, n, m, hubs):
    """Weighted forward and adjoint in FP64 (FP64 sums of FP64 products: 1e-12
    relative to the largest value) and FP32 (1e-5 of it: 40-odd iterations of
    FP32 rounding) over shapes at the edges of tiles and chunks.  A weight's
    gradient is a difference (lambda_v - (P lambda)_u) scaled by x_u / s_u, zero
    for the only edge of a row: its errors are relative to the terms."""
    import torch
    row, col, w = weighted_csr(n, m, n + m, hubs)
    rng = np.random.default_rng(1)
    t = rng.random(n).astype(np.float32)
    t /= t.sum()
    c = (rng.standard_normal(n) / n).astype(np.float32)
    print(f"row sweep n={n} m={len(col)}", flush=True)
    G = gx.Graph.from_csr(row, col, w)
    tt, cc, ww = torch.from_numpy(t).cuda(), torch.from_numpy(c).cuda(), torch.from_numpy(w).cuda()
    x_ref, gw_ref, gt_ref, terms = weighted_reference(row, col, w, t, c)
    for prec, rel in (("fp64", 1e-12), ("fp32", 1e-5)):
        x, _ = gx.pagerank_weighted(G, ww, tt, tol=1e-15, max_iter=300, precision=prec)
        gw, gt, _ = gx.pagerank_adjoint(G, ww, x, cc, tol=1e-15, max_iter=300, precision=prec)
        for got, ref, scale in ((x, x_ref, np.abs(x_ref).max()), (gw, gw_ref, terms), (gt, gt_ref, np.abs(gt_ref).max())):
            got = got.cpu().numpy().astype(np.float64)
            assert np.abs(got - ref).max() <= rel * scale, (prec, np.abs(got - ref).max(), scale)


def star_csr(degrees, n, seed):
    """Symmetric weighted CSR: vertex i joined to `degrees[i]` others, and a path
    through every vertex."""
    rng = np.random.default_rng(seed)
    u = [np.full(d, i) for i, d in enumerate(degrees)] + [np.arange(n - 1)]
    v = [rng.choice(n, d, replace=False) for d in degrees] + [np.arange(1, n)]
    u, v = np.concatenate(u), np.concatenate(v)
    keep = u != v
    u, v = u[keep], v[keep]
    lo, hi = np.minimum(u, v), np.maximum(u, v)
    key = np.unique(lo.astype(np.int64) * n + hi)
    lo, hi = key // n, key % n
    w = rng.integers(1, 60, len(lo)).astype(np.uint32)
    u, v, w = np.concatenate([lo, hi]), np.concatenate([hi, lo]), np.concatenate([w, w])
    o = np.lexsort((v, u))
    row = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(u, minlength=n), out=row[1:])
    return row, v[o].astype(np.int32), w[o]


# Degrees around the hub threshold (128) and the edges a step of the hub pass and
# of a workgroup take (1024, 4096); frontiers from one vertex to more than every
# workgroup of a launch takes at once.
@pytest.mark.parametrize("n,degrees", [(2, []), (130, [127, 128, 129]), (5000, [128, 129, 1023, 1024, 1025, 4096, 4097]),
                                       (70001, [1, 1024, 60000] + [129] * 300), (600011, [200000] * 3 + [130] * 2000)])
def test_frontier_shapes(gx, oracle, n, degrees):
    row, col, w = star_csr(degrees, n, n)
    G = gx.Graph.from_csr(row, col, w, symmetric=True)
    for src in {0, n // 2, n - 1}:
        print(f"frontier n={n} m={len(col)} src={src}", flush=True)
        lv, dist = oracle.bfs(row, col, src), oracle.sssp(row, col, w, src, 4)
        assert np.array_equal(u32(gx.bfs(G, src)[0]), lv)
        assert np.array_equal(u32(gx.bfs_do(G, src)[0]), lv)
        for refine in (0, 1):
            gx.tune_set("sssp.hub_refine", refine)
            try:
                assert np.array_equal(u32(gx.sssp(G, src, 4)[0]), dist), refine
            finally:
                gx.tune_set("sssp.hub_refine", -1)
    for k in (2, 3, 129):
        deg, alive, count, _ = gx.kcore(G, k)
        exp = oracle.kcore(row, col, k)
        assert np.array_equal(u32(deg), exp) and count == int((exp >= k).sum())
        assert np.array_equal(alive.cpu().numpy(), (exp >= k).astype(np.uint8))


@pytest.mark.parametrize("n,m,hubs,sources", [(3000, 4000, 0, 3), (3000, 30000, 2, 64), (20011, 60000, 1, 65)])
def test_bc_batched_leaves_and_split_rows(gx, oracle, n, m, hubs, sources):
    """Directed graphs with vertices without out-edges at every level (they are
    never finished by a backward level) and rows over several chunks.  FP64
    sums of at most n positive terms: 1e-10 relative."""
    row, col, _ = weighted_csr(n, m, n + m, hubs)
    srcs = np.random.default_rng(2).integers(0, n, sources).astype(np.uint32)
    print(f"bc n={n} m={len(col)} sources={sources}", flush=True)
    G = gx.Graph.from_csr(row, col)
    exp = oracle.bc(row, col, srcs)
    got = gx.betweenness_centrality_batched(G, srcs)[0].cpu().numpy()
    assert np.abs(got - exp).max() <= 1e-10 * max(1.0, np.abs(exp).max())


@pytest.mark.parametrize("n,degrees,sources", [(2, [], 1), (130, [127, 128], 63), (3000, [255, 256, 257, 2900], 65),
                                               (70000, [63, 64, 65, 20000, 60000], 3)])
def test_sssp_batched_chunks(gx, oracle, n, degrees, sources):
    """Rows around the chunk and the 64-edge block sizes, hubs over many
    chunks, groups with few and with all lanes, limits that leave lanes
    pending: every source's row equals the oracle's."""
    row, col, w = star_csr(degrees, n, n)
    G = gx.Graph.from_csr(row, col, w, symmetric=True)
    srcs = np.random.default_rng(n).integers(0, n, sources).astype(np.uint32)
    exp = {int(s): oracle.sssp(row, col, w, int(s), 4) for s in set(srcs.tolist())}
    for shift, width in ((4, 0), (0, 1), (31, 64)):
        print(f"sssp batched n={n} m={len(col)} sources={sources} shift={shift} width={width}", flush=True)
        gx.tune_set("sssp.batch_width", width)
        try:
            got = u32(gx.sssp_batched(G, srcs, shift)[0])
        finally:
            gx.tune_set("sssp.batch_width", -1)
        for i, s in enumerate(srcs):
            assert np.array_equal(got[i], exp[int(s)]), (i, shift)


@pytest.mark.parametrize("n,hubs,degree", [(4095, 3, 2500), (4097, 600, 300), (20000, 40, 6000), (70001, 2, 60000)])
def test_kcore_counted_hubs(gx, oracle, n, hubs, degree):
    """Degree words around a page, more listed hubs than the table holds, and
    frontiers above and below the size that counts them in LDS: the hubs
    themselves die in some of the rounds."""
    row, col, w = star_csr([degree] * hubs, n, n)
    G = gx.Graph.from_csr(row, col, w, symmetric=True)
    for k in (1, 2, 3, hubs + 2, hubs + 3, degree):
        print(f"kcore n={n} m={len(col)} k={k}", flush=True)
        exp = oracle.kcore(row, col, k)
        for relabel in (0, 1, 0):  # on the copy the first ids are the counted ones
            gx.tune_set("frontier.relabel", relabel)
            try:
                deg, alive, count, _ = gx.kcore(G, k)
            finally:
                gx.tune_set("frontier.relabel", -1)
            assert np.array_equal(u32(deg), exp) and count == int((exp >= k).sum())
            assert np.array_equal(alive.cpu().numpy(), (exp >= k).astype(np.uint8))


def two_communities(n, hub_degree, seed):
    """Symmetric CSR: a random community around a hub, a path of a few vertices
    out of it, and a star at the far end, whose centre is unreached while the
    first community's heavy levels run."""
    rng = np.random.default_rng(seed)
    a = n // 2
    u = [rng.integers(0, a, 4 * a), np.full(hub_degree, a // 3), np.arange(a - 1, a + 5), np.full(n - a - 6, a + 5)]
    v = [rng.integers(0, a, 4 * a), rng.integers(0, a, hub_degree), np.arange(a, a + 6), np.arange(a + 6, n)]
    u, v = np.concatenate(u), np.concatenate(v)
    u, v = np.concatenate([u, v]), np.concatenate([v, u])
    key = np.unique(u[u != v].astype(np.int64) * n + v[u != v])
    u, v = key // n, key % n
    row = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(u, minlength=n), out=row[1:])
    return row, v.astype(np.int32)


@pytest.mark.parametrize("n,hub_degree,symmetric", [(400, 150, True), (2011, 160, True), (20001, 5000, True),
                                                    (20001, 5000, False), (300007, 60000, True)])
@pytest.mark.parametrize("knob", [None, "bfs.visited_bitmap", "frontier.relabel"])
def test_bfs_narrow_wide_and_pulled_levels(gx, oracle, n, hub_degree, symmetric, knob):
    """Runs of small levels, wide ones and pulled ones in turn, vertex counts
    that end inside a bitmap word, unreached hubs during a pull, sources at
    either end; levels equal the oracle's, parents are one level up."""
    row, col = two_communities(n, hub_degree, n)
    G = gx.Graph.from_csr(row, col, symmetric=symmetric)
    owner = np.repeat(np.arange(n), np.diff(row))
    edges = owner.astype(np.int64) * n + col
    if knob:
        gx.tune_set(knob, 1)
    try:
        for src in (n // 6, 0, n // 2 + 2, n - 1):
            print(f"bfs n={n} m={len(col)} symmetric={symmetric} {knob} src={src}", flush=True)
            exp = oracle.bfs(row, col, src)
            for _ in range(2):
                assert np.array_equal(u32(gx.bfs(G, src)[0]), exp)
            out = gx.bfs_do(G, src, parents=True)
            lv, parent = u32(out[0]), u32(out[1])
            assert np.array_equal(lv, exp)
            reached = np.flatnonzero((exp != 0) & (exp < 1 << 30))
            p = parent[reached].astype(np.int64)
            assert np.array_equal(exp[p] + 1, exp[reached])
            assert np.isin(p * n + reached, edges).all()
            assert parent[src] == src and np.all(parent[exp > 1 << 30] == 0xffffffff)
    finally:
        if knob:
            gx.tune_set(knob, -1)


@pytest.mark.parametrize("layers,degree", [(4, 24), (8, 12), (9, 14), (9, 16)])
def test_bfs_more_wide_levels_than_the_first_replay(gx, oracle, layers, degree):
    """Layers of 1000 vertices, each with `degree` edges into the next one and
    a hub: every level is wide, on both sides of the edge count up to which the
    first replay is shorter (2^18)."""
    rng = np.random.default_rng(degree)
    width = 1000
    n = layers * width + 1
    u = np.repeat(np.arange((layers - 1) * width), degree)
    v = (u // width + 1) * width + rng.integers(0, width, len(u))
    heads = np.arange(layers - 1) * width  # each layer's hub, and the source's edges
    u = np.concatenate([u, np.repeat(heads, width), np.full(width, n - 1)])
    v = np.concatenate([v, (np.arange(layers - 1)[:, None] * width + width + np.arange(width)).ravel(), np.arange(width)])
    key = np.unique(np.concatenate([u * n + v, v * n + u]))
    row = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(key // n, minlength=n), out=row[1:])
    col = (key % n).astype(np.int32)
    print(f"bfs layers={layers} n={n} m={len(col)}", flush=True)
    for symmetric in (False, True):  # True pulls the heavy levels
        G = gx.Graph.from_csr(row, col, symmetric=symmetric)
        for src in (n - 1, 0, n // 2):
            exp = oracle.bfs(row, col, src)
            for _ in range(2):
                assert np.array_equal(u32(gx.bfs(G, src)[0]), exp)


def lattice_csr(rows, cols, whi, seed):
    """Symmetric weighted CSR of a rows x cols lattice with a few long edges."""
    rng = np.random.default_rng(seed)
    i = np.arange(rows * cols).reshape(rows, cols)
    extra = rng.integers(0, rows * cols, (2, max(1, rows * cols // 500)))
    u = np.concatenate([i[:, :-1].ravel(), i[:-1].ravel(), extra[0]])
    v = np.concatenate([i[:, 1:].ravel(), i[1:].ravel(), extra[1]])
    n = rows * cols
    lo, hi = np.minimum(u, v), np.maximum(u, v)
    key = np.unique(lo[lo != hi].astype(np.int64) * n + hi[lo != hi])
    lo, hi = key // n, key % n
    w = rng.integers(1, whi + 1, len(lo)).astype(np.uint32)
    u, v, w = np.concatenate([lo, hi]), np.concatenate([hi, lo]), np.concatenate([w, w])
    o = np.lexsort((v, u))
    row = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(u, minlength=n), out=row[1:])
    return row, v[o].astype(np.int32), w[o]


@pytest.mark.parametrize("rows,cols,whi,shift", [(1, 2, 1, 0), (3, 5, 7, 4), (64, 1000, 1000, 6), (700, 701, 60000, 6),
                                                 (300, 1000, 1, 13)])
def test_sssp_local_rounds(gx, oracle, rows, cols, whi, shift):
    """Steps with local rounds: one item to more than a batch per workgroup
    lists, phases of one bucket to all of them, near lists that overflow (unit
    weights in one bucket)."""
    row, col, w = lattice_csr(rows, cols, whi, rows)
    G = gx.Graph.from_csr(row, col, w, symmetric=True)
    for src in {0, rows * cols // 2, rows * cols - 1}:
        print(f"sssp {rows}x{cols} whi={whi} shift={shift} src={src}", flush=True)
        exp = oracle.sssp(row, col, w, src, shift)
        for merge in (1, 1024, -1):
            gx.tune_set("sssp.max_merge", merge)
            try:
                assert np.array_equal(u32(gx.sssp(G, src, shift)[0]), exp), merge
            finally:
                gx.tune_set("sssp.max_merge", -1)


@pytest.mark.parametrize("n,degrees", [(3000, [129, 1000, 2500]), (40000, [200] * 300), (40000, [30000, 128, 129])])
def test_sssp_local_rounds_with_hubs(gx, oracle, n, degrees):
    """Hubs met in local rounds wait for the next step."""
    row, col, w = star_csr(degrees, n, n + 1)
    G = gx.Graph.from_csr(row, col, w, symmetric=True)
    for src in (0, n - 1):
        for shift in (0, 4, 31):
            print(f"sssp n={n} m={len(col)} shift={shift} src={src}", flush=True)
            assert np.array_equal(u32(gx.sssp(G, src, shift)[0]), oracle.sssp(row, col, w, src, 4))


@pytest.mark.parametrize("n,m,hubs", [(900, 5000, 0), (40000, 300000, 3), (16384, 2200000, 0), (120011, 2600000, 2)])
def test_pagerank_fp32_sweep_choice(gx, n, m, hubs):
    """Below 2^21 edges the default FP32 solve is the pull, from there on the
    blocked sweep in fine slices; a set knob is obeyed.  Both sum in 64 bits and
    round a row once per iteration: 2e-6 relative to the FP64 solve."""
    row, col, _ = weighted_csr(n, m, n, hubs)
    print(f"pagerank fp32 n={n} m={len(col)} hubs={hubs}", flush=True)
    exp = gx.pagerank(gx.Graph.from_csr(row, col), tol=1e-12, max_iter=60, precision="fp64")[0].cpu().numpy()
    got, tasks = {}, {}
    for blocking, edges in ((-1, -1), (0, -1), (1, -1), (1, 1 << 30)):
        gx.tune_set("pr.blocking", blocking)
        gx.tune_set("pr.task_edges", edges)
        try:
            G = gx.Graph.from_csr(row, col)
            x = gx.pagerank(G, tol=0.0, max_iter=60, precision="fp32")[0].cpu().numpy()
        finally:
            gx.tune_set("pr.blocking", -1)
            gx.tune_set("pr.task_edges", -1)
        np.testing.assert_allclose(x, exp, rtol=2e-6)
        got[blocking, edges] = x
        tasks[blocking, edges] = gx.pagerank_layout_info(G).get("tasks", 0)
    blocked = len(col) >= 1 << 21
    assert tasks[-1, -1] == (tasks[1, -1] if blocked else 0) and tasks[0, -1] == 0
    assert np.array_equal(got[-1, -1], got[1 if blocked else 0, -1])
    assert np.array_equal(got[1, -1], got[1, 1 << 30])  # exact sums: slices do not matter
    assert tasks[1, 1 << 30] == -(-n // 16384) and tasks[1, -1] >= min(len(col) // (2 << 13), 64)
