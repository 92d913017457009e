"""Dispatch rules and knobs on the GPU: what a call reports about the path it
took, paths that the default rules leave to larger graphs, and inputs in orders
and of values that a path's layout could mistake."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_paths import random_csr, u32, weighted_csr
from test_gpu_paths import test_row_sweep_shapes as row_sweep_shapes

pytestmark = pytest.mark.gpu


class knobs:
    """Knobs set for a block."""

    def __init__(self, gx, **values):
        self.gx, self.values = gx, {k.replace("__", "."): v for k, v in values.items()}

    def __enter__(self):
        for k, v in self.values.items():
            self.gx.tune_set(k, v)

    def __exit__(self, *exc):
        for k in self.values:
            self.gx.tune_set(k, -1)


@pytest.mark.parametrize("n,m", [(700, 3000), (40000, 1000000), (16384, 2400000), (300000, 4000000)])
def test_layout_reports_its_slices(gx, n, m):
    """task_edges is the knob's value for the layout, slice_edges what its bins
    were cut with: as many as the knob says when it is set, m / 160 within
    [2^13, the default] otherwise.  A slice holds at most 511 edges more, and a
    bin is cut if and only if it holds more edges than a slice."""
    row, col, _ = weighted_csr(n, m, n, 1)
    m = len(col)
    print(f"layout n={n} m={m}", flush=True)
    for edges in (-1, 1 << 12, 1 << 13, 1 << 19, 1 << 30):
        G = gx.Graph.from_csr(row, col)
        with knobs(gx, pr__blocking=1, pr__task_edges=edges):
            gx.pagerank(G, tol=0.0, max_iter=1)
        info = gx.pagerank_layout_info(G)
        assert info["task_edges"] == (edges if edges > 0 else 1 << 19)
        assert info["slice_edges"] == (edges if edges > 0 else min(1 << 19, max(m // 160, 1 << 13)))
        assert info["tasks"] * (info["slice_edges"] + 511) >= m
        # A bin is 16384 destinations of the degree order.
        order = np.lexsort((np.arange(n), -np.diff(row)))
        rank = np.empty(n, np.int64)
        rank[order] = np.arange(n)
        heavy = np.bincount(rank[col] // 16384, minlength=info["bins"])
        assert info["sliced_bins"] == int((heavy > info["slice_edges"]).sum())


def hub_chain(hubs, degree, step):
    """Symmetric weighted CSR: vertex 0 joined to `hubs` hubs at distances step,
    2 * step, ...; each hub joined to `degree` leaves of its own."""
    n = 1 + hubs + hubs * degree
    hub = np.arange(1, hubs + 1)
    u = np.concatenate([np.zeros(hubs, np.int64), np.repeat(hub, degree)])
    v = np.concatenate([hub, np.arange(1 + hubs, n)])
    w = np.concatenate([step * hub, np.ones(hubs * degree, np.int64)]).astype(np.uint32)
    u, v, w = np.concatenate([u, v]), np.concatenate([v, u]), np.concatenate([w, w])
    o = np.lexsort((v, u))
    row = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(u, minlength=n), out=row[1:])
    return row, v[o].astype(np.int32), w[o]


@pytest.mark.parametrize("hubs,degree,step", [(40, 200, 1000), (60, 130, 50000)])
def test_sssp_set_slices_stay(gx, oracle, hubs, degree, step):
    """With sssp.hub_refine set, a hub step takes the pending hubs within
    2^(r - 1) of the nearest one, however few they are: hubs 1000 apart take a
    step each at r = 1, and one step at r = 32.  One bucket holds them all."""
    row, col, w = hub_chain(hubs, degree, step)
    G = gx.Graph.from_csr(row, col, w, symmetric=True)
    exp = oracle.sssp(row, col, w, 0, 31)
    steps = {}
    for r in (0, 1, 32):
        with knobs(gx, sssp__hub_refine=r):
            d, st = gx.sssp(G, 0, 31)
        assert np.array_equal(u32(d), exp)
        steps[r] = st.iterations
    print(f"sssp hubs={hubs} steps={steps}", flush=True)
    assert steps[1] >= hubs and steps[32] < 10 and steps[0] < 10


@pytest.mark.parametrize("n,m,missing", [(2000, 30000, 0), (2000, 30000, 1), (20001, 400000, 1), (20001, 400000, None)])
def test_bfs_does_not_take_the_symmetric_flag_on_trust(gx, oracle, n, m, missing):
    """Levels follow the edges as they are, also where a graph that is said to be
    symmetric lacks reverse edges (`missing` of every vertex but the last, or all
    of them): a pulled level would not see the edge that has no reverse."""
    row, col = random_csr(n, m, n, symmetric=missing is not None, shuffle_hubs=True)
    if missing:  # the last neighbour of every vertex goes
        src = np.repeat(np.arange(n), np.diff(row))
        keep = np.ones(len(col), bool)
        full = np.flatnonzero(np.diff(row) > 1)[:-1]
        keep[row[full + 1] - 1] = False
        src, col = src[keep], col[keep]
        row = np.zeros(n + 1, np.int32)
        np.cumsum(np.bincount(src, minlength=n), out=row[1:])
    for flag in (True, False):
        G = gx.Graph.from_csr(row, col, symmetric=flag)
        for src in (0, n // 3, int(np.argmax(np.diff(row)))):
            print(f"bfs n={n} m={len(col)} missing={missing} flag={flag} src={src}", flush=True)
            assert np.array_equal(u32(gx.bfs(G, src)[0]), oracle.bfs(row, col, src)), (flag, src)


def test_bfs_lists_with_repeated_edges(gx, oracle):
    """Repeated and unsorted adjacency entries: a symmetric graph whose edges come
    twice (heavy levels pulled), and one whose reverses come once."""
    n = 20001
    row, col = random_csr(n, 200000, 5, order="random", shuffle_hubs=True)
    src = np.repeat(np.arange(n), np.diff(row))
    for again in (np.ones(len(col), bool), src < col):
        u, v = np.concatenate([src, src[again]]), np.concatenate([col, col[again]])
        o = np.lexsort((np.random.default_rng(6).random(len(u)), u))
        u, v = u[o], v[o].astype(np.int32)
        r = np.zeros(n + 1, np.int32)
        np.cumsum(np.bincount(u, minlength=n), out=r[1:])
        G = gx.Graph.from_csr(r, v, symmetric=True)
        for s in (0, n - 1, int(np.argmax(np.diff(r)))):
            exp = oracle.bfs(r, v, s)
            assert np.array_equal(u32(gx.bfs(G, s)[0]), exp)
            assert np.array_equal(u32(gx.bfs_do(G, s)[0]), exp)
        assert np.array_equal(u32(gx.connected_components(G)[0]), oracle.cc(r, v))
        w = np.random.default_rng(7).integers(1, 200, len(v)).astype(np.uint32)
        W = gx.Graph.from_csr(r, v, w)
        for shift in (0, 6, 13):
            assert np.array_equal(u32(gx.sssp(W, 3, shift)[0]), oracle.sssp(r, v, w, 3, 6))
        got = u32(gx.sssp_batched(W, [3, 17], 6)[0])
        assert np.array_equal(got[0], oracle.sssp(r, v, w, 3, 6)) and np.array_equal(got[1], oracle.sssp(r, v, w, 17, 6))


def groups_of(row, col, shift, range_edges=2048):
    """(row, chunk of 2^shift sources) groups of the degree-ordered transpose, cut
    where a wavefront's range of edges ends inside a chunk."""
    n = len(row) - 1
    deg = np.diff(row)
    rank = np.empty(n, np.int64)
    rank[np.lexsort((np.arange(n), -deg))] = np.arange(n)
    u, v = rank[np.repeat(np.arange(n), deg)], rank[col]
    chunk = u >> shift
    o = np.lexsort((v, chunk))
    chunk, v = chunk[o], v[o]
    first = np.searchsorted(chunk, np.arange(chunk.max() + 2))
    at = np.arange(len(chunk)) - first[chunk]
    new = np.ones(len(chunk), bool)
    new[1:] = (chunk[1:] != chunk[:-1]) | (v[1:] != v[:-1]) | (at[1:] % range_edges == 0)
    tiles = int(sum(-(-c // 512) for c in np.diff(first)))
    return int(new.sum()), tiles


@pytest.mark.parametrize("n,m", [(600011, 9000000), (1 << 19, 8500000), (40000, 9500000)])
def test_fp64_pull_states_the_bytes_of_the_path_it_took(gx, n, m):
    """main_kernel_bytes of an FP64 sweep: blocked sums from 2^23 edges and 2^19
    vertices on (two bytes per edge position, 18 per group, eight per run of at most
    64 groups, 36 per row), the row sweep on fewer vertices and with the hot split."""
    rng = np.random.default_rng(n)
    key = np.unique(rng.integers(0, n, m) * n + np.minimum(rng.integers(0, n, m), rng.integers(0, n, m)))
    row = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(key // n, minlength=n), out=row[1:])
    col = (key % n).astype(np.int32)
    m = len(col)
    assert m >= 1 << 23
    G = gx.Graph.from_csr(row, col)
    st = gx.pagerank(G, tol=0.0, max_iter=2, precision="fp64")[1]
    groups, tiles = groups_of(row, col, 13)
    fixed = 2 * 512 * tiles + 18 * groups + 36 * n
    print(f"bytes n={n} m={m} groups={groups} fixed={fixed} stated={st.main_kernel_bytes}", flush=True)
    if n < 1 << 19:
        assert st.main_kernel_bytes == 4 * m + 4 * (n + 1) + 36 * n
        return
    assert fixed + 8 * -(-groups // 64) <= st.main_kernel_bytes <= fixed + 8 * groups
    with knobs(gx, pr__hot_sources=1000):
        st = gx.pagerank(G, tol=0.0, max_iter=2, precision="fp64")[1]
    assert st.main_kernel_bytes == 4 * m + 8 * (n + 1) + 36 * n + 16 * n


def test_sums_without_room_for_the_blocked_layout(gx):
    """Where device memory holds the row sweep but not the layout of the blocked
    sums (32 bytes of working memory an edge), a solve takes the row sweep instead
    of failing, and the layout once there is room again."""
    import torch
    G = gx.Graph.rmat(20, 16, symmetric=False, weights="lognormal")
    n, m = G.n, G.m
    assert m >= 1 << 23
    alone = gx.Graph.rmat(20, 16, symmetric=False, weights="lognormal")
    w = torch.from_numpy(alone.to_host()[2]).cuda()
    t = torch.full((n,), 1.0 / n, device="cuda")
    c = torch.linspace(-1, 1, n, device="cuda")

    def solve(H):
        a = gx.pagerank(H, tol=0.0, max_iter=5, precision="fp64")[0]
        x = gx.pagerank_weighted(H, w, t, tol=0.0, max_iter=5)[0]
        return (a, x, *gx.pagerank_adjoint(H, w, x, c, tol=0.0, max_iter=5)[:2])

    exp = [v.cpu().numpy() for v in solve(alone)]
    alone.free()
    # What both paths need: the degree order, the transpose, their vectors.
    with knobs(gx, pr__blocking=0):
        gx.pagerank(G, tol=0.0, max_iter=1)
    G.build_transpose()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    room = 28 * m  # the layouts want more, the row sweeps with their outputs about 16 m
    free, _ = torch.cuda.mem_get_info()
    hold = torch.empty(free - room, dtype=torch.uint8, device="cuda")
    print(f"m={m} free={free} held={free - room}", flush=True)
    got = [v.cpu().numpy() for v in solve(G)]
    del hold
    torch.cuda.empty_cache()
    again = [v.cpu().numpy() for v in solve(G)]
    for a, b, e in zip(got, again, exp):
        rel = 1e-12 if e.dtype == np.float64 else 1e-5
        assert np.abs(a - e).max() <= rel * np.abs(e).max()
        assert np.array_equal(b, e)


def two_out(n, dest, rng):
    """Every vertex with two weighted out-edges: one to dest[v], one to a random
    vertex (none is dangling; no vertex twice in a list)."""
    other = rng.integers(0, n, n)
    other = np.where(other == dest, (other + 1) % n, other)
    lo, hi = np.minimum(dest, other), np.maximum(dest, other)
    col = np.stack([lo, hi], 1).ravel().astype(np.int32)
    return np.arange(0, 2 * n + 1, 2, dtype=np.int32), col, (rng.random(2 * n) + 0.5).astype(np.float32)


def ulps(got, row, col, w, rows):
    """How far the values of `rows` after one iteration with alpha = 1/2 and no
    teleport are from half the exact row sum, in units of the last place: the
    iteration starts from the rounded 1 / n, halving is exact."""
    n = len(row) - 1
    src = np.repeat(np.arange(n), np.diff(row))
    wl = w.astype(np.longdouble)
    terms = np.longdouble(got.dtype.type(1.0 / n)) * wl / np.add.reduceat(wl, row[:-1])[src]
    keep = np.flatnonzero(np.isin(col, rows))
    keep = keep[np.argsort(col[keep], kind="stable")]
    at = np.searchsorted(col[keep], rows)
    exact = np.add.reduceat(terms[keep], at) / 2
    return np.abs(got[rows].astype(np.longdouble) - exact) / np.spacing(got[rows]).astype(np.longdouble)


@pytest.mark.parametrize("n,hubs", [(300007, 60), (1900003, 64), (1900003, 500), (1900003, 6000)])
def test_long_rows_are_rounded_once_in_fp64(gx, n, hubs):
    """Rows with hundreds to thousands of terms, spread over the tiles of the row
    sweep (fewer than 7 * 2^19 edges) or the chunks of the blocked sums: the sum is
    within half a unit of the last place of the exact one, and the parts' own
    roundings (each at a small share of the row: 0.09 units in all, four times
    that at most)."""
    import torch
    rng = np.random.default_rng(hubs)
    rows = np.sort(rng.choice(n, hubs, replace=False))
    row, col, w = two_out(n, rows[np.arange(n) % hubs], rng)
    G = gx.Graph.from_csr(row, col, w)
    t = torch.zeros(n, device="cuda")
    x, _ = gx.pagerank_weighted(G, torch.from_numpy(w).cuda(), t, alpha=0.5, tol=0.0, max_iter=1, precision="fp64")
    off = ulps(x.cpu().numpy(), row, col, w, rows)
    print(f"ulps n={n} hubs={hubs} mean {float(off.mean()):.3f} max {float(off.max()):.3f}", flush=True)
    assert off.max() <= 0.86


def test_rows_of_two_parts_are_rounded_once_in_fp32(gx):
    """FP32 rows whose terms lie in two chunks of the blocked sums: a part is not
    rounded to FP32 before it is added (0.5 units each, at half of the row), so
    that the row is within half a unit and the terms' own roundings (200 terms of
    0.4 units: 0.03 of the row's, four times that at most)."""
    import torch
    rng = np.random.default_rng(3)
    n = 116 * 16384
    v = np.arange(n)
    dest = (v >> 15) * 163 + np.minimum((v & 16383) // 100, 162)
    row, col, w = two_out(n, dest, rng)
    G = gx.Graph.from_csr(row, col, w)
    x, _ = gx.pagerank_weighted(G, torch.from_numpy(w).cuda(), torch.zeros(n, device="cuda"), alpha=0.5, tol=0.0,
                                max_iter=1)
    off = ulps(x.cpu().numpy(), row, col, w, np.unique(dest))
    print(f"ulps fp32 rows={len(off)} mean {float(off.mean()):.3f} max {float(off.max()):.3f}", flush=True)
    assert off.max() <= 0.65


# The blocked sums' side of the size rule (7 * 2^19 edges, 2^15 rows): few chunks and
# many, rows with edges in every chunk and over many of a wavefront's ranges, mostly
# empty rows, a last chunk of one vertex, few rows with many edges (small bins).
@pytest.mark.parametrize("n,m,hubs", [(32768, 3900000, 0), (65537, 7800000, 2), (1 << 20, 6000000, 1),
                                      (200000, 9000000, 0)])
def test_blocked_sums_shapes(gx, n, m, hubs):
    """As the row sweep's shapes, with the same tolerances."""
    assert len(weighted_csr(n, m, n + m, hubs)[1]) >= 7 << 19
    row_sweep_shapes(gx, n, m, hubs)


def test_dangling_mass_of_equal_ranks_in_fp64(gx):
    """Two million vertices without edges have one rank, v' = (1 + k v) / 2n with k
    of them and alpha = 1/2 (halving and n = 2^21 are exact).  Equal addends round
    alike, so a mass added up one by one is off by several units whatever the
    number of lanes; here it is off by at most one (a workgroup's part is rounded
    once, the parts are added pairwise but for four in a row), and the rank by half
    of that and half a unit of its own, plus the half of what the iteration before
    left: two units at most."""
    from fractions import Fraction
    rng = np.random.default_rng(9)
    n, busy = 1 << 21, 100003
    key = np.unique(rng.integers(0, busy, 9500000) * busy + rng.integers(0, busy, 9500000))
    row = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(key // busy, minlength=n), out=row[1:])
    col = (key % busy).astype(np.int32)
    assert len(col) >= 1 << 23 and np.diff(row)[:busy].min() > 0
    G = gx.Graph.from_csr(row, col)
    v = Fraction(1, n)
    worst = 0.0
    for k in range(1, 9):
        v = (1 + (n - busy) * v) / (2 * n)
        x = gx.pagerank(G, alpha=0.5, tol=0.0, max_iter=k, precision="fp64")[0].cpu().numpy()[busy:]
        assert np.all(x == x[0])
        off = abs(Fraction(float(x[0])) - v) / Fraction(float(np.spacing(x[0])))
        worst = max(worst, float(off))
        print(f"dangling k={k} off by {float(off):.3f} units", flush=True)
    assert worst <= 2.0
