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


def blocked_shapes():
    """A source with 600K out-edges (one chunk in several phase-1 pieces), a
    destination with 600K in-edges (its bin cut into slices), one vertex past a 16K
    chunk boundary, a band of vertices without edges, dangling vertices."""
    rng = np.random.default_rng(23)
    n = 5 * 16384 + 16385
    k = 600000
    src = np.concatenate([np.full(k, 70000), rng.integers(0, n, k), rng.integers(0, 16384, 200000)])
    dst = np.concatenate([rng.integers(0, n, k), np.full(k, 3), rng.integers(0, n, 200000)])
    quiet = (src >= 32768) & (src < 49152) | (dst >= 32768) & (dst < 49152)
    src, dst = np.append(src[~quiet], n - 1), np.append(dst[~quiet], 0)
    key = np.unique(src[src != dst] * n + dst[src != dst])
    row = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(key // n, minlength=n), out=row[1:])
    return row, (key % n).astype(np.int32)


@pytest.mark.parametrize("edges", [-1, 1 << 12, 1 << 30])
@pytest.mark.parametrize("shape", ["tables", "rmat16", "rmat20", "one chunk"])
def test_blocked_fp32_sweep(gx, oracle, shape, edges):
    """The propagation-blocked FP32 sweep where the default rule would pull (the
    knob is set): 1e-6 in L1 of the FP64 oracle, bit for bit the same again, on a
    second handle and however its bins are cut.  Sums are exact, so that only a
    lost or doubled contribution could differ."""
    if shape == "tables":
        row, col = blocked_shapes()
    elif shape == "one chunk":
        row, col, _ = weighted_csr(16384, 50000, 2, 1)
    else:
        row, col, _ = gx.Graph.rmat(int(shape[4:]), 16, symmetric=False).to_host()
    print(f"blocked {shape} n={len(row) - 1} m={len(col)} task_edges={edges}", flush=True)
    exp, it, _ = oracle.pagerank(row, col, tol=1e-10, max_iter=200, threads=8)
    got = []
    with knobs(gx, pr__blocking=1):
        A = gx.Graph.from_csr(row, col)
        got.append(gx.pagerank(A, tol=1e-10, max_iter=200)[0].cpu().numpy())
        assert gx.pagerank_layout_info(A)["tasks"] > 0  # the blocked sweep ran
        with knobs(gx, pr__task_edges=edges):
            B = gx.Graph.from_csr(row, col)
            for _ in range(2):
                got.append(gx.pagerank(B, tol=1e-10, max_iter=200)[0].cpu().numpy())
        info = gx.pagerank_layout_info(B)
        assert info["tasks"] > 0 and (edges != 1 << 30 or info["sliced_bins"] == 0)
        assert edges != 1 << 12 or shape == "one chunk" or info["sliced_bins"] > 0
    assert np.abs(got[0].astype(np.float64) - exp).sum() < 1e-6
    for x in got[1:]:
        assert np.array_equal(got[0], x)
    with knobs(gx, pr__blocking=0):  # the pull agrees to rounding, on a graph without a layout
        C = gx.Graph.from_csr(row, col)
        pulled = gx.pagerank(C, tol=1e-10, max_iter=200)[0].cpu().numpy()
        assert gx.pagerank_layout_info(C) == {}
    assert np.abs(pulled.astype(np.float64) - exp).sum() < 1e-6


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


def one_step(row, col, w, t, c, alpha):
    """One forward iteration from 1/n and, from c, one adjoint iteration with the
    gradients, in FP64 numpy with its infinities and NaNs; beside each value the
    sum of its terms' magnitudes, and how far the worst row's weights cancel."""
    n = len(row) - 1
    src = np.repeat(np.arange(n), np.diff(row))
    w = w.astype(np.float64)

    def rows(at, vals):
        out = np.zeros(n)
        np.add.at(out, at, vals)
        return out

    def step(w, t, c, inv, none, sign):
        x0 = np.full(n, 1.0 / n)
        x = (1 - alpha) * t + alpha * x0[none].sum() / n + alpha * rows(col, (x0 * inv)[src] * w)

        def below(lam):
            return np.where(none, lam.sum() / n, rows(src, lam[col] * w) * inv)

        lam = c + alpha * below(c)
        return x, alpha * t[src] * (lam[col] + sign * below(lam)[src]) * inv[src], (1 - alpha) * lam

    with np.errstate(all="ignore"):
        s = rows(src, w)
        inv = np.where(s > 0, 1.0 / np.where(s > 0, s, 1.0), 0.0)
        none = inv == 0
        cancel = (rows(src, np.abs(w)) * inv)[~none].max()
        return step(w, t, c, inv, none, -1), step(np.abs(w), t, np.abs(c), inv, none, 1), cancel


@pytest.mark.parametrize("n,m", [(5000, 40000), (32768, 3900000), (100003, 3900000)])
@pytest.mark.parametrize("values", ["signs", "scales", "not finite"])
@pytest.mark.parametrize("order", ["ascending", "random", "repeated"])
def test_row_sums_of_any_values_and_orders(gx, n, m, values, order):
    """The row sweep and the blocked sums on adjacency lists in any order and with
    repeated entries, on sums of either sign, of scales far apart, with infinities
    and NaNs in some rows: FP64 as numpy's to 1e-12 of the terms' magnitudes (times
    the worst cancellation in a row's weight sum), and not finite in exactly the
    same places."""
    import torch
    rng = np.random.default_rng(n + len(order))
    row, col, w = weighted_csr(n, m, n, 1 if n < 10000 else 0)
    if order != "ascending":
        src = np.repeat(np.arange(n), np.diff(row))
        if order == "repeated":
            again = rng.random(len(col)) < 0.2
            src, col, w = (np.concatenate([a, a[again]]) for a in (src, col, w))
        o = np.lexsort((rng.random(len(src)), src))
        src, col, w = src[o], col[o], w[o]
        row = np.zeros(n + 1, np.int32)
        np.cumsum(np.bincount(src, minlength=n), out=row[1:])
    t = (rng.random(n) / n).astype(np.float32)
    c = rng.standard_normal(n).astype(np.float32)
    if values == "signs":
        w[rng.random(len(w)) < 0.1] *= -0.5  # a row whose sum is not positive counts as dangling
    elif values == "scales":
        w = np.exp2(rng.integers(-40, 40, len(w))).astype(np.float32)
        c *= np.exp2(rng.integers(-30, 30, n)).astype(np.float32)
    else:
        w[rng.integers(0, len(w), 5)] = [np.inf, np.nan, np.inf, np.nan, np.inf]
        c[rng.integers(0, n, 3)] = [np.inf, -np.inf, np.nan]
    print(f"row sums n={n} m={len(col)} {values} {order}", flush=True)
    G = gx.Graph.from_csr(row, col, w)
    ww, tt, cc = (torch.from_numpy(a).cuda() for a in (w, t, c))
    x, _ = gx.pagerank_weighted(G, ww, tt, alpha=0.5, tol=0.0, max_iter=1, precision="fp64")
    gw, gt, _ = gx.pagerank_adjoint(G, ww, tt.double(), cc, alpha=0.5, tol=0.0, max_iter=1, precision="fp64")
    got = [a.cpu().numpy() for a in (x, gw, gt)]
    ref, size, cancel = one_step(row, col, w, t.astype(np.float64), c.astype(np.float64), 0.5)
    for name, a, b, mag in zip(("x", "grad_w", "grad_t"), got, ref, size):
        assert np.array_equal(np.isnan(a), np.isnan(b)), name
        inf = np.isinf(b)
        assert np.array_equal(np.isinf(a), inf) and np.array_equal(a[inf], b[inf]), name
        ok = np.isfinite(b) & np.isfinite(mag)
        # At most 2^20 FP64 roundings of the terms, and of the inverse row sums.
        assert np.abs(a[ok] - b[ok]).max() <= 1e-12 * cancel * mag[ok].max(), name


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
