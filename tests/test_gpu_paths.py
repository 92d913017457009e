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
