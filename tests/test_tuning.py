"""Defaults of the tuning knobs, and the autotuner's cache key: workloads whose best
knob values differ do not share an entry.  No GPU."""
from __future__ import annotations

from types import SimpleNamespace

import numpy as np

from galois_amd import autotune


def graph():
    row = np.array([0, 2, 3, 4], np.int32)
    return SimpleNamespace(n=3, m=4, flags=1, to_host=lambda: (row, None, None))


def test_signature_holds_the_arguments_that_change_the_best_values():
    G = graph()
    key = lambda algo, **args: autotune.signature(None, G, algo, args)  # noqa: E731
    # How many hub slices a bucket holds depends on its width.
    assert key("sssp", shift=6) != key("sssp", shift=13)
    assert key("sssp") == key("sssp", shift=6, source=2)  # the runner's default shift
    assert key("pagerank", precision="fp32") != key("pagerank", precision="fp64")
    assert key("bc", sources=range(64)) != key("bc", sources=range(65))
    assert key("bfs", source=0) == key("bfs", source=1)
    assert key("bfs") != key("cc")


def test_hub_slices_are_a_matter_of_vertices():
    """The default of sssp.hub_refine does not depend on the edges: below 2^24
    vertices an entry point uses 0 whatever their number, from there on 1."""
    import galois_amd as gx
    for m in (0, 7 << 24, (1 << 31) - 1):
        assert gx.tune_effective("sssp.hub_refine", (1 << 24) - 1, m) == 0, m
        assert gx.tune_effective("sssp.hub_refine", 1 << 24, m) == 1, m
