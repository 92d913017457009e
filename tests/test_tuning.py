"""Defaults of the tuning knobs.  No GPU."""
from __future__ import annotations


def test_hub_slices_are_a_matter_of_vertices():
    """The default of sssp.hub_refine does not depend on the edges: below 2^24
    vertices an entry point uses 0 whatever their number, from there on 1."""
    import galois_amd as gx
    for m in (0, 7 << 24, (1 << 31) - 1):
        assert gx.tune_effective("sssp.hub_refine", (1 << 24) - 1, m) == 0, m
        assert gx.tune_effective("sssp.hub_refine", 1 << 24, m) == 1, m
