"""PageRank's tile sweep against the FP64 oracle where its segments can go
wrong: in-degrees around a lane's 32 adds times the lanes a segment gets, around
a tile's 2048 edges and over many tiles, tiles of one segment and of single
edges, vertices without in- or out-edges, and more vertices than one head band
serves (2^22)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def run(ctx, n, h, t, iters):
    order = np.lexsort((t, h))
    h, t = h[order].astype(np.uint32), t[order].astype(np.uint32)
    deg = np.bincount(h, minlength=n).astype(np.uint32)
    g = ctx.graph_from_arrays(n, deg, W=4096, S=16, csr_edges=t)
    try:
        a, _ = g.pagerank(iters, 0.85, 1.0 / n)
        b, _ = g.pagerank(iters, 0.85, 1.0 / n)
    finally:
        g.free()
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))      # a fixed order of additions
    ref = O.pagerank_f64(n, h, t, deg, iters, 0.85, 1.0 / n)
    assert float(np.abs(a.astype(np.float64) - ref).sum()) < 1e-6
    assert np.allclose(a, ref, rtol=2e-6, atol=0)


@pytest.mark.parametrize("indeg", [[1], [2048], [2047, 1, 2], [2049, 3], [5000, 1, 5000], [32, 33] * 40,
                                   [64, 65, 127, 128, 129] * 9, [1] * 5000, [31, 1] * 300 + [12_001],
                                   [0, 7, 0, 0, 4096, 0, 2048, 2049, 0, 1]])
def test_segment_lengths(ctx, indeg):
    """Tail i gets indeg[i] in-edges, from as many different heads."""
    n = max(len(indeg), max(indeg)) + 13
    print(f"case: pagerank in-degrees {indeg[:6]}... n={n}", flush=True)
    rng = np.random.default_rng(len(indeg) + indeg[0])
    h = np.concatenate([rng.permutation(n)[:c] for c in indeg])
    t = np.repeat(np.arange(len(indeg)), indeg)
    run(ctx, n, h, t, 3)


@pytest.mark.parametrize("n", [(1 << 22) - 1, (1 << 22) + 700_001])
def test_one_band_and_several(ctx, n):
    """Around the vertex count past which heads are cut into bands; the last
    window of heads has no edges, tail 5 has in-edges from every window."""
    print(f"case: pagerank n={n}", flush=True)
    rng = np.random.default_rng(1)
    hi = n - (1 << 19)
    h = np.concatenate([rng.integers(0, hi, 3_000_000), np.arange(0, hi, 37)])
    t = np.concatenate([rng.integers(0, n, 3_000_000), np.full(len(range(0, hi, 37)), 5)])
    e = np.unique(h * n + t)
    run(ctx, n, e // n, e % n, 2)
