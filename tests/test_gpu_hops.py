"""Hop relaxation with skipped chunks and heads: against BFS levels over tile
widths around the LDS row window (4096 vertices), both tile orders, sparse rows
whose chunks span many tile rows, limited sweeps, and paths whose sweeps pass
the ring of sweep records and the byte stamps."""
import numpy as np
import pytest

import oracle as O
import bfs_simd_benchmarks_amd as G

pytestmark = pytest.mark.gpu
INF = O.INT_MAX - 2


def graph(ctx, n, h, t, W, S, order):
    e = np.unique(h.astype(np.int64) * n + t)
    h, t = (e // n).astype(np.uint32), (e % n).astype(np.uint32)
    deg = np.bincount(h, minlength=n).astype(np.uint32)
    g = ctx.graph_from_arrays(n, deg, W=W, S=S, csr_edges=t)
    g.retile(W, S, order)
    return g, deg, t


def want(n, deg, cols, src):
    lv = O.bfs_levels(n, deg, cols, src)
    return np.where(lv >= 0, lv, INF).astype(np.uint32)


@pytest.mark.parametrize("order", [G.TILES_ROW_MAJOR, G.TILES_COL_STRIPE])
@pytest.mark.parametrize("W", [7, 64, 1000, 2048, 4096, 4097, 70000])
def test_hops_equal_levels(ctx, W, order):
    n = 20_011
    rng = np.random.default_rng(W)
    h = np.concatenate([rng.integers(0, n, 60_000), np.zeros(3000, np.int64), rng.integers(0, 300, 40_000)])
    t = np.concatenate([rng.integers(0, n, 60_000), rng.integers(0, n, 3000), rng.integers(0, n, 40_000)])
    g, deg, cols = graph(ctx, n, h, t, W, 4, order)
    try:
        for src in (0, 5000, n - 1):
            print(f"case: hops W={W} order={order} src={src}", flush=True)
            d, run, ms = g.bellman_ford(src)
            assert np.array_equal(d, want(n, deg, cols, src))
            assert 1 <= run < 99 and ms > 0
    finally:
        g.free()


@pytest.mark.parametrize("order", [G.TILES_ROW_MAJOR, G.TILES_COL_STRIPE])
def test_hops_on_a_shuffled_path(ctx, order):
    """600 vertices of a path in random order: hundreds of sweeps."""
    n = 600
    p = np.random.default_rng(2).permutation(n)
    g, deg, cols = graph(ctx, n, p[:-1], p[1:], 16, 4, order)
    try:
        print(f"case: hops shuffled path order={order}", flush=True)
        d, run, _ = g.bellman_ford(int(p[0]), 10_000)
        ref = np.empty(n, np.uint32)
        ref[p] = np.arange(n)
        assert np.array_equal(d, ref) and run <= n
        # after s sweeps every vertex within s hops holds its distance
        for s in (0, 1, 2, 7, 300):
            d, run, _ = g.bellman_ford(int(p[0]), s)
            assert run <= s and np.array_equal(d[p[:s + 1]], np.arange(s + 1))
            assert (d[p[s + 1:]] >= s + 1).all()
            if s == 0:
                assert (d[p[1:]] == INF).all()
    finally:
        g.free()
