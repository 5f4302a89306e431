"""Results on their way to the host: row and vertex counts around the 32
values a lane packs, one slot and several slots of staging, levels that need 4
bits, 8 bits and whole words, rows of odd length, and calls from several
threads and contexts at once."""
import threading

import numpy as np
import pytest

import oracle as O
import bfs_simd_benchmarks_amd as G

pytestmark = pytest.mark.gpu


def path_graph(ctx, n, extra):
    """A path 0 -> 1 -> ... -> extra, every later vertex hanging off it: vertex
    v > extra is a child of v % (extra + 1)."""
    h = np.concatenate([np.arange(extra), np.arange(extra + 1, n) % (extra + 1)]).astype(np.uint32)
    t = np.arange(1, n, dtype=np.uint32)
    order = np.lexsort((t, h))
    deg = np.bincount(h, minlength=n).astype(np.uint32)
    g = ctx.graph_from_arrays(n, deg, W=4096, S=16, csr_edges=t[order], csr_weights=np.ones(n - 1, np.uint32))
    g.retile(4096, 16)
    lv = np.arange(n, dtype=np.int64)
    lv[extra + 1:] = np.arange(extra + 1, n) % (extra + 1) + 1
    return g, lv


# depth 13, 14, 15: 4 bits or 8; 253..256: 8 bits or whole words
@pytest.mark.parametrize("depth", [13, 14, 15, 253, 254, 255, 256])
@pytest.mark.parametrize("n", [300, 4099])
def test_levels_by_depth(ctx, depth, n):
    g, lv = path_graph(ctx, n, depth)
    try:
        print(f"case: copy-out depth={depth} n={n}", flush=True)
        got, pa, _ = g.bfs(0)
        assert np.array_equal(got, lv)
        assert pa[0] == 0 and np.array_equal(lv[pa[1:]] + 1, lv[1:])
        mid, _, _ = g.bfs(5, parents=False)      # vertices before the source stay unreached
        ref = O.bfs_levels(g.n, *csr(g), 5)
        assert np.array_equal(mid, ref)
        if depth < 254:
            rows, _ = g.bfs_batch([0, 5, 0])
            assert np.array_equal(rows[0], lv.astype(np.uint8)) and np.array_equal(rows[2], rows[0])
            assert np.array_equal(rows[1].astype(np.int64), np.where(ref < 0, 255, ref))
    finally:
        g.free()


def csr(g):
    d = g.download(tiles=False)
    return d["deg"], d["cols"]


@pytest.mark.parametrize("n", [31, 32, 33, 1000, 524_287, 524_289, 4_194_305, 4_200_001])
def test_sizes_around_slots(ctx, n):
    """One source per row of an odd length, words (SSSP, hops, ranks) and levels
    over one and several 2 MiB slots."""
    g, lv = path_graph(ctx, n, 10)
    try:
        print(f"case: copy-out n={n}", flush=True)
        assert np.array_equal(g.bfs(0, parents=False)[0], lv)
        assert np.array_equal(g.sssp(0)[0], lv.astype(np.uint32))
        assert np.array_equal(g.bellman_ford(0)[0], lv.astype(np.uint32))
        for k in (1, 3):
            d, _ = g.sssp_batch([0] * k)
            assert d.shape == (k, n) and (d == lv.astype(np.uint32)).all()
            rows, _ = g.bfs_batch([0] * k)
            assert (rows == lv.astype(np.uint8)).all()
        r, _ = g.pagerank(1, 0.85, 1.0)
        ref = np.zeros(n)
        deg, cols = csr(g)
        np.add.at(ref, cols, 1.0 / np.repeat(deg, deg))
        assert np.allclose(r, 0.15 / n + 0.85 * ref, rtol=1e-5, atol=0)
    finally:
        g.free()


def test_concurrent_contexts():
    """More copy-outs at once than idle staging is kept for, several slots each."""
    n, threads = 2_500_003, 6
    bad = []

    def work(i):
        with G.Context(0) as c:
            c.set_level_timing(False)
            g, lv = path_graph(c, n, 3 + i)
            try:
                for _ in range(4):
                    if not np.array_equal(g.bfs(0, parents=False)[0], lv):
                        bad.append((i, "bfs"))
                    if not np.array_equal(g.sssp(0)[0], lv.astype(np.uint32)):
                        bad.append((i, "sssp"))
            finally:
                g.free()
    print(f"case: copy-out from {threads} contexts at once", flush=True)
    ths = [threading.Thread(target=work, args=(i,)) for i in range(threads)]
    for t in ths:
        t.start()
    for t in ths:
        t.join()
    assert not bad


@pytest.mark.parametrize("top", [14, 15, 254, 255, 65_534, 65_535, 70_000])
@pytest.mark.parametrize("n", [262_144, 300_013])
def test_distances_by_width(ctx, top, n):
    """A star whose largest distance is `top`: 4, 8 or 16 bits per distance on
    the way, or whole words; every third vertex is unreached."""
    rng = np.random.default_rng(top)
    t = np.flatnonzero(np.arange(n) % 3 != 2)[1:].astype(np.uint32)
    w = rng.integers(1, top + 1, len(t)).astype(np.uint32)
    w[:2] = (top, 1)
    deg = np.zeros(n, np.uint32)
    deg[0] = len(t)
    g = ctx.graph_from_arrays(n, deg, W=4096, S=16, csr_edges=t, csr_weights=w)
    g.retile(4096, 16)
    try:
        print(f"case: copy-out top={top} n={n}", flush=True)
        ref = np.full(n, O.INT_MAX, np.uint32)
        ref[0], ref[t] = 0, w
        assert np.array_equal(g.sssp(0)[0], ref)
        rows, _ = g.sssp_batch([0, 1, 0])
        one = np.full(n, O.INT_MAX, np.uint32)
        one[1] = 0
        assert np.array_equal(rows[0], ref) and np.array_equal(rows[1], one) and np.array_equal(rows[2], ref)
        hops = np.full(n, O.INT_MAX - 2, np.uint32)
        hops[0], hops[t] = 0, 1
        assert np.array_equal(g.bellman_ford(0)[0], hops)
    finally:
        g.free()
