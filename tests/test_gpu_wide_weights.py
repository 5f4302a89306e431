"""SSSP with weights near 2^32, whose sums do not fit 32 bits: such a path is
longer than any distance and lowers nothing, in every level loop (one launch,
two launches per level, five kernels per level) and by push and by sweep.
A cycle of such edges reached at a finite distance must not lower itself on
and on: the graphs have a few edges, so a traversal takes a few levels."""
import numpy as np
import pytest

import oracle as O
import bfs_simd_benchmarks_amd as G

pytestmark = pytest.mark.gpu

BIG = 0xFFFFFFFF
EDGES = [(0, 1, 10 ** 9), (1, 2, BIG), (2, 1, 0),             # a cycle a wrapping sum lowers by 1 a round
         (0, 3, 0x7FFFFFFE), (3, 4, 0), (3, 5, 1),            # the largest distance; one past it
         (0, 6, 0x80000000), (1, 7, BIG - 10 ** 9 + 8),       # past INT_MAX; past 2^32 by 7
         (0, 8, 5), (8, 1, 10 ** 9 - 6), (4, 9, BIG), (9, 0, 0)]


# n: one launch, two launches per level; t_ratio 1: every step a push, 20: sweeps after the first
@pytest.mark.parametrize("timing", [False, True])
@pytest.mark.parametrize("t_ratio", [1, 20])
@pytest.mark.parametrize("n", [10, 8193])
def test_wide_weights(n, t_ratio, timing):
    h, t, w = (np.array(x, np.uint32) for x in zip(*EDGES))
    g = O.tile_edgelist(n, h, t, 64, 2, w)
    with G.Context(0, t_ratio=t_ratio) as c:
        c.set_level_timing(timing)
        gg = c.graph_from_arrays(g.n, g.deg, W=g.W, S=g.S, csr_edges=g.cols, csr_weights=g.cw, tile_heads=g.sh,
                                 tile_tails=g.st, tile_weights=g.sw, tile_offsets=g.soff)
        try:
            for src in (0, 1, 3, 9):
                print(f"case: wide weights n={n} t_ratio={t_ratio} timing={timing} src={src}", flush=True)
                d, st = gg.sssp(src)
                ref = O.sssp_dijkstra(g.n, g.deg, g.cols, g.cw, src)
                assert np.array_equal(d, ref), (d[:10], ref[:10])
                assert st.steps <= 8
            rows, _ = gg.sssp_batch([0, 9])
            assert np.array_equal(rows[1], O.sssp_dijkstra(g.n, g.deg, g.cols, g.cw, 9))
        finally:
            gg.free()
