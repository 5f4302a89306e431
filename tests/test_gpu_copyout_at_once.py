"""Copy-outs of several contexts at the same time that really share what there
is: more rings of many slots under way than are kept idle, more single slots
than are kept, and both at once with the helper threads between them.  Results
are whole words, which cross the link as they are: 2,500,003 of them are five
slots, where levels or small distances would be packed into one."""
import threading

import numpy as np
import pytest

import bfs_simd_benchmarks_amd as G

pytestmark = pytest.mark.gpu


def star(ctx, n, seed):
    """Vertex 0 points at every other vertex with weights up to 2^30, whose
    distances take whole words; (graph, distances)."""
    w = np.random.default_rng(seed).integers(1 << 20, 1 << 30, n - 1).astype(np.uint32)
    deg = np.zeros(n, np.uint32)
    deg[0] = n - 1
    g = ctx.graph_from_arrays(n, deg, W=4096, S=16, csr_edges=np.arange(1, n, dtype=np.uint32), csr_weights=w)
    g.retile(4096, 16)
    return g, np.concatenate([np.zeros(1, np.uint32), w])


@pytest.mark.parametrize("big,small", [(6, 0), (0, 20), (4, 10)])
def test_at_once(big, small):
    print(f"case: {big} copy-outs of several slots and {small} of one at once", flush=True)
    bad, rounds = [], 6
    start = threading.Barrier(big + small)

    def work(i):
        n = 2_500_003 if i < big else 3_001 + i
        try:
            with G.Context(0) as c:
                c.set_level_timing(False)
                g, ref = star(c, n, i)
                try:
                    for r in range(rounds):
                        start.wait(60)
                        if not np.array_equal(g.sssp(0)[0], ref):
                            bad.append((i, r, "distances"))
                        lv, pa, _ = g.bfs(0)
                        if lv[0] != 0 or not (lv[1:] == 1).all() or pa.any():
                            bad.append((i, r, "levels, parents"))
                        rows, _ = g.sssp_batch([1, 0])
                        if not np.array_equal(rows[1], ref):
                            bad.append((i, r, "rows"))
                finally:
                    g.free()
        except Exception as e:
            bad.append((i, repr(e)))
            start.abort()
    ths = [threading.Thread(target=work, args=(i,)) for i in range(big + small)]
    for t in ths:
        t.start()
    for t in ths:
        t.join()
    assert not bad
