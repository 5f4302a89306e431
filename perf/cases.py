"""The work a user has this framework do, as cases that can be timed and compared.

A case is one call (or, for serving, one burst of queries) on a resident
graph: `prepare` makes the graph and keeps its handle, as a program does that
answers many queries on it, and `run` is the call, with its results where
the entry point puts them: host arrays, or device arrays for the BFS that
allocates nothing.

The graphs are RMAT edge lists (a=0.57 b=0.19 c=0.19 d=0.05, self-loops and
duplicates dropped, ids in descending out-degree order), the distribution of
bfs_simd_benchmarks_amd/workloads.py, drawn with torch from the seed and handed
over as arrays; the 1.2e9-edge graph comes from the framework's own generator.

BFS cases ask for levels without parents: any valid parent may win a race, so
parents differ from run to run.  The number of sweeps of the hop relaxation is
left out for the same reason.
"""
import ctypes

import numpy as np
import torch

import bfs_simd_benchmarks_amd as gphi

DAMPING = float(np.float32(0.85))


def listed():
    return [
        # a toy graph: nothing but latency and launches
        dict(name="bfs-rmat10", kind="bfs", n=1 << 10, ef=16, W=128, S=4),
        # the smallest benchmark configuration (rmat16, edge factor 16)
        dict(name="bfs-rmat16", kind="bfs", n=1 << 16, ef=16, W=1024, S=16),
        # the pokec shape (1.6M vertices, about 30M edges), levels left on the
        # device by the call that allocates nothing
        dict(name="bfs-dev-pokec", kind="bfs_dev", n=1_632_803, ef=21, W=1024, S=16),
        # the headline graph: rmat25, edge factor 36, levels to the host
        dict(name="bfs-rmat25", kind="bfs_gen", n=1 << 25, ef=36, W=2048, S=32),
        # many queries on one graph of the serving mix, one bit each
        dict(name="batch64-rmat22", kind="batch", n=1 << 22, ef=16, W=1024, S=16, k=64),
        # the widest batch, on a smaller graph of odd size
        dict(name="batch256-300007", kind="batch", n=300_007, ef=12, W=512, S=8, k=256),
        # the weighted benchmark configuration (weights 1..255)
        dict(name="sssp-rmat16", kind="sssp", n=1 << 16, ef=16, W=1024, S=16, wmax=255),
        # one shortest-path query on a large graph of odd size
        dict(name="sssp-3000017", kind="sssp", n=3_000_017, ef=16, W=1024, S=16, wmax=255),
        # as many shortest-path queries as one traversal takes
        dict(name="sssp16-rmat20", kind="sssp_batch", n=1 << 20, ef=16, W=1024, S=16, wmax=255, k=16),
        # PageRank of the pokec shape, the benchmark's 20 iterations
        dict(name="pagerank-pokec", kind="pagerank", n=1_632_803, ef=21, W=1024, S=16, iters=20),
        # hop relaxation to the fixpoint over row-major tiles
        dict(name="hops-rmat22", kind="hops", n=1 << 22, ef=16, W=1024, S=16),
        # a burst of 60 queries on three resident graphs of the serving mix
        dict(name="serve-60", kind="serve", n=1 << 20, ef=16, W=1024, S=16, wmax=255, queries=60),
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["bfs", "bfs", "bfs_dev", "batch", "batch", "sssp", "sssp", "sssp_batch", "pagerank", "hops",
                       "serve"])
    hi = {"bfs": 1 << 23, "bfs_dev": 4_500_000, "batch": 1 << 22, "sssp": 1 << 22, "sssp_batch": 1 << 21,
          "pagerank": 1 << 22, "hops": 1 << 22, "serve": 1 << 20}[kind]
    n = _log_uniform(rng, 1 << 10, hi)
    c = dict(kind=kind, n=n, ef=rng.randint(4, 24), W=rng.choice([256, 512, 1000, 1024, 2048, 4096]),
             S=rng.choice([4, 8, 16, 32]))
    if kind == "batch":
        c["k"] = max(1, min(_log_uniform(rng, 2, 256), (1 << 28) // n))
    if kind == "sssp_batch":
        c["k"] = rng.randint(2, 16)
    if kind in ("sssp", "sssp_batch", "serve"):
        c["wmax"] = rng.choice([1, 255, 255, 65535])
    if kind == "pagerank":
        c["iters"] = rng.choice([1, 5, 20])
    if kind == "serve":
        c["n"] = max(n, 1 << 14)
        c["queries"] = rng.randint(8, 60)
    return c


def _graph(n, ef, seed, wmax=0):
    """(degrees, tails in CSR order, weights or None) of an RMAT graph, on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    scale = max(1, (n - 1).bit_length())
    m = n * ef
    h = torch.zeros(m, dtype=torch.int64, device="cuda")
    t = torch.zeros(m, dtype=torch.int64, device="cuda")
    for _ in range(scale):
        u = torch.rand(m, generator=g, device="cuda")
        h = 2 * h + (u >= 0.76)
        t = 2 * t + (((u >= 0.57) & (u < 0.76)) | (u >= 0.95))
    keep = (h < n) & (t < n) & (h != t)
    e = torch.unique(h[keep] * n + t[keep])
    h, t = e // n, e % n
    order = torch.argsort(torch.bincount(h, minlength=n), descending=True, stable=True)
    new = torch.empty_like(order)
    new[order] = torch.arange(n, device="cuda")
    e = torch.sort(new[h] * n + new[t]).values
    h, t = e // n, e % n
    w = torch.randint(1, wmax + 1, (len(t),), generator=g, device="cuda") if wmax else None
    return torch.bincount(h, minlength=n), t, w


def _sources(deg, k, seed):
    """k vertices with out-edges, in the order of the seed."""
    g = torch.Generator(device="cuda").manual_seed(seed + 7)
    live = int((deg > 0).sum())     # descending degrees: they come first
    return torch.randint(0, live, (k,), generator=g, device="cuda").cpu().numpy().astype(np.uint32)


def _host(x):
    return None if x is None else x.to(torch.int32).cpu().numpy().view(np.uint32)


class _Resident:
    """What a program keeps: its context, graph and sources; released with it."""

    def __init__(self, case, seed):
        self.case = case
        self.server = None
        n, row_major = case["n"], case["kind"] == "hops"
        self.ctx = gphi.Context(0)
        self.ctx.set_level_timing(False)
        if case["kind"] == "bfs_gen":
            self.graph = self.ctx.generate(scale=(n - 1).bit_length(), nverts=n, seed=seed & 0xFFFFF,
                                           samples=n * case["ef"], W=case["W"], S=case["S"])
            deg = torch.from_numpy(self.graph.download(csr=False, tiles=False)["deg"].astype(np.int64)).cuda()
        else:
            deg = self.load(self.ctx, n, seed, case.get("wmax", 0), row_major)
        self.sources = _sources(deg, case.get("k", 1), seed)
        if case["kind"] == "bfs_dev":
            self.levels = torch.empty(n, dtype=torch.int32, device="cuda")
            self.stats = gphi.Stats()
        del deg
        torch.cuda.empty_cache()    # the framework allocates beside torch

    def load(self, ctx, n, seed, wmax, row_major=False):
        c = self.case
        deg, cols, w = _graph(n, c["ef"], seed, wmax)
        self.graph = ctx.graph_from_arrays(n, _host(deg), W=c["W"], S=c["S"], csr_edges=_host(cols),
                                           csr_weights=_host(w))
        self.graph.retile(c["W"], c["S"], gphi.TILES_ROW_MAJOR if row_major else gphi.TILES_COL_STRIPE)
        return deg

    def __del__(self):
        if self.server:
            self.server.close()
        elif getattr(self, "graph", None):
            self.graph.free()
            self.ctx.close()


class _Serving(_Resident):
    """Three resident graphs, the second one weighted, and a burst of queries
    (20% of them shortest paths) with the arrays their answers go to."""

    def __init__(self, case, seed):
        self.case = case
        self.server = gphi.Server(max_batch=64)
        ids, srcs, ns = [], [], [case["n"] // 4, case["n"] // 2, case["n"]]
        for i, n in enumerate(ns):
            ctx = gphi.Context(0)
            deg = self.load(ctx, n, seed + i, case["wmax"] if i == 1 else 0)
            srcs.append(_sources(deg, case["queries"], seed + i))
            ids.append(self.server.add_graph(self.graph))
            del deg
        torch.cuda.empty_cache()
        self.burst = []
        for q in range(case["queries"]):
            sssp = q % 5 == 4
            i = 1 if sssp else q % 3
            kind = gphi.QUERY_SSSP if sssp else gphi.QUERY_BFS
            out = np.zeros(ns[i], np.uint32 if sssp else np.int32)
            self.burst.append((ids[i], kind, int(srcs[i][q]), out))


def prepare(case, seed):
    return (_Serving if case["kind"] == "serve" else _Resident)(case, seed)


def run(state):
    kind, g = state.case["kind"], state.graph
    if kind in ("bfs", "bfs_gen"):
        return g.bfs(int(state.sources[0]), parents=False)[0]
    if kind == "bfs_dev":
        lib = state.ctx.lib
        state.ctx.check(lib.gphi_bfs_noalloc(g.h, int(state.sources[0]), state.levels.data_ptr(), None,
                                             ctypes.byref(state.stats)))
        return state.levels
    if kind == "batch":
        return g.bfs_batch(state.sources)[0]
    if kind == "sssp":
        return g.sssp(int(state.sources[0]))[0]
    if kind == "sssp_batch":
        return g.sssp_batch(state.sources)[0]
    if kind == "pagerank":
        return g.pagerank(state.case["iters"], DAMPING, 1.0 / g.n)[0]
    if kind == "hops":
        return g.bellman_ford(int(state.sources[0]))[0]
    tickets = [state.server.submit(*q) for q in state.burst]
    for t in tickets:
        state.server.wait(t)
    return [q[3] for q in state.burst]


def work(case):
    """Each edge (a 4-byte id, and its weight) and vertex read once, per
    iteration of PageRank and per traversal otherwise, and the results written
    once.  Traversals do no floating-point arithmetic."""
    n, m, kind = case["n"], case["n"] * case["ef"], case["kind"]
    weight = 0 if not case.get("wmax") else 1 if case["wmax"] < 256 else 4
    if kind == "pagerank":
        return {"bytes": case["iters"] * (4 * m + 12 * n), "flops": case["iters"] * (m + 4 * n)}
    if kind == "batch":
        return {"bytes": 4 * m + 4 * n + case["k"] * n, "flops": 0}
    if kind == "sssp_batch":
        return {"bytes": (4 + weight) * m + 4 * n + 4 * case["k"] * n, "flops": 0}
    if kind == "serve":
        # each of the three graphs (n/4, n/2, n) once, and every answer
        return {"bytes": int(1.75 * (4 * m + 4 * n)) + int(case["queries"] * 4 * n * 0.58), "flops": 0}
    return {"bytes": (4 + weight) * m + 8 * n, "flops": 0}


def exact(case, seed):
    """PageRank in 64 bits; the other results are whole numbers."""
    if case["kind"] != "pagerank":
        return None
    n = case["n"]
    deg, tails, _ = _graph(n, case["ef"], seed)
    heads = torch.repeat_interleave(torch.arange(n, device="cuda"), deg)
    rank = torch.full((n,), 1.0 / n, dtype=torch.float64, device="cuda")
    d = deg.double()
    for _ in range(case["iters"]):
        contrib = torch.where(deg > 0, rank / d, torch.zeros_like(rank))
        got = torch.zeros_like(rank).index_add_(0, tails, contrib[heads])
        rank = (1.0 - DAMPING) / n + DAMPING * got
    return rank.cpu().numpy()
