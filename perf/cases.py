"""The work that users of this framework have it do, as measurable cases.

Each case is one call of a public entry point on a resident graph: single
queries (BFS, SSSP, single-source BC), whole-graph PageRank, and batched
queries. Graphs are the two kinds the repository's tests and benchmark use: R-MAT
(a, b, c, d) = (0.57, 0.19, 0.19, 0.05) with self-loops and duplicates removed,
directed or symmetrised, and 4-neighbour grids with a tenth of the edges
deleted (road-network-like, high diameter). They are generated here with torch
from the seed; the sizes run from graphs whose queries cost a few launches'
latency to the benchmark's RMAT-22.

Integers (levels, distances) have one right answer; ranks and dependencies are
recomputed in 64 bits by `exact`.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sep-graph_amd"))
import sepgraph as sg  # noqa: E402

DEVICE = "cuda" if torch.cuda.is_available() else "cpu"
DAMPING, TOL = 0.85, 1e-6


def _rmat(name, op, n, ef=16, sym=False, **more):
    return {"name": name, "op": op, "graph": "rmat", "n": n, "ef": ef, "sym": sym, **more}


def _grid(name, op, rows, cols, **more):
    return {"name": name, "op": op, "graph": "grid", "rows": rows, "cols": cols, **more}


def listed():
    return [
        # the smallest call: a query on a graph that fits any cache, all latency
        _rmat("bfs-rmat12-sym", "bfs", 1 << 12, sym=True),
        # an ordinary traversal, ragged vertex count
        _rmat("bfs-rmat18-ragged", "bfs", 200_003),
        # the benchmark's query: directed RMAT-22
        _rmat("bfs-rmat22", "bfs", 1 << 22),
        # road-network-like: thousands of rounds with small frontiers
        _grid("bfs-grid2048", "bfs", 2048, 2048),
        # weighted shortest paths on a large skewed graph
        _rmat("sssp-rmat21", "sssp", 1 << 21, priority=False),
        # weighted shortest paths on a road-like graph, two-level priority (--sparse)
        _grid("sssp-grid1024-prio", "sssp", 1024, 1024, priority=True),
        # topology-driven PageRank to the default tolerance
        _rmat("pagerank-rmat21", "pr", 1 << 21, mode="pull"),
        # data-driven (residual) PageRank on an ordinary graph, ragged
        _rmat("pagerank-dd-rmat17-ragged", "pr", 100_003, mode="dd"),
        # one BC-dependency query of the serving mix
        _rmat("bc-one-rmat20", "bc_dep", 1 << 20),
        # batched queries: 64 BFS sharing their sweeps of the adjacency
        _rmat("bfs-multi64-rmat19", "bfs_multi", 1 << 19, k=64),
        # batched weighted queries, fewer than a full batch, ragged
        _rmat("sssp-multi24-rmat18", "sssp_multi", 230_017, k=24),
        # sampled betweenness centrality: the sum over 64 sources of a symmetrised graph
        _rmat("bc-sum64-rmat16-sym", "bc_sum", 1 << 16, sym=True, k=64),
    ]


def draw(rng):
    def size(lo, hi):
        n = int(math.exp(rng.uniform(math.log(lo), math.log(hi))))
        return min(hi, max(lo, n | rng.randint(0, 1)))

    def rmat(op, lo, hi, **more):
        return {"op": op, "graph": "rmat", "n": size(lo, hi), "ef": rng.choice([8, 11, 16, 16]),
                "sym": rng.random() < 0.3, **more}

    def grid(op, lo, hi, **more):
        return {"op": op, "graph": "grid", "rows": size(lo, hi), "cols": size(lo, hi), **more}

    def fit(case):  # a symmetrised graph has twice the edges: no more of them than the largest listed one
        if case.get("sym"):
            case["n"] = max(1 << 10, case["n"] // 2)
        return case

    kind = rng.choice(["bfs", "bfs", "bfs_grid", "sssp", "sssp", "sssp_grid", "pr", "pr", "pr_dd", "bc_dep", "bc_dep",
                       "bc_grid", "bfs_multi", "sssp_multi", "bc_sum"])
    k = rng.choice([2, 8, 17, 33, 64])
    if kind == "bfs":
        return fit(rmat("bfs", 1 << 10, 1 << 22))
    if kind == "bfs_grid":
        return grid("bfs", 64, 2048)
    if kind == "sssp":
        return fit(rmat("sssp", 1 << 10, 1 << 21, priority=False))
    if kind == "sssp_grid":
        return grid("sssp", 64, 1024, priority=rng.random() < 0.7)
    if kind == "pr":
        return fit(rmat("pr", 1 << 10, 1 << 21, mode="pull"))
    if kind == "pr_dd":
        return fit(rmat("pr", 1 << 10, 1 << 17, mode="dd"))
    if kind == "bc_dep":
        return fit(rmat("bc_dep", 1 << 10, 1 << 20))
    if kind == "bc_grid":
        return grid("bc_dep", 32, 400)
    if kind == "bfs_multi":
        return fit(rmat("bfs_multi", 1 << 12, 1 << 19, k=k))
    if kind == "sssp_multi":
        return fit(rmat("sssp_multi", 1 << 12, 1 << 17, k=k))
    return fit(rmat("bc_sum", 1 << 12, 1 << 16, k=k))


# ---------------------------------------------------------------- the graphs
def _edges(case, seed):
    """(n, src, dst) as int64 tensors, sorted by (src, dst), without duplicates or self-loops."""
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(1_000_003 * (seed + 1))
    if case["graph"] == "rmat":
        n = case["n"]
        scale = max(1, (n - 1).bit_length())
        count = case["ef"] * n
        src = torch.zeros(count, dtype=torch.int64, device=DEVICE)
        dst = torch.zeros(count, dtype=torch.int64, device=DEVICE)
        for _ in range(scale):
            r = torch.rand(count, generator=gen, device=DEVICE)
            src = src * 2 + (r >= 0.76)
            dst = dst * 2 + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
        keep = (src != dst) & (src < n) & (dst < n)
        src, dst = src[keep], dst[keep]
        sym = case["sym"]
    else:
        rows, cols = case["rows"], case["cols"]
        n, sym = rows * cols, True
        v = torch.arange(n, dtype=torch.int64, device=DEVICE)
        right, down = v[v % cols != cols - 1], v[: n - cols]
        src, dst = torch.cat([right, down]), torch.cat([right + 1, down + cols])
        keep = torch.rand(len(src), generator=gen, device=DEVICE) >= 0.1
        src, dst = src[keep], dst[keep]
    if sym:
        src, dst = torch.cat([src, dst]), torch.cat([dst, src])
    key = torch.unique(src * n + dst)
    return n, key // n, key % n


def _sources(src, n, k, seed):
    """k distinct vertices that have out-edges."""
    live = torch.unique(src).cpu().numpy()
    return np.random.RandomState(seed % (1 << 32)).choice(live, size=min(k, len(live)), replace=False).astype(np.uint32)


def _host_graph(case, seed):
    n, src, dst = _edges(case, seed)
    row = np.zeros(n + 1, np.uint32)
    row[1:] = torch.cumsum(torch.bincount(src, minlength=n), 0).cpu().numpy()
    w = None
    if case["op"] in ("sssp", "sssp_multi"):
        # one weight for an edge and its reverse, [1, 64) on R-MAT graphs and [1, 1000) on grids
        lo, hi = torch.minimum(src, dst), torch.maximum(src, dst)
        mix = (lo * 2_654_435_761 + hi * 40_503 + seed) % 1_000_000_007
        mix = (mix * 48_271) % 2_147_483_647
        w = (1 + mix % (63 if case["graph"] == "rmat" else 999)).cpu().numpy().astype(np.uint32)
    sources = _sources(src, n, case.get("k", 1), seed)
    undirected = case["graph"] == "grid" or case["sym"]
    return sg.HostGraph(n, row, dst.cpu().numpy().astype(np.uint32), w, undirected=undirected), sources


class _View:
    """Device memory of the engine's value array, for torch.as_tensor."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 2}


def prepare(case, seed):
    hg, sources = _host_graph(case, seed)
    graph = sg.Graph(hg)
    opts = {"priority": 1} if case.get("priority") else {}
    engine = sg.Engine(graph, stream=torch.cuda.current_stream().cuda_stream, **opts)
    return {"case": case, "n": hg.n, "graph": graph, "engine": engine, "sources": sources, "view": (None, None)}


def _value(state, rows, typestr):
    """The engine's value array as a tensor; levels and distances as int32 (-1: unreached)."""
    ptr, _ = state["engine"].value_ptr()
    if state["view"][0] != ptr:
        shape = (rows, state["n"]) if rows > 1 else (state["n"],)
        view = torch.as_tensor(_View(ptr, shape, typestr), device="cuda")
        view.engine = state["engine"]  # the memory is the engine's: it lives as long as the result
        state["view"] = (ptr, view)
    return state["view"][1]


def run(state):
    e, s, op = state["engine"], state["sources"], state["case"]["op"]
    if op == "bfs":
        e.bfs(s[0])
        return _value(state, 1, "<i4")
    if op == "sssp":
        e.sssp(s[0])
        return _value(state, 1, "<i4")
    if op == "pr":
        e.pagerank(DAMPING, TOL, 0, sg.PR_PULL_TD if state["case"]["mode"] == "pull" else sg.PR_PUSH_DD)
        return _value(state, 1, "<f4")
    if op == "bc_dep":
        e.bc_dependency(s, 1)
        return _value(state, 1, "<f4")
    if op == "bfs_multi":
        e.bfs_multi(s)
        return _value(state, len(s), "<i4")
    if op == "sssp_multi":
        e.sssp_multi(s)
        return _value(state, len(s), "<i4")
    e.bc(s)
    return _value(state, 1, "<f4")


def work(case):
    if case["graph"] == "rmat":
        n = case["n"]
        m = 0.9 * case["ef"] * n * (2 if case["sym"] else 1)
    else:
        n = case["rows"] * case["cols"]
        m = 3.6 * n
    k = case.get("k", 1)
    graph = 4 * (n + 1) + 4 * m
    op = case["op"]
    if op in ("bfs", "bfs_multi"):
        return {"bytes": graph + 4 * n * k, "flops": m * k}
    if op in ("sssp", "sssp_multi"):
        return {"bytes": graph + 4 * m + 4 * n * k, "flops": 2 * m * k}
    if op == "pr":
        # about sixteen sweeps of the edges at this tolerance
        return {"bytes": 16 * (graph + 8 * n), "flops": 16 * 2 * m}
    # Brandes: the edges forward and backward, path counts and dependencies in between
    return {"bytes": 2 * graph + 16 * n + 4 * n, "flops": 4 * m * k}


# ----------------------------------------------------------- 64-bit results
def _exact_pagerank(n, src, dst, mode):
    outdeg = torch.bincount(src, minlength=n).double()
    inv = torch.where(outdeg > 0, 1.0 / outdeg, torch.zeros_like(outdeg))
    dangling = outdeg == 0
    x = torch.full((n,), 1.0 / n, dtype=torch.float64, device=src.device)
    tol = TOL if mode == "pull" else 1e-13  # residual propagation approaches the fixed point itself
    for _ in range(1000):
        s = torch.zeros_like(x).index_add_(0, dst, (x * inv)[src])
        y = (1 - DAMPING) / n + DAMPING * (s + x[dangling].sum() / n)
        change = float((y - x).abs().sum())
        x = y
        if change < tol:
            break
    return x


def _exact_dependency(n, src, dst, s):
    level = torch.full((n,), -1, dtype=torch.int64, device=src.device)
    level[s] = 0
    sigma = torch.zeros(n, dtype=torch.float64, device=src.device)
    sigma[s] = 1.0
    steps = []
    while True:
        at = level[src] == len(steps)
        fresh = at & (level[dst] < 0)
        level[dst[fresh]] = len(steps) + 1
        u, w = src[at], dst[at]
        dag = level[w] == len(steps) + 1
        u, w = u[dag], w[dag]
        if not len(u):
            break
        sigma.index_add_(0, w, sigma[u])
        steps.append((u, w))
    delta = torch.zeros_like(sigma)
    for u, w in reversed(steps):
        delta.index_add_(0, u, sigma[u] / sigma[w] * (1.0 + delta[w]))
    delta[s] = 0.0
    return 0.5 * delta


def exact(case, seed):
    op = case["op"]
    if op not in ("pr", "bc_dep", "bc_sum"):
        return None  # whole numbers
    n, src, dst = _edges(case, seed)
    if op == "pr":
        return _exact_pagerank(n, src, dst, case["mode"])
    total = torch.zeros(n, dtype=torch.float64, device=src.device)
    for s in _sources(src, n, case.get("k", 1), seed):
        total += _exact_dependency(n, src, dst, int(s))
    return total
