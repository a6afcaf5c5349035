"""Round kernels at the sizes where their tiles end: in-degrees around the
rows and chunks a wave keeps in flight, frontiers around the limits of the
small-round path."""
import numpy as np
import pytest


def fan_in_graph(sg, degrees, extra=0):
    """One vertex per entry of `degrees` with that many in-edges, from sources
    that follow them in id order; `extra` isolated vertices at the end."""
    k = len(degrees)
    nsrc = max(degrees) if len(degrees) else 0
    n = k + nsrc + extra
    src = np.concatenate([k + np.arange(d) for d in degrees]).astype(np.uint32)
    dst = np.repeat(np.arange(k), degrees).astype(np.uint32)
    # the fanned-in vertices link back to the sources, so mass keeps moving
    back = np.arange(min(k, nsrc))
    src = np.concatenate([src, back.astype(np.uint32)])
    dst = np.concatenate([dst, (k + back).astype(np.uint32)])
    row, col = sg.build_csr(n, src, dst)
    return sg.HostGraph(n, row, col, None)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["pull", "dd"])
@pytest.mark.parametrize("degrees", [
    [1], [7, 8, 9, 15, 16, 17], list(range(1, 71)),
    [63, 64, 65, 127, 128, 255, 256, 257, 511, 512, 513, 1025], [64] * 64 + [65] * 3,
])
def test_pagerank_in_degree_edges(sg, orc, gpu, degrees, mode):
    hg = fan_in_graph(sg, degrees, extra=3)
    e = sg.Engine(sg.Graph(hg))
    e.pagerank(0.85, 1e-9, 0, sg.PR_PULL_TD if mode == "pull" else sg.PR_PUSH_DD)
    got = e.gather(np.float32).astype(np.float64)
    ref = orc.pagerank(hg.row, hg.col, 0.85, 1e-12)
    ref = ref[0] if isinstance(ref, tuple) else ref
    # FP32 ranks: one rounding each, sums compensated
    assert np.abs(got - ref).sum() / ref.sum() < 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("relabel", [False, True])
@pytest.mark.parametrize("block_size,n", [(256, 9983), (256, 9985), (512, 19969), (1024, 39935), (1024, 39937), (1024, 45001)])
def test_pagerank_pull_staged_ids_and_hub_chunks(sg, orc, gpu, block_size, n, relabel):
    """Ids around the last one whose contribution is staged, in-hubs of one
    chunk, of several, and of more than eight lanes add up."""
    rng = np.random.default_rng(n)
    hubs = [d for d in (65, 256, 257, 2048, 2049, 16384, 16385, 30000) if d < n]
    src = np.concatenate([rng.choice(n, d, replace=False) for d in hubs] + [rng.integers(0, n, 4 * n), np.arange(n)])
    dst = np.concatenate([np.full(d, i * 7) for i, d in enumerate(hubs)] + [rng.integers(0, n, 4 * n), (np.arange(n) * 5 + 1) % n])
    row, col = sg.build_csr(n, src.astype(np.uint32), dst.astype(np.uint32))
    hg = sg.HostGraph(n, row, col, None)
    e = sg.Engine(sg.Graph(hg, relabel=relabel), block_size=block_size)
    e.pagerank(0.85, 1e-10, 0, sg.PR_PULL_TD)
    got = e.gather(np.float32).astype(np.float64)
    ref = orc.pagerank(hg.row, hg.col, 0.85, 1e-12)
    ref = ref[0] if isinstance(ref, tuple) else ref
    # three FP32 roundings per rank and iteration, carried on by 1 / (1 - d)
    assert np.abs(got - ref).sum() / ref.sum() < 3 * 2.0**-24 / 0.15


def path_graph(sg, n):
    v = np.arange(n - 1, dtype=np.uint32)
    row, col = sg.build_csr(n, v, v + 1, symmetrize=True)
    return sg.HostGraph(n, row, col, None, undirected=True)


def random_graph(sg, n, degree, seed, weights=None):
    rng = np.random.default_rng(seed)
    src = rng.integers(0, n, n * degree).astype(np.uint32)
    dst = rng.integers(0, n, n * degree).astype(np.uint32)
    row, col = sg.build_csr(n, src, dst)
    w = None if weights is None else rng.integers(weights[0], weights[1], len(col)).astype(np.uint32)
    return sg.HostGraph(n, row, col, w)


def star_chain(sg, n, leaves):
    """A path whose every 50th vertex also has `leaves` leaves."""
    hubs = np.arange(0, n, 50)
    src = np.concatenate([np.arange(n - 1), np.repeat(hubs, leaves)]).astype(np.uint32)
    dst = np.concatenate([np.arange(1, n), n + np.arange(len(hubs) * leaves)]).astype(np.uint32)
    total = n + len(hubs) * leaves
    row, col = sg.build_csr(total, src, dst, symmetrize=True)
    return sg.HostGraph(total, row, col, None, undirected=True)


SMALL_ROUND_GRAPHS = {
    # the whole query on one XCD's blocks: words and their remainders, the limit, hubs
    "n1": lambda sg: sg.HostGraph(1, np.zeros(2, np.uint32), np.zeros(0, np.uint32), None),
    "n63": lambda sg: random_graph(sg, 63, 3, 1),
    "n64": lambda sg: random_graph(sg, 64, 3, 2),
    "n65": lambda sg: random_graph(sg, 65, 3, 3),
    "n16384": lambda sg: random_graph(sg, 16384, 8, 4),
    "n16385": lambda sg: random_graph(sg, 16385, 8, 5),
    "stars": lambda sg: star_chain(sg, 300, 257),
    "path9000": lambda sg: path_graph(sg, 9000),
    "rmat13": lambda sg: sg.rmat_graph(13, 16, symmetrize=True, seed=6),
    # narrow rounds of a larger graph: more rounds than one phase holds, a
    # frontier that outgrows the limit and shrinks again, hubs on the way
    "path20000": lambda sg: path_graph(sg, 20000),
    "random": lambda sg: random_graph(sg, 60000, 3, 7),
    "dense": lambda sg: random_graph(sg, 40000, 40, 8),
    "stars-long": lambda sg: star_chain(sg, 17000, 300),
    "grid": lambda sg: sg.grid_graph(131, 257, 0.1, seed=9, weights=None),
    "rmat17": lambda sg: sg.rmat_graph(17, 16, symmetrize=False, seed=10),
}


@pytest.mark.gpu
@pytest.mark.parametrize("opts", [{}, {"block_size": 256}, {"grid_blocks": 1}, {"force_variant": "async_pull_dd"},
                                  {"force_variant": "async_push_dd"}, {"max_iteration": 3}])
@pytest.mark.parametrize("name", list(SMALL_ROUND_GRAPHS))
def test_bfs_small_rounds(sg, orc, gpu, name, opts):
    if name in ("path9000", "path20000", "stars-long") and opts and "max_iteration" not in opts:
        pytest.skip("long traversal: default schedule and round limit only")
    hg = SMALL_ROUND_GRAPHS[name](sg)
    e = sg.Engine(sg.Graph(hg), **opts)
    for s in sorted({0, hg.n // 2, hg.n - 1}):
        e.bfs(s)
        got = e.gather(np.int32)
        ref = orc.bfs(hg.row, hg.col, s)
        cap = opts.get("max_iteration")
        if cap:
            ref = np.where(ref > cap, -1, ref)
        assert np.array_equal(got, ref), s
        assert e.stats()["rounds"] == (min(cap, ref.max() + 1) if cap else ref.max() + 1)


def weighted(sg, hg, lo, hi, seed):
    w = sg.gen_weights(hg.row, hg.col, lo, hi, seed=seed, symmetric=hg.undirected)
    return sg.HostGraph(hg.n, hg.row, hg.col, w, undirected=hg.undirected)


def distances(orc, hg, w, s, weights):
    """Shortest distances; where sums pass 2^32, which the oracle's 32-bit sums
    would wrap, 64-bit ones cut off at the unreached mark, as the engine's."""
    if weights is None or weights[1] < 1 << 20:
        return orc.sssp_dijkstra(hg.row, hg.col, w, s)
    from scipy.sparse import csr_matrix
    from scipy.sparse.csgraph import dijkstra

    g = csr_matrix((w.astype(np.float64), hg.col.astype(np.int64), hg.row.astype(np.int64)), shape=(hg.n, hg.n))
    return np.minimum(dijkstra(g, indices=s), 2.0**32 - 1).astype(np.uint32)


@pytest.mark.gpu
@pytest.mark.parametrize("opts", [{}, {"priority": 1}, {"block_size": 256}, {"grid_blocks": 1},
                                  {"force_variant": "async_pull_dd"}, {"priority": 1, "priority_threshold": 3.0}])
@pytest.mark.parametrize("weights", [None, (1, 64), (0, 3), (1 << 30, 1 << 31)])
@pytest.mark.parametrize("name", list(SMALL_ROUND_GRAPHS))
def test_sssp_small_rounds(sg, orc, gpu, name, weights, opts):
    if name in ("path9000", "path20000", "stars-long") and (opts or weights != (1, 64)):
        pytest.skip("long traversal: default schedule and one weight range only")
    hg = SMALL_ROUND_GRAPHS[name](sg)
    if weights:
        hg = weighted(sg, hg, *weights, seed=3)
    e = sg.Engine(sg.Graph(hg), **opts)
    w = hg.w if weights else np.ones(hg.m, np.uint32)
    for s in sorted({0, hg.n - 1}):
        e.sssp(s)
        assert np.array_equal(e.gather(np.uint32), distances(orc, hg, w, s, weights)), s
        # and a BFS on the same engine in between
        e.bfs(s)
        assert np.array_equal(e.gather(np.int32), orc.bfs(hg.row, hg.col, s)), s


@pytest.mark.gpu
@pytest.mark.parametrize("opts", [{}, {"block_size": 256}, {"grid_blocks": 1}, {"force_variant": "async_pull_dd"},
                                  {"force_variant": "async_push_dd"}])
@pytest.mark.parametrize("name", [n for n in SMALL_ROUND_GRAPHS if n != "n1"])
def test_bc_small_levels(sg, orc, gpu, name, opts):
    if name in ("path9000", "path20000", "stars-long") and opts:
        pytest.skip("long traversal: default schedule only")
    hg = SMALL_ROUND_GRAPHS[name](sg)
    e = sg.Engine(sg.Graph(hg), **opts)
    sources = sorted({0, hg.n // 3, hg.n - 1})
    e.bc_dependency(sources, 1)
    got = e.gather(np.float32).reshape(len(sources), hg.n)
    st = e.stats()
    total = np.zeros(hg.n)
    depth = 0
    for i, s in enumerate(sources):
        ref, _ = orc.bc_single(hg.row, hg.col, s)
        total += ref
        depth = max(depth, int(orc.bfs(hg.row, hg.col, s).max()))
        # FP64 sums, one rounding to FP32
        np.testing.assert_allclose(got[i], ref, rtol=1e-6, atol=1e-6)
    assert st["iterations"] == len(sources) and st["max_depth"] == depth
    e.bc(sources, 1)
    np.testing.assert_allclose(e.gather(np.float32), total, rtol=1e-6, atol=1e-6)


BATCH_GRAPHS = ["n65", "n16385", "stars", "rmat13", "rmat17", "dense", "grid"]


@pytest.mark.gpu
@pytest.mark.parametrize("k", [1, 2, 9, 33, 64, 70])
@pytest.mark.parametrize("name", BATCH_GRAPHS)
def test_bfs_batches(sg, orc, gpu, name, k):
    hg = SMALL_ROUND_GRAPHS[name](sg)
    e = sg.Engine(sg.Graph(hg))
    src = np.random.default_rng(k).integers(0, hg.n, k)  # repeats among them
    e.bfs_multi(src)
    got = e.gather(np.int32).reshape(k, hg.n)
    for i in sorted({0, k // 2, k - 1}):
        assert np.array_equal(got[i], orc.bfs(hg.row, hg.col, int(src[i]))), i
    assert e.stats()["status"] == 0
    e.bc(src)
    # FP64 sums, one rounding to FP32
    np.testing.assert_allclose(e.gather(np.float32), orc.bc(hg.row, hg.col, src), rtol=1e-5, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("opts", [{}, {"force_variant": "async_push_dd"}, {"block_size": 256}])
@pytest.mark.parametrize("weights", [None, (0, 3), (1, 64), (1 << 30, 1 << 31)])
@pytest.mark.parametrize("k", [1, 2, 7, 16, 24, 64, 70])
@pytest.mark.parametrize("name", BATCH_GRAPHS)
def test_sssp_batches(sg, orc, gpu, name, k, weights, opts):
    if opts and (weights != (1, 64) or k not in (16, 64)):
        pytest.skip("options: one weight range, two batch sizes")
    hg = SMALL_ROUND_GRAPHS[name](sg)
    if weights:
        hg = weighted(sg, hg, *weights, seed=5)
    w = hg.w if weights else np.ones(hg.m, np.uint32)
    e = sg.Engine(sg.Graph(hg), **opts)
    src = np.random.default_rng(k).integers(0, hg.n, k)
    e.sssp_multi(src)
    got = e.gather(np.uint32).reshape(k, hg.n)
    for i in sorted({0, k - 1}):
        assert np.array_equal(got[i], distances(orc, hg, w, int(src[i]), weights)), i


@pytest.mark.gpu
@pytest.mark.parametrize("call", ["bfs", "sssp", "pull", "dd", "bfs_multi", "sssp_multi", "bc", "bc_one", "bc_dependency"])
@pytest.mark.parametrize("k", [1, 5])
def test_calls_back_to_back_and_their_time(sg, gpu, call, k):
    """Calls queued one behind the other, each with sources of its own, give
    what each gives alone; the reported time is within the call's own."""
    import time
    hg = random_graph(sg, 5000, 6, 3, weights=(1, 64))
    graph = sg.Graph(hg)
    run = {
        "bfs": lambda e, s: e.bfs(int(s[0])),
        "sssp": lambda e, s: e.sssp(int(s[0])),
        "pull": lambda e, s: e.pagerank(0.85, 1e-6, 0, sg.PR_PULL_TD),
        "dd": lambda e, s: e.pagerank(0.85, 1e-6, 0, sg.PR_PUSH_DD),
        "bfs_multi": lambda e, s: e.bfs_multi(s, 4),
        "sssp_multi": lambda e, s: e.sssp_multi(s, 4),
        "bc": lambda e, s: e.bc(s, 4),
        "bc_one": lambda e, s: e.bc(s, 1),
        "bc_dependency": lambda e, s: e.bc_dependency(s, 4),
    }[call]
    dtype = np.float32 if call in ("pull", "dd", "bc", "bc_one", "bc_dependency") else np.uint32
    rng = np.random.default_rng(k)
    sets = [rng.choice(hg.n, k, replace=False).astype(np.uint32) for _ in range(4)]
    e = sg.Engine(graph)
    for s in sets:
        run(e, s)
    got = e.gather(dtype)
    e.stats()
    t = time.perf_counter()
    run(e, sets[0])
    ms = e.stats()["kernel_ms"]
    wall = (time.perf_counter() - t) * 1e3
    assert 0.0 < ms < wall
    alone = sg.Engine(graph)
    run(alone, sets[-1])
    want = alone.gather(dtype)
    if call == "dd" or call.startswith("bc"):  # atomic additions in any order
        assert np.allclose(got, want, rtol=1e-5, atol=1e-12)
    else:
        assert np.array_equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("relabel", [False, True])
@pytest.mark.parametrize("block_size,n", [(256, 7679), (256, 7681), (512, 15361), (1024, 30719), (1024, 30721), (0, 20000)])
def test_residual_pull_rounds_and_push_rounds_agree(sg, orc, gpu, block_size, n, relabel):
    """Pull rounds activate in the pass that sums; push rounds in one of their
    own. Stopped after the same number of rounds, whatever the directions, the
    ranks are the same; run to the end they are the oracle's."""
    rng = np.random.default_rng(n)
    hubs = [d for d in (65, 256, 257, 2049, 16385, 20000) if d < n]
    src = np.concatenate([rng.choice(n, d, replace=False) for d in hubs] + [rng.integers(0, n, 4 * n)])
    dst = np.concatenate([np.full(d, i * 7) for i, d in enumerate(hubs)] + [rng.integers(0, n, 4 * n) // 2])
    row, col = sg.build_csr(n, src.astype(np.uint32), dst.astype(np.uint32))
    graph = sg.Graph(sg.HostGraph(n, row, col, None), relabel=relabel)
    bound = 3 * 2.0**-24 / 0.15  # three FP32 roundings per rank and round, carried on by 1 / (1 - d)

    def ranks(max_iter, tol, **opts):
        e = sg.Engine(graph, block_size=block_size, **opts)
        e.pagerank(0.85, tol, max_iter, sg.PR_PUSH_DD)
        return e.gather(np.float32).astype(np.float64), e.stats()

    for rounds in (1, 2, 3, 7):
        push, ps = ranks(rounds, 1e-9, force_variant="async_push_dd")
        pull, qs = ranks(rounds, 1e-9, force_variant="async_pull_dd")
        assert ps["rounds"] == qs["rounds"] == rounds and ps["pull_rounds"] == 0 and qs["pull_rounds"] == rounds
        assert np.abs(push - pull).sum() / push.sum() < bound
    ref = orc.pagerank(row, col, 0.85, 1e-12)
    ref = ref[0] if isinstance(ref, tuple) else ref
    # thresholds from "every round pulls" to "none does": both directions, either after the other
    mixed = 0
    for alpha in (1e9, 1e4, 1e3, 300.0, 100.0, 30.0, 10.0, 1e-3):
        got, st = ranks(0, 1e-9, alpha=alpha)
        mixed += st["push_rounds"] > 0 and st["pull_rounds"] > 0
        assert np.abs(got - ref).sum() / ref.sum() < bound
    assert mixed


@pytest.mark.gpu
@pytest.mark.parametrize("nsrc", [1, 3, 4, 5, 8, 9, 16, 17, 33, 64])
@pytest.mark.parametrize("graph", ["path", "random", "islands"])
def test_bfs_batch_level_rows(sg, gpu, graph, nsrc):
    """Levels of a renumbered graph, kept as bytes until the end: rows of each
    width, levels around the last a byte holds, sources that share a vertex,
    vertices that no source reaches."""
    if graph == "path":
        hg = path_graph(sg, 600)  # levels up to 599
    elif graph == "random":
        hg = random_graph(sg, 3001, 3, nsrc)
    else:
        v = np.arange(0, 900, 2, dtype=np.uint32)
        row, col = sg.build_csr(901, v, v + 1, symmetrize=True)
        hg = sg.HostGraph(901, row, col, None, undirected=True)
    rng = np.random.default_rng(nsrc)
    src = rng.integers(0, hg.n, nsrc).astype(np.uint32)
    if nsrc > 2:
        src[1] = src[0]
        src[2] = 0
    g = sg.Graph(hg, relabel=True)
    e = sg.Engine(g)
    one = sg.Engine(g)
    for batch in (64, max(1, nsrc - 1)):
        e.bfs_multi(src, batch)
        got = e.gather(np.int32).reshape(nsrc, hg.n)
        for i, s in enumerate(src):
            one.bfs(int(s))
            assert np.array_equal(got[i], one.gather(np.int32)), (batch, i)
