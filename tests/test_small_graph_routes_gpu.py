"""Small graphs on either side of the lines between queries run whole by one
XCD's blocks and by rounds of the whole grid (team_whole_graph)."""
import numpy as np
import pytest


def exact_graph(sg, n, m, seed):
    """n vertices, exactly m edges, weights in [1, 64)."""
    rng = np.random.default_rng(seed)
    key = np.sort(rng.choice(n * n, m, replace=False))
    row = np.zeros(n + 1, np.uint32)
    row[1:] = np.cumsum(np.bincount(key // n, minlength=n))
    return sg.HostGraph(n, row, (key % n).astype(np.uint32), rng.integers(1, 64, m).astype(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("over", [0, 1])
@pytest.mark.parametrize("call,n,m,opts", [
    ("bfs", 3000, 1 << 18, {}),
    ("bfs", 5000, 64 * 5000, {}),
    ("bfs", 3000, 65536, {"force_variant": "async_push_dd"}),
    ("bfs", 3000, 1_000_000, {"force_variant": "async_pull_dd"}),
    ("sssp", 3000, 1 << 18, {}),
    ("sssp", 10000, 32 * 10000, {}),
    ("sssp", 3000, 24576, {"force_variant": "async_push_dd"}),
    ("sssp", 10000, 4 * 10000, {"priority": 1}),
    ("sssp", 3000, 1 << 18, {"force_variant": "async_pull_dd"}),
    ("bc", 3000, 1 << 18, {}),
    ("bc", 3000, 1_000_000, {"force_variant": "async_pull_dd"}),
])
def test_results_on_both_sides_of_a_line(sg, orc, gpu, call, n, m, opts, over):
    hg = exact_graph(sg, n, m + over, seed=m)
    e = sg.Engine(sg.Graph(hg), **opts)
    for s in (0, n - 1):
        if call == "bfs":
            e.bfs(s)
            assert np.array_equal(e.gather(np.int32), orc.bfs(hg.row, hg.col, s))
        elif call == "sssp":
            e.sssp(s)
            assert np.array_equal(e.gather(np.uint32), orc.sssp_dijkstra(hg.row, hg.col, hg.w, s))
        else:
            e.bc_dependency([s], 1)
            # FP64 sums, one rounding to FP32
            np.testing.assert_allclose(e.gather(np.float32), orc.bc_single(hg.row, hg.col, s)[0], rtol=1e-6, atol=1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("n,m,opts", [(4000, 930_000, {}), (4000, 930_000, {"force_variant": "async_push_dd"}),
                                      (16000, 930_000, {"force_variant": "async_push_dd"})])
def test_dense_graphs_are_not_left_to_one_xcd(sg, gpu, n, m, opts):
    """A query whose rounds walk many edges takes no longer than by rounds of
    the whole grid, which is what stage_hubs runs (2 to 3 times as long by one
    XCD's blocks)."""
    g = sg.Graph(exact_graph(sg, n, m, seed=1))

    def median(**more):
        e = sg.Engine(g, **opts, **more)
        ms = []
        for s in range(25):
            e.bfs(s * (n // 25))
            ms.append(e.stats()["kernel_ms"])
        return float(np.median(ms[4:]))

    assert median() < 1.4 * median(stage_hubs=1)
