"""Batched SSSP: which batches pull, and the same distances either way."""
import numpy as np
import pytest


def graph(sg, n, hub_in):
    """A random graph of mean degree 8; `hub_in`: in-edges of vertex 0 beside."""
    rng = np.random.default_rng(n)
    src = np.concatenate([rng.integers(0, n, 8 * n), np.arange(1, hub_in + 1)])
    dst = np.concatenate([rng.integers(0, n, 8 * n), np.zeros(hub_in, np.int64)])
    row, col = sg.build_csr(n, src.astype(np.uint32), dst.astype(np.uint32))
    return sg.HostGraph(n, row, col, rng.integers(1, 64, len(col)).astype(np.uint32))


# groups of 16 lanes pull on graphs of 12 288 vertices and more, or without an
# in-hub (in-degree above 64); wider ones always, narrower ones never
@pytest.mark.gpu
@pytest.mark.parametrize("n,hub_in,k,pulls", [
    (12287, 300, 16, False), (12288, 300, 16, True), (12287, 0, 16, True), (2000, 300, 9, False),
    (12287, 300, 17, True), (2000, 300, 64, True), (12288, 0, 8, False),
])
def test_which_batches_pull(sg, orc, gpu, n, hub_in, k, pulls):
    hg = graph(sg, n, hub_in)
    e = sg.Engine(sg.Graph(hg))
    src = np.random.default_rng(k).choice(n, k, replace=False)
    e.sssp_multi(src)
    got = e.gather(np.uint32).reshape(k, n)
    assert (e.stats()["pull_rounds"] > 0) == pulls
    for i in (0, k - 1):
        assert np.array_equal(got[i], orc.sssp_dijkstra(hg.row, hg.col, hg.w, int(src[i])))
