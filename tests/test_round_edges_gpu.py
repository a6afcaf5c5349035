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
