"""Team phases with the blocks outside the team late: they read the counters
of the round that started a phase long after its members have gone on (a
build of the library that holds them up, tests/cpp/late_blocks.hpp)."""
import importlib.util
import os
import sys

import numpy as np
import pytest

import test_round_edges_gpu as R

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "tests", "cpp", "bin", "libsepgraph_late.so")


@pytest.fixture(scope="module")
def late():
    if not os.path.exists(LIB):
        pytest.fail("tests/cpp/bin/libsepgraph_late.so is not built: run __graft_entry__.build()")
    spec = importlib.util.spec_from_file_location("sepgraph_late", os.path.join(ROOT, "sep-graph_amd", "sepgraph.py"))
    mod = importlib.util.module_from_spec(spec)
    sys.modules[spec.name] = mod
    spec.loader.exec_module(mod)
    mod.LIB_PATH = LIB
    mod.lib()
    return mod


# phases of every length: to the end, thousands of rounds, a few between wide
# rounds, one
GRAPHS = {
    "path": lambda sg: R.path_graph(sg, 20000),
    "grid": lambda sg: sg.grid_graph(131, 257, 0.1, seed=9, weights=None),
    "random": lambda sg: R.random_graph(sg, 60000, 3, 7),
    "dense": lambda sg: R.random_graph(sg, 40000, 40, 8),
    "stars": lambda sg: R.star_chain(sg, 3400, 300),
    "rmat": lambda sg: sg.rmat_graph(17, 8, symmetrize=False, seed=10),
}


def sources(hg):
    """Several queries one after the other: the state each leaves is the next one's."""
    live = np.flatnonzero(np.diff(hg.row.astype(np.int64)))
    return [int(s) for s in (live[0], live[len(live) // 2], live[-1], live[len(live) // 3])]


@pytest.mark.gpu
@pytest.mark.parametrize("block_size", [0, 256])
@pytest.mark.parametrize("name", list(GRAPHS))
def test_bfs_with_late_blocks(late, orc, gpu, name, block_size):
    hg = GRAPHS[name](late)
    e = late.Engine(late.Graph(hg), block_size=block_size)
    for s in sources(hg):
        e.bfs(s)
        assert np.array_equal(e.gather(np.int32), orc.bfs(hg.row, hg.col, s)), s
        assert e.stats()["status"] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("opts", [{}, {"block_size": 256}, {"priority": 1}])
@pytest.mark.parametrize("name", list(GRAPHS))
def test_sssp_with_late_blocks(late, orc, gpu, name, opts):
    hg = R.weighted(late, GRAPHS[name](late), 1, 64, seed=3)
    e = late.Engine(late.Graph(hg), **opts)
    for s in sources(hg)[:2]:
        e.sssp(s)
        assert np.array_equal(e.gather(np.uint32), orc.sssp_dijkstra(hg.row, hg.col, hg.w, s)), s


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(GRAPHS))
def test_bc_with_late_blocks(late, orc, gpu, name):
    hg = GRAPHS[name](late)
    e = late.Engine(late.Graph(hg))
    for s in sources(hg)[:2]:
        e.bc_dependency([s], 1)
        ref, _ = orc.bc_single(hg.row, hg.col, s)
        # FP64 sums, one rounding to FP32
        np.testing.assert_allclose(e.gather(np.float32), ref, rtol=1e-6, atol=1e-6)
