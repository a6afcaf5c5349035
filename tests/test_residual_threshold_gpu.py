"""Residual PageRank where a residual, kept as hi + lo, stands on either side
of the threshold by its rounding errors: no vertex may be left with a residual
that grows without being passed on."""
import numpy as np
import pytest

D = 0.85
F = np.float32


def trap(sg, k, leaves):
    """k feeders with an edge to each of k targets, so that every target's
    first residual is k equal additions; each target feeds one vertex of its
    own. `leaves` vertices feed feeder 0, whose second push brings far more."""
    n = 3 * k + leaves
    target, feeder, end = np.arange(k), k + np.arange(k), 2 * k + np.arange(k)
    src = np.concatenate([np.repeat(feeder, k), target, 3 * k + np.arange(leaves)])
    dst = np.concatenate([np.tile(target, k), end, np.full(leaves, feeder[0])])
    row, col = sg.build_csr(n, src.astype(np.uint32), dst.astype(np.uint32))
    return sg.HostGraph(n, row, col, None)


def first_residual(n, k):
    """A target's hi + lo after the first round, its exact last sum, in the engine's FP32."""
    r0 = F((1 - D) / n)
    a = F(F(F(D) * r0) / F(k))
    hi = lo = F(0)
    for _ in range(k):
        exact = float(hi) + float(a)
        s = F(hi + a)
        lo = F(lo + F(exact - float(s)))
        hi = s
    return hi, lo, exact


def between(kind, leaves):
    """The fewest feeders with which the residual stands on both sides of some
    threshold, and that threshold."""
    for k in range(6, 64):
        n = 3 * k + leaves
        hi, lo, exact = first_residual(n, k)
        below = float(F(hi + lo)) if kind == "compensated" else exact
        if below < float(hi):
            return k, 0.5 * (below + float(hi))
    raise AssertionError("no such sum")


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["compensated", "rounded"])
@pytest.mark.parametrize("leaves,opts", [
    (2000, {"force_variant": "async_push_dd"}),  # activated from the queue
    (40, {"force_variant": "async_push_dd"}),    # by a scan
    (2000, {"pull_first": True}),                # in a pull round, then pushed to
    (40, {"pull_first": True}),
    (2000, {"force_variant": "async_push_dd", "iterative": True}),
    (40, {"force_variant": "async_push_dd", "iterative": True}),
])
def test_no_residual_is_left_behind(sg, gpu, kind, leaves, opts):
    k, theta = between(kind, leaves)
    hg = trap(sg, k, leaves)
    n = hg.n
    opts = dict(opts)
    mode = sg.PR_ITERATIVE if opts.pop("iterative", False) else sg.PR_PUSH_DD
    pull_first = opts.pop("pull_first", False)
    e = sg.Engine(sg.Graph(hg), **({"alpha": 2.0, "edge_factor": 1.0} if pull_first else opts))
    tol = theta * n / (1 - D)
    e.pagerank(D, tol, 0, mode)
    x, st = e.gather(np.float32).astype(np.float64), e.stats()
    if pull_first:
        assert st["pull_rounds"] >= 1 and st["push_rounds"] >= 1, st
    # y(v) = 1 + d sum (y(u) - r(u)) / outdeg(u), in units of (1 - d)/n, the
    # leaves' rank, with residuals 0 <= r(u) < tol left over; a residual and
    # its FP32 sum differ by their rounding errors
    y = x / x[-1]
    deg = np.diff(hg.row.astype(np.int64))
    src = np.repeat(np.arange(n), deg)

    def passed_on(left):
        return 1 + D * np.bincount(hg.col, weights=np.maximum(y - left, 0)[src] / deg[src], minlength=n)

    eps = 1e-5
    assert (y >= passed_on(tol * (1 + eps)) * (1 - eps)).all(), (k, tol, y[:k], y[2 * k:3 * k])
    assert (y <= passed_on(0.0) * (1 + eps)).all()
