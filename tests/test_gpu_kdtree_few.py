"""kd-tree lists of launches that do not fill the chip: one query a wave, or the
wave's last one, is walked by all 64 lanes, with the other group's memory for its
stack. Counts around the rule's edges (6144 queries: one a wave; 98304, and 49152 for
k = 33 to 64: no wave walks a lone query any more; 3072 below k = 8), the buffer sizes' edges in k, searches that open
far more nodes than the stack holds, and queries that are not numbers, which find
nothing and cost next to nothing. Lists are exact against the oracle."""
import time

import numpy as np
import pytest

import pyoracle as O

pytestmark = pytest.mark.gpu


def _map(n, nq, seed):
    """Half the photons on a floor, with a tight cluster and two stacks; half
    the queries on it, some outside the map and some not numbers."""
    rng = np.random.default_rng(seed)
    pos = rng.random((3, n), dtype=np.float32)
    q = rng.random((3, nq), dtype=np.float32)
    pos[1, : n // 2] = 0.0
    pos[0, : n // 8] = 0.3 + 0.002 * pos[0, : n // 8]
    pos[2, : n // 8] = 0.6 + 0.002 * pos[2, : n // 8]
    pos[:, 500:540] = pos[:, 500:501]
    pos[:, 1000:1700] = pos[:, 1000:1001]
    q[1, : nq // 2] = 0.0
    q[:, : nq // 10] = q[:, : nq // 10] * 2.0 - 0.5
    q[:, nq // 2: nq // 2 + nq // 20] = pos[:, rng.integers(0, n, nq // 20)]
    q[rng.integers(0, 3, nq // 50), rng.integers(0, nq, nq // 50)] = np.nan
    q[:, 0] = pos[:, 500]
    if nq > 2:
        q[:, 1], q[:, 2] = pos[:, 1000], (np.inf, -np.inf, 0.5)
    return pos, q


@pytest.mark.parametrize("n,nq,r,k", [
    (33_000, 1, 0.05, 64),
    (33_000, 3, 0.05, 7),
    (33_000, 3, 0.05, 8),
    (33_000, 3072, 0.05, 7),
    (33_000, 3073, 0.05, 7),
    (33_000, 1001, 0.05, 32),
    (33_000, 1001, 0.05, 33),
    (33_000, 1001, 0.1, 128),
    (33_000, 1001, 0.1, 129),
    (33_000, 6144, 0.1, 64),
    (33_000, 6145, 0.1, 64),
    (20_000, 49_151, 0.05, 50),
    (20_000, 49_152, 0.05, 50),
    (20_000, 98_303, 0.05, 30),
    (20_000, 98_304, 0.05, 30),
    (20_000, 20_001, 0.1, 256),
    (300_000, 301, 3.0, 256),   # everything in reach
    (300_000, 6201, 0.6, 200),
    (300_000, 777, 0.4, 100),
])
def test_lists(ctx, n, nq, r, k):
    pos, q = _map(n, nq, n + nq + k)
    ph = np.ones((9, n), np.float32)
    ph[0:3] = pos
    gi, gd, gc = ctx.kdtree_knn(ctx.kdtree_build(ph), q, r, k)
    ctx.sync()
    ni, npl = O.kdtree_build(pos)
    oi, od, oc = O.kdtree_knn(pos, ni, npl, q, r, k)
    assert np.array_equal(gc.cpu().numpy().view(np.uint32), oc)
    assert np.array_equal(gi.cpu().numpy().view(np.uint32), oi)
    assert np.array_equal(gd.cpu().numpy().view(np.uint32), od.view(np.uint32))


def test_open_search_of_a_deep_tree(ctx):
    """24 levels with every photon in one place, k for the smallest stack: all
    nodes are opened. Subtrees of five levels, taken whatever room was left, filled
    the stack past its end (613 entries of 608, counted on the CPU). The nearest are the first."""
    import torch

    n, nq, k = 8_400_000, 2, 64
    ph = torch.full((9, n), 0.25, device="cuda")
    q = np.array([[0.25, 0.3], [0.25, 0.25], [0.25, 0.25]], np.float32)
    gi, gd, gc = ctx.kdtree_knn(ctx.kdtree_build(ph), q, 0.5, k)
    ctx.sync()
    d = (np.float32(0.25) - q[0]) * (np.float32(0.25) - q[0])
    assert gc.tolist() == [k] * nq
    assert gi.tolist() == [list(range(k))] * nq
    for i in range(nq):
        assert len(set(gd[i].tolist())) == 1 and abs(float(gd[i, 0]) - np.sqrt(d[i])) <= 1e-6


@pytest.mark.parametrize("k", [1, 50])
def test_queries_that_are_not_numbers_cost_nothing(ctx, k):
    """They walked the whole tree, 300k photons' in 83 ms; the others' walk
    takes tens of microseconds."""
    import torch

    n, nq, r = 300_000, 256, 0.01
    pos, q = _map(n, nq, 9)
    ph = np.ones((9, n), np.float32)
    ph[0:3] = pos
    tree = ctx.kdtree_build(ph)
    qs = [torch.from_numpy(np.nan_to_num(q, nan=0.5)).cuda(), torch.full((3, nq), float("nan"), device="cuda")]
    best = [1e9, 1e9]
    for _ in range(5):
        for i in range(2):
            ctx.sync()
            t0 = time.perf_counter()
            out = ctx.kdtree_knn(tree, qs[i], r, k)
            ctx.sync()
            best[i] = min(best[i], time.perf_counter() - t0)
    assert int(out[2].abs().sum()) == 0
    assert best[1] < 3 * best[0], best
