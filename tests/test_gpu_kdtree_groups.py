"""kd-tree lists with two queries a wave, a group of lanes each: waves of one
query a group and of several (the ball then sized from the wave's earlier
queries), a last wave with fewer, the buffer sizes' edges in k, and maps where
the first ball holds none, too few, enough or far too many photons. Lists are
exact against the oracle."""
import numpy as np
import pytest

import pyoracle as O

pytestmark = pytest.mark.gpu

SPLIT = 2 * 12288  # queries above which a group takes a second one


@pytest.mark.parametrize("n,nq,r,k", [
    (1, 3, 0.1, 1),
    (20_000, 2 * SPLIT - 1, 0.03, 1),
    (20_000, 2 * SPLIT + 1, 0.05, 64),
    (20_000, 2 * SPLIT + 1, 0.05, 65),
    (20_000, 3 * SPLIT + 5, 0.03, 10),
    (20_000, 2 * SPLIT + 3, 0.07, 128),
    (20_000, 2 * SPLIT + 3, 0.07, 129),
    (20_000, 2 * SPLIT + 3, 0.12, 256),
    (33_000, 9 * SPLIT + 1, 0.02, 20),
    (33_000, 2 * SPLIT + 1, 0.0, 20),
    (33_000, 777, 1e-23, 40),  # a denormal threshold
    (33_000, 777, 3.0, 200),   # everything in reach
])
def test_lists(ctx, n, nq, r, k):
    rng = np.random.default_rng(n + nq + k)
    pos = rng.random((3, n), dtype=np.float32)
    q = rng.random((3, nq), dtype=np.float32)
    if n > 1:
        pos[1, : n // 2] = 0.0  # half on a floor, with a tight cluster and two stacks
        pos[0, : n // 8] = 0.3 + 0.002 * pos[0, : n // 8]
        pos[2, : n // 8] = 0.6 + 0.002 * pos[2, : n // 8]
        pos[:, 500:540] = pos[:, 500:501]
        pos[:, 1000:1700] = pos[:, 1000:1001]
        q[1, : nq // 2] = 0.0
        q[:, : nq // 20] = pos[:, rng.integers(0, n, nq // 20)]
        q[:, 0], q[:, 1], q[:, 2] = pos[:, 500], pos[:, 1000], (1.9, -0.5, 0.5)
        rng.shuffle(q, axis=1)
    ph = np.ones((9, n), np.float32)
    ph[0:3] = pos
    gi, gd, gc = ctx.kdtree_knn(ctx.kdtree_build(ph), q, r, k)
    ctx.sync()
    ni, npl = O.kdtree_build(pos)
    oi, od, oc = O.kdtree_knn(pos, ni, npl, q, r, k)
    assert np.array_equal(gc.cpu().numpy().view(np.uint32), oc)
    assert np.array_equal(gi.cpu().numpy().view(np.uint32), oi)
    assert np.array_equal(gd.cpu().numpy().view(np.uint32), od.view(np.uint32))
