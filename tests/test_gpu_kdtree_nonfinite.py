"""kd-tree builds over coordinates that are NaN, infinite or huge: the tree of the
total order the sorts work in (-inf < numbers < inf < NaN, ties by photon
index), with every photon in one node. The levels finished in LDS used to compare
coordinates; where all of a subtree's were NaN its medians came from memory that
nothing had written. Checked against the same build in numpy; the lists hold no photon
of a NaN coordinate."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _build(pos):
    """(node_idx, node_plane) by recursion over the three orders."""
    n = pos.shape[1]
    u = (pos + np.float32(0)).view(np.uint32).astype(np.int64)
    key = np.where(u & 0x80000000, 0xFFFFFFFF - u, u | 0x80000000)
    rank = np.empty((3, n), np.int64)
    orders = []
    for a in range(3):
        o = np.argsort(key[a], kind="stable")
        rank[a, o] = np.arange(n)
        orders.append(o)
    cap = 1
    while cap - 1 < n:
        cap *= 2
    idx, plane = np.full(cap - 1, 0xFFFFFFFF, np.uint32), np.full(cap - 1, -1, np.int8)
    todo = [(0, orders)]
    while todo:
        node, o = todo.pop()
        d = [abs(pos[a, o[a][-1]] - pos[a, o[a][0]]) for a in range(3)]
        p, mx = (1, d[1]) if d[1] > d[0] else (0, d[0])
        if d[2] > mx:
            p = 2
        m = o[p][len(o[p]) // 2]
        idx[node], plane[node] = m, p
        left = [x[rank[p, x] < rank[p, m]] for x in o]
        right = [x[rank[p, x] > rank[p, m]] for x in o]
        if len(left[0]):
            todo.append((2 * node + 1, left))
        if len(right[0]):
            todo.append((2 * node + 2, right))
    return idx, plane


@pytest.mark.parametrize("n,share,axis", [
    (7, 0.3, None),
    (500, 0.02, None),
    (1024, 0.5, None),
    (1025, 0.02, None),
    (3000, 1.0, 0),      # no number on an axis
    (3000, 1.0, 2),
    (40_000, 0.02, None),
    (40_000, 0.2, 0),    # whole subtrees of NaN
])
def test_build(ctx, n, share, axis):
    rng = np.random.default_rng(n)
    pos = rng.random((3, n), dtype=np.float32)
    bad = rng.random((3, n)) < share
    if axis is not None:
        bad[[a for a in range(3) if a != axis]] = False
    odd = np.array([np.nan, np.inf, -np.inf, 1e30, -1e30] if axis is None else [np.nan], np.float32)
    pos[bad] = rng.choice(odd, int(bad.sum()))
    ph = np.ones((9, n), np.float32)
    ph[0:3] = pos
    tree = ctx.kdtree_build(ph)
    gi, gp = (np.asarray(x) for x in tree.to_host()[:2])
    with np.errstate(invalid="ignore", over="ignore"):
        ei, ep = _build(pos)
    assert np.array_equal(gi.view(np.uint32), ei)
    assert np.array_equal(gp.view(np.int8), ep)
    used = ei[ei != 0xFFFFFFFF]
    assert np.array_equal(np.sort(used), np.arange(n))
    q = rng.random((3, 64), dtype=np.float32)
    idx, dist, cnt = (x.cpu().numpy() for x in ctx.kdtree_knn(tree, q, 0.3, 10))
    for i in range(64):
        got = idx[i, : cnt[i]].astype(np.int64)
        assert np.isfinite(pos[:, got]).all() and (dist[i, : cnt[i]] <= 0.3).all()
