"""The streaming gather's wave split: several queries per wave (set-up worked
side by side in the lanes), every row count the split distinguishes (9, 25 and
49 rows of the first box; more than 64 and Morton: rows taken 64 at a time),
query counts around the split's edges and a last wave with fewer queries.
Lists are exact against the oracle; the estimate is within 1e-5 of the
oracle's FP64 value over the same kept set (a sum of at most k positive FP32
terms, each within a few ulps)."""
import numpy as np
import pytest

import pm355
import pyoracle as O
from pm355.workloads import gather_microbench

pytestmark = pytest.mark.gpu

FILL = 16384  # waves below which a wave takes a single query
R = 0.03


@pytest.fixture(scope="module")
def inputs():
    ph, q, qn, aabb = gather_microbench(seed=31, n_photons=60_000, n_queries=7 * FILL + 5, n_clusters=6)
    # equal keys: a point with more photons than a crossing bin may hold, and
    # one with more than the key buffer
    ph[0:3, 1000:1040] = np.array([[0.5], [0.0], [0.5]], np.float32)
    ph[0:3, 2000:2700] = np.array([[0.25], [0.0], [0.75]], np.float32)
    q[:, 0] = (0.5, 0.0, 0.5)
    q[:, 1] = (0.25, 0.0, 0.75)
    q[:, 2] = (0.2501, 0.0, 0.7502)
    q[:, 3] = (1.7, -0.4, 0.5)  # outside the box, nothing in reach
    return ph, q, qn, aabb


@pytest.mark.parametrize("cell,layout,flags,nq,k", [
    (1.0, 0, 0, 1, 64),
    (1.0, 0, pm355.KNN_SORT_QUERIES, 2 * FILL - 1, 20),
    (1.0, 0, pm355.KNN_SORT_QUERIES, 2 * FILL, 1),
    (1.0, 0, pm355.KNN_SORT_QUERIES, 7 * FILL + 5, 64),
    (1.0, 0, 0, 7 * FILL + 5, 200),
    (0.4, 0, pm355.KNN_INNER_BOX | pm355.KNN_SORT_QUERIES, 7 * FILL + 1, 16),
    (0.5, 0, 0, 2 * FILL + 7, 50),
    (0.34, 0, 0, 2 * FILL + 3, 50),
    (0.25, 0, 0, 2 * FILL + 3, 50),
    (0.2, 0, pm355.KNN_INNER_BOX, 2 * FILL + 3, 30),
    (1.0, 1, pm355.KNN_SORT_QUERIES, 2 * FILL + 3, 50),
    (1.0, 0, pm355.KNN_LARGE_BUFFER | pm355.KNN_SORT_QUERIES, 3 * FILL + 3, 100),
    (1.0, 0, pm355.KNN_XCD_CONTIGUOUS, 3 * FILL + 3, 100),
    (1.0, 0, pm355.KNN_NO_XCD_REMAP, 3 * FILL + 3, 100),
])
def test_lists_and_estimate(ctx, inputs, cell, layout, flags, nq, k):
    ph, q, qn, aabb = inputs
    q, qn = np.ascontiguousarray(q[:, :nq]), np.ascontiguousarray(qn[:, :nq])
    g = ctx.grid_build(ph, aabb, cell_size=R * cell, layout=layout)
    og = O.OracleGrid(ph, aabb, cell_size=R * cell, layout=layout)
    oi, od, oc = og.knn(q, R, k)
    _, o64 = O.radiance(oi, od, oc, og.photons, qn, k)
    idx, dist, cnt = ctx.knn(g, q, R, k, flags)
    rgb, rcnt = ctx.gather_radiance(g, q, qn, R, k, flags, want_count=True)
    both = ctx.gather_batch([(g, q, qn, R, k), (g, q[:, :777].copy(), qn[:, :777].copy(), R, k)], flags,
                            want_knn=True)
    few = ctx.gather_radiance(g, q[:, :777].copy(), qn[:, :777].copy(), R, k, flags)
    ctx.sync()
    # a query's estimate does not depend on the launch it is part of
    assert np.array_equal(few.cpu().numpy().view(np.uint32), rgb[:, :777].cpu().numpy().view(np.uint32))
    for i, d, c in ((idx, dist, cnt), (both[0]["idx"], both[0]["dist"], both[0]["count"])):
        assert np.array_equal(c.cpu().numpy().view(np.uint32), oc)
        assert np.array_equal(i.cpu().numpy().view(np.uint32), oi)
        assert np.array_equal(d.cpu().numpy(), od)
    assert np.array_equal(rcnt.cpu().numpy().view(np.uint32), oc)
    assert np.array_equal(both[1]["idx"].cpu().numpy().view(np.uint32), oi[:777])
    for got, want in ((rgb, o64), (both[0]["rgb"], o64), (both[1]["rgb"], o64[:, :777])):
        got = got.cpu().numpy().astype(np.float64)
        # (k photons at the query itself: the filter radius is 0 and both are NaN)
        nan = np.isnan(want)
        assert np.array_equal(np.isnan(got), nan)
        assert np.all(np.abs(got - want)[~nan] <= 1e-5 * np.abs(want)[~nan])
    g.close()


# (the mid kernel up to k = 512, the wide one above: few enough in reach, more
# than expected, many more; a point's equal distances fill a crossing bin)
@pytest.mark.parametrize("r,cell,flags,nq,k", [
    (0.15, 1.0, pm355.KNN_SORT_QUERIES, 2 * FILL + 3, 300),
    (0.2, 0.5, 0, 3001, 512),
    (0.15, 1.0, pm355.KNN_SORT_QUERIES, 2 * FILL + 3, 513),
    (0.2, 0.4, pm355.KNN_INNER_BOX, 3001, 600),
    (0.25, 1.0, 0, 3001, 700),
    (0.3, 1.0, pm355.KNN_SORT_QUERIES, 2 * FILL + 1, 2000),
    (0.3, 0.2, 0, 777, 2048),
])
def test_large_k_estimate(ctx, inputs, r, cell, flags, nq, k):
    ph, q, qn, aabb = inputs
    q, qn = np.ascontiguousarray(q[:, :nq]), np.ascontiguousarray(qn[:, :nq])
    g = ctx.grid_build(ph, aabb, cell_size=r * cell)
    og = O.OracleGrid(ph, aabb, cell_size=r * cell)
    oi, od, oc = og.knn(q, r, k)
    _, o64 = O.radiance(oi, od, oc, og.photons, qn, k)
    rgb, cnt = ctx.gather_radiance(g, q, qn, r, k, flags, want_count=True)
    few = ctx.gather_radiance(g, q[:, :77].copy(), qn[:, :77].copy(), r, k, flags)
    ctx.sync()
    assert np.array_equal(cnt.cpu().numpy().view(np.uint32), oc)
    assert np.array_equal(few.cpu().numpy().view(np.uint32), rgb[:, :77].cpu().numpy().view(np.uint32))
    got = rgb.cpu().numpy().astype(np.float64)
    nan = np.isnan(o64)  # (k photons at the query itself)
    assert np.array_equal(np.isnan(got), nan)
    assert np.all(np.abs(got - o64)[~nan] <= 1e-5 * np.abs(o64)[~nan])
    g.close()


# Lists on a map with a density step: beside it the first walk's guess from the
# candidate count falls short, by little (a second bound from the keys it
# found), by a lot or with no key at all (the radius).
@pytest.mark.parametrize("sparse,k", [(0, 50), (200, 50), (2000, 50), (20_000, 10), (20_000, 200)])
def test_lists_beside_a_density_step(ctx, sparse, k):
    rng = np.random.default_rng(41)
    nq = 2 * FILL + 1
    pos = rng.random((3, 60_000 + sparse), dtype=np.float32)
    pos[0, :60_000] *= 0.5  # crowded below x = 0.5
    pos[0, 60_000:] = 0.5 + 0.5 * pos[0, 60_000:]
    pos[1] = 0.0
    ph = np.concatenate([pos, np.full_like(pos, 1e-6), np.full_like(pos, -0.57)], 0)
    q = rng.random((3, nq), dtype=np.float32)
    q[0] = 0.45 + 0.1 * q[0]
    q[1] = 0.0
    aabb = (0.0, 0.0, 0.0, 1.0, 1.0, 1.0)
    g = ctx.grid_build(ph, aabb, cell_size=R)
    oi, od, oc = O.OracleGrid(ph, aabb, cell_size=R).knn(q, R, k)
    idx, dist, cnt = ctx.knn(g, q, R, k, pm355.KNN_SORT_QUERIES)
    ctx.sync()
    assert np.array_equal(cnt.cpu().numpy().view(np.uint32), oc)
    assert np.array_equal(idx.cpu().numpy().view(np.uint32), oi)
    assert np.array_equal(dist.cpu().numpy(), od)
    g.close()


# Lists above k = 256: the 768-key buffer's stream, one query a wave (its first
# walk to a guessed bound), two, a guess off (inner box), and the buffered
# kernel from k = 513 on.
@pytest.mark.parametrize("r,cell,flags,nq,k", [
    (0.15, 1.0, 0, 777, 257),
    (0.15, 1.0, pm355.KNN_SORT_QUERIES, 3001, 300),
    (0.2, 0.5, 0, 777, 512),
    (0.2, 0.4, pm355.KNN_INNER_BOX, 777, 400),
    (0.1, 1.0, pm355.KNN_SORT_QUERIES, 8 * FILL + 1, 257),
    (0.3, 0.2, 0, 300, 512),
    (0.2, 1.0, 0, 777, 513),
])
def test_large_k_lists(ctx, inputs, r, cell, flags, nq, k):
    ph, q, qn, aabb = inputs
    q, qn = np.tile(q, (1, 2))[:, :nq].copy(), np.tile(qn, (1, 2))[:, :nq].copy()
    g = ctx.grid_build(ph, aabb, cell_size=r * cell)
    og = O.OracleGrid(ph, aabb, cell_size=r * cell)
    oi, od, oc = og.knn(q, r, k)
    idx, dist, cnt = ctx.knn(g, q, r, k, flags)
    both = ctx.gather_batch([(g, q, qn, r, k)], flags, want_knn=True)[0]
    ctx.sync()
    for i, d, c in ((idx, dist, cnt), (both["idx"], both["dist"], both["count"])):
        assert np.array_equal(c.cpu().numpy().view(np.uint32), oc)
        assert np.array_equal(i.cpu().numpy().view(np.uint32), oi)
        assert np.array_equal(d.cpu().numpy(), od)
    _, o64 = O.radiance(oi, od, oc, og.photons, qn, k)
    got = both["rgb"].cpu().numpy().astype(np.float64)
    nan = np.isnan(o64)  # (k photons at the query itself)
    assert np.array_equal(np.isnan(got), nan)
    assert np.all(np.abs(got - o64)[~nan] <= 1e-5 * np.abs(o64)[~nan])
    g.close()
