"""The streaming gather with one query a wave (launches that do not fill the
chip), whose set-up is worked for one query alone: every row count that it
distinguishes (9, 25 and 49 rows of the first box; more than 64 and Morton: rows
taken 64 at a time), the inner box, the processing orders, the smallest launches,
queries outside the map and ones that are not numbers. Lists are exact against
the oracle; an estimate has the same bits as in a launch that gives a wave
several queries, and is within 1e-5 of the oracle's FP64 value over the same kept
set (a sum of at most k positive FP32 terms, each within a few ulps)."""
import numpy as np
import pytest

import pm355
import pyoracle as O
from pm355.workloads import gather_microbench

pytestmark = pytest.mark.gpu

R, MANY = 0.03, 8 * 49152  # MANY: several queries a wave, whatever the map


@pytest.fixture(scope="module")
def inputs():
    ph, q, qn, aabb = gather_microbench(seed=32, n_photons=60_000, n_queries=2003, n_clusters=6)
    ph[0:3, 1000:1040] = np.array([[0.5], [0.0], [0.5]], np.float32)
    ph[0:3, 2000:2700] = np.array([[0.25], [0.0], [0.75]], np.float32)
    q[:, 0] = (0.5, 0.0, 0.5)
    q[:, 1] = (0.2501, 0.0, 0.7502)
    q[:, 2] = (1.7, -0.4, 0.5)  # outside the box, nothing in reach
    q[:, 3] = (np.nan, 0.2, 0.3)
    q[:, 4] = (0.0, 1.0, 1.0)
    return ph, q, qn, aabb


@pytest.mark.parametrize("nq", [1, 2, 2003])
@pytest.mark.parametrize("cell,layout,flags,k", [
    (1.0, 0, 0, 64),
    (1.0, 0, pm355.KNN_SORT_QUERIES, 1),
    (1.0, 0, pm355.KNN_XCD_CONTIGUOUS, 256),
    (1.0, 0, pm355.KNN_NO_XCD_REMAP, 20),
    (0.5, 0, 0, 50),
    (0.34, 0, pm355.KNN_SORT_QUERIES, 200),
    (0.25, 0, 0, 50),
    (0.4, 0, pm355.KNN_INNER_BOX, 16),
    (0.2, 0, pm355.KNN_INNER_BOX | pm355.KNN_SORT_QUERIES, 64),
    (0.08, 0, pm355.KNN_INNER_BOX, 30),
    (1.0, 1, 0, 50),
    (0.5, 1, pm355.KNN_INNER_BOX, 50),
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
    many = ctx.gather_radiance(g, np.tile(q, (1, -(-MANY // nq))), np.tile(qn, (1, -(-MANY // nq))), R, k, flags)
    ctx.sync()
    assert np.array_equal(cnt.cpu().numpy().view(np.uint32), oc)
    assert np.array_equal(idx.cpu().numpy().view(np.uint32), oi)
    assert np.array_equal(dist.cpu().numpy(), od)
    assert np.array_equal(rcnt.cpu().numpy().view(np.uint32), oc)
    got = rgb.cpu().numpy()
    assert np.array_equal(got.view(np.uint32), many[:, :nq].cpu().numpy().view(np.uint32))
    nan = np.isnan(o64)  # (k photons at the query itself: the filter radius is 0 and both are NaN)
    assert np.array_equal(np.isnan(got), nan)
    assert np.all(np.abs(got.astype(np.float64) - o64)[~nan] <= 1e-5 * np.abs(o64)[~nan])
    g.close()
