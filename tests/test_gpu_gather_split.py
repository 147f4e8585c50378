"""The gather's rule for several queries a wave, on both sides of its lines:
estimates of sorted and unsorted launches, on sparse and on crowded maps, with the
inner box, and above k = 256 (131072 queries on: the guessed bound of the wide
kernel, its second walk where the guess falls short, and the k-th key below a
lowered bound). A few hundred distinct queries are repeated to the launch's size;
each of their estimates must have the bits of a launch that gives every query a
wave, and lie within 1e-5 of the oracle's FP64 value over the same kept set (a sum
of at most k positive FP32 terms, each within a few ulps)."""
import time

import numpy as np
import pytest

import pm355
import pyoracle as O
from pm355.workloads import gather_inputs_device, gather_microbench

pytestmark = pytest.mark.gpu

# waves below which a wave takes a single query (twice as many queries: two)
FILL, FILL_UNEVEN, FILL_LARGE = 16384, 49152, 65536
SORT, INNER = pm355.KNN_SORT_QUERIES, pm355.KNN_INNER_BOX


def _even(n, nq):
    ph, q, qn, aabb = gather_microbench(seed=33, n_photons=n, n_queries=nq, n_clusters=6)
    ph[0:3, 1000:1040] = np.array([[0.5], [0.0], [0.5]], np.float32)  # equal keys
    ph[0:3, 2000:2700] = np.array([[0.25], [0.0], [0.75]], np.float32)
    q[:, 0], q[:, 1], q[:, 2] = (0.5, 0.0, 0.5), (0.2501, 0.0, 0.7502), (1.7, -0.4, 0.5)
    return ph, q, qn, aabb


def _step(n, nq):
    """A floor that is crowded below x = 0.5 and sparse beyond: beside the step a
    guess from the rows' count falls short."""
    rng = np.random.default_rng(43)
    pos = rng.random((3, n), dtype=np.float32)
    pos[0, : n - n // 30] *= 0.5
    pos[0, n - n // 30:] = 0.5 + 0.5 * pos[0, n - n // 30:]
    pos[1] = 0.0
    ph = np.concatenate([pos, np.full_like(pos, 1e-6), np.full_like(pos, -0.57)], 0)
    q = rng.random((3, nq), dtype=np.float32)
    q[0] = 0.35 + 0.3 * q[0]
    q[1] = 0.0
    qn = np.zeros_like(q)
    qn[1] = 1.0
    return ph, q, qn, (0.0, 0.0, 0.0, 1.0, 1.0, 1.0)


def _check(ctx, make, n, nd, nq, r, cell, flags, k):
    ph, q, qn, aabb = make(n, nd)
    g = ctx.grid_build(ph, aabb, cell_size=r * cell)
    og = O.OracleGrid(ph, aabb, cell_size=r * cell)
    oi, od, oc = og.knn(q, r, k)
    _, o64 = O.radiance(oi, od, oc, og.photons, qn, k)
    reps = -(-nq // nd)
    big = [np.ascontiguousarray(np.tile(a, (1, reps))[:, :nq]) for a in (q, qn)]
    rgb, cnt = ctx.gather_radiance(g, *big, r, k, flags, want_count=True)
    few = ctx.gather_radiance(g, q, qn, r, k, flags)
    ctx.sync()
    rgb, cnt, few = rgb.cpu().numpy(), cnt.cpu().numpy().view(np.uint32), few.cpu().numpy()
    assert np.array_equal(cnt, np.tile(oc, reps)[:nq])
    assert np.array_equal(rgb.view(np.uint32), np.tile(few, (1, reps))[:, :nq].view(np.uint32))
    nan = np.isnan(o64)  # (k photons at the query itself)
    assert np.array_equal(np.isnan(few), nan)
    assert np.all(np.abs(few.astype(np.float64) - o64)[~nan] <= 1e-5 * np.abs(o64)[~nan])
    g.close()


@pytest.mark.parametrize("make", [_even, _step])
@pytest.mark.parametrize("n,nq,r,cell,flags,k", [
    (60_000, 2 * FILL, 0.03, 1.0, SORT, 20),                 # two a wave
    (60_000, 2 * FILL + 2000, 0.03, 1.0, SORT, 64),          # a round just over: one
    (60_000, 3 * FILL + 5, 0.03, 1.0, SORT, 64),
    (60_000, 6 * FILL + 700, 0.03, 1.0, SORT, 100),          # just over: as many as fit
    (60_000, 7 * FILL + 5000, 0.03, 1.0, SORT, 200),
    (60_000, 3 * FILL + 5, 0.1, 1.0, 0, 16),                 # unsorted, the guess saves much
    (60_000, 2 * FILL_UNEVEN - 1, 0.03, 1.0, 0, 64),
    (60_000, 2 * FILL_UNEVEN + 7000, 0.03, 1.0, 0, 64),
    (60_000, 2 * FILL_UNEVEN - 1, 0.03, 0.4, INNER | SORT, 16),
    (60_000, 2 * FILL_UNEVEN + 7000, 0.03, 0.4, INNER | SORT, 16),
    (60_000, 2 * FILL_UNEVEN + 7000, 0.03, 0.2, INNER, 16),
    (300_000, 2 * FILL_UNEVEN - 1, 0.1, 1.0, SORT, 64),      # crowded
    (300_000, 2 * FILL_UNEVEN + 7000, 0.1, 1.0, SORT, 64),
    (60_000, 3 * FILL_UNEVEN, 0.03, 0.5, 0, 50),             # 25 rows
    (60_000, 3 * FILL_UNEVEN, 0.03, 0.34, 0, 50),            # 49: one a wave
])
def test_estimates(ctx, make, n, nq, r, cell, flags, k):
    _check(ctx, make, n, 499, nq, r, cell, flags, k)


@pytest.mark.parametrize("make", [_even, _step])
@pytest.mark.parametrize("nq,r,cell,flags,k", [
    (2 * FILL_LARGE + 1, 0.1, 1.0, SORT, 300),
    (3 * FILL_LARGE + 1, 0.15, 1.0, 0, 512),
    (2 * FILL_LARGE + 1, 0.15, 0.5, SORT, 400),
    (2 * FILL_LARGE + 1, 0.15, 1.0, SORT, 513),
    (5 * FILL_LARGE + 1, 0.12, 1.0, SORT, 600),
    (2 * FILL_LARGE + 1, 0.2, 0.5, 0, 1000),
    (2 * FILL_LARGE + 1, 0.3, 1.0, SORT, 2000),
    (2 * FILL_LARGE + 1, 0.3, 0.5, SORT, 2048),
])
def test_large_k_estimates(ctx, make, nq, r, cell, flags, k):
    _check(ctx, make, 60_000, 307, nq, r, cell, flags, k)


def test_crowded_estimates_cost_what_lists_do(ctx):
    """65536 sorted queries in 3.78M photons within 0.047: with several such
    queries a wave the estimate took 1.8 times the lists' time, with one 1.1."""
    ph, q, qn, aabb = gather_inputs_device(3_783_000, 65_536, 5, ctx.device)
    g = ctx.grid_build(ph, aabb, cell_size=0.047)
    best = {}
    for _ in range(6):
        for name, run in (("rgb", lambda: ctx.gather_radiance(g, q, qn, 0.047, 64, SORT)),
                          ("lists", lambda: ctx.knn(g, q, 0.047, 64, SORT))):
            ctx.sync()
            t0 = time.perf_counter()
            run()
            ctx.sync()
            best[name] = min(best.get(name, 1e9), time.perf_counter() - t0)
    g.close()
    assert best["rgb"] < 1.45 * best["lists"], best
