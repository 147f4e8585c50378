"""The radiance estimate's error against its value in 64 bits (distances, weights
and sums from the FP32 positions, over the neighbours that the FP32 order keeps).

Bounds, with u = 2^-24: a sum of k <= 2048 positive terms by 64 lanes and a
reduction has at most 32 + 6 roundings in a chain, the weights, the filter radius
and the factor before the sum some ten more, so no value is off by more than 50 u =
3.0e-6. Roundings are spread like random ones of rms u / sqrt(3) = 3.4e-8: the
lanes' partial sums contribute 1.4e-8 (32 growing sums, the mean of 64 lanes), the
reduction 4.8e-8, the filter radius, which enters squared, 6.8e-8, the factor's
reciprocal and products 6.2e-8; together 1.05e-7 rms, of which a fifth more is let
pass."""
import numpy as np
import pytest

import pyoracle as O
from pm355.workloads import gather_microbench

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,r,k", [
    (200_000, 0.03, 64),
    (200_000, 0.05, 200),
    (200_000, 0.06, 300),
    (200_000, 0.08, 512),
    (200_000, 0.08, 513),
    (200_000, 0.1, 1000),
    (200_000, 0.15, 2000),
    (40_000, 0.1, 2000),   # everything in reach kept
])
def test_error(ctx, n, r, k):
    ph, q, qn, aabb = gather_microbench(seed=34, n_photons=n, n_queries=3000, n_clusters=16)
    g = ctx.grid_build(ph, aabb, cell_size=r)
    og = O.OracleGrid(ph, aabb, cell_size=r)
    rgb = ctx.gather_radiance(g, q, qn, r, k)
    oi, _, oc = og.knn(q, r, k)
    ctx.sync()
    got = rgb.cpu().numpy().astype(np.float64)
    p = og.photons.astype(np.float64)
    errs = []
    for j in range(q.shape[1]):
        m = int(oc[j])
        if m == 0:
            assert np.all(got[:, j] == 0)
            continue
        s = p[:, oi[j, :m]]
        d2 = ((s[0:3] - q[:, j:j + 1].astype(np.float64)) ** 2).sum(0)
        w = 1.818 * (1 - (1 - np.exp(-1.953 * d2 / (2 * d2.max()))) / (1 - np.exp(-1.953)))
        c = qn[:, j:j + 1] * -s[6:9].astype(np.float32)
        cos = (c[0] + c[1]) + c[2]  # (the reference's FP32 test)
        want = (s[3:6] * np.where(cos > 0, w, 0.0)).sum(1) / (np.float64(np.float32(np.pi)) * d2.max())
        lit = want > 0
        errs.append(((got[:, j] - want)[lit] / want[lit]))
    errs = np.abs(np.concatenate(errs))
    assert errs.max() <= 50 * 2.0 ** -24
    assert np.sqrt((errs ** 2).mean()) <= 1.2 * 1.05e-7
    g.close()
