"""Batches whose job tables travel as kernel arguments (one launch, several)
and batches whose tables are copied, back to back without a synchronisation
between them: each equals its single-grid gathers."""
import numpy as np
import pytest

import pm355
from pm355.workloads import gather_microbench

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [(1, 14, 15), (40, 3, 70), (300, 2, 64)])
def test_back_to_back(ctx, counts):
    ph, q, qn, aabb = gather_microbench(seed=5, n_photons=20_000, n_queries=400, n_clusters=4)
    g = ctx.grid_build(ph, aabb, cell_size=0.05)
    q, qn = (x.reshape(3, -1) for x in (q, qn))
    outs = []
    for n in counts:
        jobs = [(g, np.ascontiguousarray(q[:, j % 97:j % 97 + 50]), np.ascontiguousarray(qn[:, j % 97:j % 97 + 50]),
                 0.05, 10 + j % 30) for j in range(n)]
        outs.append((jobs, ctx.gather_batch(jobs, pm355.KNN_SORT_QUERIES)))
    ctx.sync()
    for jobs, out in outs:
        for (grid, qq, nn, r, k), o in zip(jobs, out):
            want = ctx.gather_radiance(grid, qq, nn, r, k)
            ctx.sync()
            assert np.array_equal(o["rgb"].cpu().numpy().view(np.uint32), want.cpu().numpy().view(np.uint32))
    g.close()
