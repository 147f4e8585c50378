"""The sizing rule's density test at its edge: the fullest cell holds exactly
5 x desired photons (the cells stay) or one more (they shrink), with as many
cells as are counted in LDS and with more, for counts from one workgroup and
from several, dense photons first, last and spread in the input."""
import numpy as np
import pytest

import pyoracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("where", ["first", "last", "spread"])
@pytest.mark.parametrize("n,desired", [(5, 5), (3000, 50), (100_000, 5), (60_000, 1000), (78_125, 5), (300_000, 10)])
def test_density_edge(ctx, n, desired, where):
    rng = np.random.default_rng(n + desired)
    dims = []
    for extra in (0, 1):
        dense = min(5 * desired + extra, n)
        cell = 1.0 / np.cbrt(-(-n // desired))  # the reference's size, and whole cells a side
        g = max(1, int(1.0 / cell + 1e-4))
        at = (1 + np.arange(n) % max(1, g ** 3 - 1)) % g ** 3  # every cell but the first alike
        pos = (np.stack([at % g, at // g % g, at // g ** 2]) + 0.5) * cell
        sel = {"first": np.arange(dense), "last": np.arange(n - dense, n),
               "spread": rng.permutation(n)[:dense]}[where]
        pos[:, sel] = 0.25 * cell
        ph = np.ones((9, n), np.float32)
        ph[0:3] = pos
        grid = ctx.grid_build(ph, (0, 0, 0, 1, 1, 1), desired=desired)
        og = O.OracleGrid(ph, (0, 0, 0, 1, 1, 1), cell_size=0.0, desired=desired)
        dims.append(tuple(og.dims))
        assert tuple(grid.info.dims) == dims[-1]
        starts, sizes, _, perm = grid.to_host()
        assert np.array_equal(starts, og.starts) and np.array_equal(sizes, og.counts)
        assert np.array_equal(perm, og.perm)
        grid.close()
    if n > 5 * desired:
        assert dims[0] != dims[1]
