"""The key sort's digits: key widths of one to three passes, at and beside the
widths where a pass is added, digits of 9 bits and fewer, counts at the edges
of its tiles of 4096 keys. A grid's permutation is exact against the oracle:
photons of a cell stay in input order."""
import numpy as np
import pytest

import pyoracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [2, 8, 255, 512, 513, 1 << 17, 1 << 18, (1 << 18) + 1, 1 << 19, (1 << 21) + 3])
@pytest.mark.parametrize("n", [1, 4095, 4097, 20_000])
def test_permutation(ctx, cells, n):
    rng = np.random.default_rng(cells + n)
    # a row of cells along z (at most a million), several rows for more
    rows = 1 + cells // (1 << 19)
    per = cells // rows
    aabb = (0.0, 0.0, 0.0, 1.0, float(rows), float(per))
    ph = rng.random((9, n), dtype=np.float32)
    ph[1] *= rows
    ph[2] = np.minimum(ph[2] * ph[2] * per, np.float32(per) * np.float32(0.9999))  # crowded at one end
    ph[2, : n // 4] = 0.5
    g = ctx.grid_build(ph, aabb, cell_size=1.0)
    og = O.OracleGrid(ph, aabb, cell_size=1.0)
    assert g.info.n_cells == og.n_cells == rows * per
    starts, sizes, _, perm = g.to_host()
    assert np.array_equal(sizes, og.counts) and np.array_equal(starts, og.starts)
    assert np.array_equal(perm, og.perm)
    g.close()
