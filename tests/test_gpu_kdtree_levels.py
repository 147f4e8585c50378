"""kd-tree levels at the edges of the partition's tiles (8192 positions): nodes
that just fill a tile, reach one position past it, span several, levels whose
tiles wait for earlier ones and levels that do not. Exact against the oracle."""
import numpy as np
import pytest

import pyoracle as O

pytestmark = pytest.mark.gpu

TILE = 8192


@pytest.mark.parametrize("n", [TILE - 1, TILE, TILE + 1, TILE + 2, TILE + 3, 2 * TILE, 2 * TILE + 3, 2 * TILE + 5,
                               4 * TILE - 1, 7 * TILE + 13, 40 * TILE + 1])
def test_build(ctx, n):
    rng = np.random.default_rng(n)
    pos = rng.random((3, n), dtype=np.float32)
    pos[0, : n // 2] = np.float32(0.1) * rng.integers(0, 4, n // 2)  # ties on one axis
    pos[:, n // 3:n // 3 + 50] = pos[:, n // 3:n // 3 + 1]
    ph = np.ones((9, n), np.float32)
    ph[0:3] = pos
    for _ in range(2):  # (the second build finds the first one's scratch)
        ni, npl = ctx.kdtree_build(ph).to_host()
        oi, opl = O.kdtree_build(pos)
        assert np.array_equal(ni, oi)
        assert np.array_equal(npl, opl)
