"""The caustic map where its batches mark their storing paths by bits (a million
paths and more in a batch): bit for bit the oracle's, to its last photon, which
lies inside a word of 32 paths."""
import numpy as np
import pytest

import pyoracle as O
from pm355.scenes import cornell_box

pytestmark = pytest.mark.gpu

BIT_PATHS = 1 << 20  # a caustic batch of this many paths and more


@pytest.mark.parametrize("n_g,n_c", [(5_003, 120_001), (20_000, 200_017)])
def test_caustic_map_equals_the_oracles(ctx, n_g, n_c):
    scene = cornell_box()
    g, c, st = ctx.trace_photons(ctx.upload_scene(scene, accel=True), 91, n_g, n_c)
    # the first batch is of n_g + n_c paths; one of the next, sized to fill the map at
    # the first's yield, takes nearly all the others
    assert st[0] > n_g + n_c + 1.5 * BIT_PATHS
    og, oc, ost = O.trace_photons(scene, 91, n_g, n_c)
    assert st[1:] == ost[1:] == (n_g, n_c)
    assert np.array_equal(g.cpu().numpy().view(np.uint32), og.view(np.uint32))
    assert np.array_equal(c.cpu().numpy().view(np.uint32), oc.view(np.uint32))
