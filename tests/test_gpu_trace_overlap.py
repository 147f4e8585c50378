"""Photon maps of scenes whose models share triangles (a patch of a mesh with a
material of its own, meshes that overlap in part, one range as two models, a
light that is part of a mesh), with and without an acceleration structure, bit
for bit against the oracle, which tests every triangle of every model in order."""
import numpy as np
import pytest

import pyoracle as O
from pm355.scenes import PM_MODEL_DTYPE, Scene, _model, cornell_box, uv_sphere

pytestmark = pytest.mark.gpu

MIRROR, GLASS = dict(ks=(1, 1, 1), shininess=0.0), dict(ks=(1, 1, 1), opaque=0.0, ior=1.4)
GREY, RED = dict(kd=(0.5, 0.5, 0.5)), dict(kd=(0.8, 0.1, 0.1))


def _scene(spheres, ranges, light=None):
    """cornell_box, the triangles of `spheres` behind it, and a model for each
    (first, last, material) of `ranges`, counted from the first sphere's; light:
    the one of `ranges` that emits."""
    base = cornell_box()
    tris, nrms, models = [base.tris9], [base.normals9], [m for m in base.models]
    n0 = base.tris9.shape[0]
    for s in spheres:
        t, n = uv_sphere(*s)
        tris.append(t)
        nrms.append(n)
    for i, (a, b, mat) in enumerate(ranges):
        models.append(_model(n0 + a, n0 + b, mid=100 + i, **mat))
    return Scene(np.concatenate(tris), np.concatenate(nrms), np.array(models, PM_MODEL_DTYPE),
                 light_model=base.light_model if light is None else len(base.models) + light)


S1, S2 = ((0.35, 0.3, 0.4), 0.2, 12, 10), ((0.6, 0.45, 0.55), 0.18, 11, 9)
N1, N2 = uv_sphere(*S1)[0].shape[0], uv_sphere(*S2)[0].shape[0]
SCENES = {
    "patch_after": lambda: _scene([S1], [(0, N1, GREY), (N1 // 2, N1 // 2 + 7, MIRROR)]),
    "patch_before": lambda: _scene([S1], [(N1 // 2, N1 // 2 + 15, MIRROR), (0, N1, GLASS)]),
    "tree_in_tree": lambda: _scene([S1], [(0, N1, GREY), (N1 // 3, N1 // 3 + 40, MIRROR)]),
    "overlap": lambda: _scene([S1, S2], [(0, N1 + N2 // 2, MIRROR), (N1 // 2, N1 + N2, RED)]),
    "same_range": lambda: _scene([S1], [(0, N1, RED), (0, N1, MIRROR), (N1 // 2, N1 // 2, GREY)]),
    "light_patch": lambda: _scene([S2], [(0, N2, GREY), (N2 // 2, N2 // 2 + 4, GREY)], light=1),
    "models_33": lambda: _scene([S1, S2], [(7 * i, 7 * i + 20 + i, GREY if i % 3 else MIRROR) for i in range(25)]),
}


@pytest.mark.parametrize("name", list(SCENES))
@pytest.mark.parametrize("accel", [True, False])
def test_maps_equal_the_oracles(ctx, name, accel):
    scene = SCENES[name]()
    ds = ctx.upload_scene(scene, accel=accel)
    n_g, n_c = 20_011, 503
    g, c, st = ctx.trace_photons(ds, 78, n_g, n_c, max_bounces=8, max_paths=200_000)
    og, oc, ost = O.trace_photons(scene, 78, n_g, n_c, max_bounces=8, max_paths=200_000)
    assert st[1:] == ost[1:]
    g, c = g.cpu().numpy(), c.cpu().numpy()
    assert np.array_equal(g[:, :st[1]].view(np.uint32), og[:, :st[1]].view(np.uint32))
    assert np.array_equal(c[:, :st[2]].view(np.uint32), oc[:, :st[2]].view(np.uint32))
