"""Photon maps of scenes at the edges of the tracer's ray walk, bit for bit
against the oracle (which tests every triangle of every model): models of just
under and over 16 triangles (no tree / a tree), one tree and many, more models
than a lane's mask holds (33: the model-by-model walk), a surface exactly
through the emission origins (hits at t == 0), and batch sizes around the
emission segments."""
import numpy as np
import pytest

import pyoracle as O
from pm355.scenes import PM_MODEL_DTYPE, Scene, _model, _quad, cornell_box, uv_sphere

pytestmark = pytest.mark.gpu


def _scene(extra):
    """cornell_box with the parts `extra` (triangles, normals, material) added."""
    base = cornell_box()
    tris, nrms, models = [base.tris9], [base.normals9], [m for m in base.models]
    t0 = base.tris9.shape[0]
    for i, (t, n, mat) in enumerate(extra):
        tris.append(t)
        nrms.append(n)
        models.append(_model(t0, t0 + len(t), mid=100 + i, **mat))
        t0 += len(t)
    return Scene(np.concatenate(tris), np.concatenate(nrms), np.array(models, PM_MODEL_DTYPE),
                 light_model=base.light_model)


def _spheres(n, slices, stacks, seed):
    rng = np.random.default_rng(seed)
    kinds = [dict(kd=(0.6, 0.5, 0.4)), dict(ks=(1, 1, 1), shininess=0.0), dict(ks=(1, 1, 1), opaque=0.0, ior=1.4)]
    out = []
    for i in range(n):
        r = float(rng.uniform(0.04, 0.15))
        c = rng.uniform(r, 0.9 - r, 3)
        out.append((*uv_sphere(c, r, slices, stacks), kinds[i % 3]))
    return out


def _at_origins():
    # the light's emission origins lie 1e-4 below it
    y = np.float32(0.999) + np.float32(-1.0) * np.float32(0.0001)
    P = lambda *a: np.array(a, np.float32)  # noqa: E731
    return [(*_quad(P(0.3, y, 0.3), P(0.7, y, 0.3), P(0.7, y, 0.7), P(0.3, y, 0.7), P(0, -1, 0)),
             dict(kd=(0.5, 0.5, 0.5)))]


SCENES = {
    "cornell": lambda: _scene([]),
    "under_16": lambda: _scene(_spheres(3, 3, 3, 1)),   # 12 triangles each
    "at_16": lambda: _scene(_spheres(3, 4, 3, 2)),      # 16
    "over_16": lambda: _scene(_spheres(4, 5, 3, 3)),    # 20
    "trees": lambda: _scene(_spheres(24, 9, 7, 4)),     # 32 models
    "models_33": lambda: _scene(_spheres(25, 9, 7, 5)),
    "t_zero": lambda: _scene(_at_origins()),
}


@pytest.mark.parametrize("name", list(SCENES))
@pytest.mark.parametrize("accel", [True, False])
def test_maps_equal_the_oracles(ctx, name, accel):
    scene = SCENES[name]()
    ds = ctx.upload_scene(scene, accel=accel)
    n_g, n_c = 20_011, 1_003
    g, c, st = ctx.trace_photons(ds, 77, n_g, n_c, max_bounces=8, max_paths=400_000)
    og, oc, ost = O.trace_photons(scene, 77, n_g, n_c, max_bounces=8, max_paths=400_000)
    assert st[1:] == ost[1:]
    g, c = g.cpu().numpy(), c.cpu().numpy()
    assert np.array_equal(g[:, :st[1]].view(np.uint32), og[:, :st[1]].view(np.uint32))
    assert np.array_equal(c[:, :st[2]].view(np.uint32), oc[:, :st[2]].view(np.uint32))


@pytest.mark.parametrize("max_paths", [1, 255, 256, 257, 65_535, 65_537, 300_001])
def test_path_limits_around_the_segments(ctx, max_paths):
    scene = cornell_box()
    ds = ctx.upload_scene(scene, accel=True)
    g, c, st = ctx.trace_photons(ds, 5, 400_000, 2_000, max_paths=max_paths)
    og, oc, ost = O.trace_photons(scene, 5, 400_000, 2_000, max_paths=max_paths)
    assert st == ost
    assert np.array_equal(g.cpu().numpy()[:, :st[1]].view(np.uint32), og[:, :st[1]].view(np.uint32))
    assert np.array_equal(c.cpu().numpy()[:, :st[2]].view(np.uint32), oc[:, :st[2]].view(np.uint32))


def test_caustic_phase_bits(ctx):
    """Caustic-phase batches of a million paths and more mark their storing
    paths by bits, smaller ones by counts: the photons (the first n in path
    order, whatever the batches) are the same."""
    scene = ctx.upload_scene(SCENES["cornell"](), accel=True)
    maps = [ctx.trace_photons(scene, 77, 20_000, nc)[1].cpu().numpy().view(np.uint32)
            for nc in (1_000, 30_000, 70_000, 160_000)]
    for few, more in zip(maps, maps[1:]):
        assert np.array_equal(more[:, :few.shape[1]], few)
    assert maps[-1][0].max() > 0
