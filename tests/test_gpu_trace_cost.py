"""What a trace costs beside another trace of the same scene. A scene of up to 32
models is walked through its triangle records, one of more (here: the same
models and empty ones) model by model; both walks find the same hits and
neither may take several times as long as the other. Times are the least of
several calls in turn; the bounds lie between what the right and a wrong walk
measured, well apart."""
import time

import numpy as np
import pytest

from pm355.scenes import PM_MODEL_DTYPE, Scene, _model, cornell_box, random_scene, uv_sphere

pytestmark = pytest.mark.gpu


def _padded(scene, n):
    """The same scene with empty models up to n."""
    extra = [_model(0, 0, mid=1000 + i) for i in range(n - len(scene.models))]
    return Scene(scene.tris9, scene.normals9, np.concatenate([scene.models, np.array(extra, PM_MODEL_DTYPE)]),
                 light_model=scene.light_model)


def _spheres(n):
    base = cornell_box()
    rng = np.random.default_rng(3)
    tris, nrms, models, t0 = [base.tris9], [base.normals9], [m for m in base.models], base.tris9.shape[0]
    for i in range(n):
        r = float(rng.uniform(0.02, 0.08))
        t, nr = uv_sphere(rng.uniform(r, 0.9 - r, 3), r, 12, 10)
        tris.append(t)
        nrms.append(nr)
        models.append(_model(t0, t0 + len(t), mid=50 + i, kd=(0.6, 0.5, 0.4)))
        t0 += len(t)
    return Scene(np.concatenate(tris), np.concatenate(nrms), np.array(models, PM_MODEL_DTYPE),
                 light_model=base.light_model)


def _times(ctx, scenes, n, reps=6):
    """The least time of a trace of each scene, and their global maps."""
    ds = [ctx.upload_scene(s, accel=True) for s in scenes]
    best, maps = [1e9] * len(ds), [None] * len(ds)
    for _ in range(reps):
        for i, d in enumerate(ds):
            ctx.sync()
            t0 = time.perf_counter()
            maps[i] = ctx.trace_photons(d, 9, n, 0, max_paths=65536 + n)[0]
            ctx.sync()
            best[i] = min(best[i], time.perf_counter() - t0)
    return best, [m.cpu().numpy().view(np.uint32) for m in maps]


def test_lanes_without_a_path_open_no_box(ctx):
    """65536 paths, a lane each: most lanes wait for the last paths. With the
    waiting lanes' boxes opened the model-by-model walk took 5.4 times the
    other's time, without 2.3 times."""
    scene = _spheres(24)
    assert len(scene.models) <= 32
    (rec, by_model), maps = _times(ctx, [scene, _padded(scene, 33)], 1000)
    assert np.array_equal(*maps)
    assert by_model < 3.5 * rec


def test_rays_of_the_general_walk_take_the_trees(ctx):
    """A few rays of this scene of 44k triangles leave the records' walk for the
    general one (a hit at t == 0): past all triangles a trace took 5.8 times the
    model-by-model time, by the trees half of it."""
    scene = random_scene(3)
    (rec, by_model), maps = _times(ctx, [scene, _padded(scene, 33)], 1000)
    assert np.array_equal(*maps)
    assert rec < 1.5 * by_model
