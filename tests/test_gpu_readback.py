"""xpbd_body_read: one packed launch per call, any subset of the arrays, before the first update, after
updates and after a write, for bodies of every storage."""
import ctypes as C

import numpy as np
import pytest

from joltphysics_amd import scenes
from joltphysics_amd.records import SHAPE_PLANE, VERTEX, BodyParams, Collider, SettingsArrays, GROUP
from joltphysics_amd.xpbd import Context, build_settings

pytestmark = pytest.mark.gpu

ARRAYS = ("pos", "prev", "vel", "plane", "shape_idx", "contact", "body_pos", "body_rot")


def _settings(n, m):
    if n * m == 1:
        return SettingsArrays(np.ones(1, VERTEX), groups=np.zeros(1, GROUP))
    v, f = scenes.cloth(n, 0.05, 100.0, jitter=0.005, seed=n, nz=m)
    v["vel"] = np.random.default_rng(n).uniform(-1, 1, (len(v), 3))
    return build_settings(scenes.MeshSpec(vertices=v, faces=f, attrs=scenes.attrs(1e-4, 1e-4, 1e-3)))


def _partial(ctx, body, names):
    whole = ctx.read(body)
    out = {k: np.full_like(whole[k], 7) for k in names}
    args = [out[k].ctypes.data_as(C.c_void_p) if k in out else None for k in ARRAYS]
    assert ctx.lib.xpbd_body_read(ctx.h, body, *args) == 0
    for k in names:
        assert np.array_equal(out[k], whole[k]), k
    return whole


@pytest.mark.parametrize("n,m", [(1, 1), (2, 2), (13, 5), (64, 4), (120, 120), (160, 160)])
def test_read_subsets_and_moments(n, m):
    s = _settings(n, m)
    plane = Collider(SHAPE_PLANE, (0.0, 0.0, 1.0, 0.0, 1000.0))
    plane.bounds = scenes.collider_world_bounds(plane)
    ctx = Context(0)
    ctx.set_gravity((0.0, 0.0, -9.81))
    ctx.set_colliders([plane])
    st = ctx.create_settings(s)
    a = ctx.create_body(st, (0.0, 0.0, 0.01), params=BodyParams(num_iterations=2, allow_sleeping=False))
    first = ctx.read(a)
    assert np.array_equal(first["pos"], s.vertices["pos"]) and np.array_equal(first["vel"], s.vertices["vel"])
    assert np.array_equal(first["body_pos"], np.float32((0.0, 0.0, 0.01)))
    ctx.update(1 / 60, 1, 2)
    for names in (ARRAYS, ("pos",), ("vel", "body_pos"), ("plane", "contact"), ("prev", "shape_idx", "body_rot"), ("body_pos",)):
        _partial(ctx, a, names)
    # a body created after an update has no row on the device yet
    b = ctx.create_body(st, (1.0, 2.0, 3.0), params=BodyParams(num_iterations=2, allow_sleeping=False))
    assert np.array_equal(ctx.read(b)["body_pos"], np.float32((1.0, 2.0, 3.0)))
    kept = ctx.read(a)
    ctx.write(a, pos=kept["pos"] + np.float32(1.0))
    assert np.array_equal(ctx.read(a)["pos"], kept["pos"] + np.float32(1.0))
    ctx.close()
