"""A streamed body of two parallel-group windows runs on a team of two workgroups while all such
bodies' teams fit the card at once (224 workgroups), and on one workgroup otherwise or when the
number of windows is set.  Both ways give the same floats, so every comparison is exact."""
import numpy as np
import pytest

from joltphysics_amd import scenes
from joltphysics_amd.records import SHAPE_SPHERE, Collider
from joltphysics_amd.xpbd import Context, build_settings

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def settings():
    return build_settings(scenes.MeshSpec(*scenes.cloth(120, 0.1)[:2], attrs=scenes.attrs(1e-5, 1e-5, 1e-5)))


def _run(settings, count, min_windows=None, frames=2):
    ctx = Context(0)
    try:
        ctx.set_gravity((0.0, 0.0, -9.81))
        colliders = [Collider(SHAPE_SPHERE, (1.0,), pos=(5.0 * k, 0.0, 0.0)) for k in range(3)]
        for c in colliders:
            c.bounds = scenes.collider_world_bounds(c)
        ctx.set_colliders(colliders)
        st = ctx.create_settings(settings)
        assert st.stats()["parallel_windows"] == 2
        if min_windows is not None:
            ctx.set_team_min_windows(min_windows)
        ids = [ctx.create_body(st, (4.0 * k, 0.0, 1.1), (0.0, 0.0, 0.0, 1.0)) for k in range(count)]
        ctx.update(1.0 / 60.0, 1, frames)
        out = [ctx.read(i) for i in (ids[0], ids[-1])]
        return {ctx.placement(i)[0] for i in ids}, ctx.placement(ids[0])[3], out
    finally:
        ctx.close()


@pytest.mark.parametrize("count, kind", [(1, "team"), (3, "team"), (112, "team"), (113, "streamed")])
def test_two_window_bodies(settings, count, kind):
    kinds, size, got = _run(settings, count)
    assert kinds == {kind} and (kind != "team" or size == 2)
    for windows in (3, 0):
        kinds, _, want = _run(settings, count, windows)
        assert kinds == {"streamed"}
        for g, w in zip(got, want):
            for key in ("pos", "vel", "body_pos"):
                assert np.array_equal(np.asarray(g[key]), np.asarray(w[key])), key
