"""Teams of workgroups beside a running batch.  Members of a team sit on different XCDs and hand
positions to each other through memory, while the bundles of the same update fill every XCD's L2 with
dirty lines.  A body gives the same floats on a team as on one workgroup, so the comparison is exact."""
import numpy as np
import pytest

from joltphysics_amd import scenes
from joltphysics_amd.records import SHAPE_PLANE, BodyParams, Collider
from joltphysics_amd.xpbd import Context, build_settings

pytestmark = pytest.mark.gpu

LARGE, SMALL = 40, 700


@pytest.fixture(scope="module")
def settings():
    def cloth(n):
        v, f = scenes.cloth(n, 0.05, 100.0, jitter=0.005, seed=n)
        return build_settings(scenes.MeshSpec(vertices=v, faces=f, attrs=scenes.attrs(1e-4, 1e-4, 1e-3)))
    return [cloth(n) for n in (118, 122, 125, 128)], cloth(44)


def _run(settings, schedule, min_windows):
    large, small = settings
    rng = np.random.default_rng(3)
    ctx = Context(0)
    try:
        ctx.set_gravity((0.0, 0.0, -9.81))
        plane = Collider(SHAPE_PLANE, (0.0, 0.0, 1.0, 0.0, 1000.0))
        plane.bounds = scenes.collider_world_bounds(plane)
        ctx.set_colliders([plane])
        ctx.set_team_min_windows(min_windows)
        params = BodyParams(num_iterations=5, allow_sleeping=False)
        handles = [ctx.create_settings(s, schedule) for s in large]
        assert all(h.stats()["parallel_windows"] == 2 for h in handles)
        # tilted, so that corners touch the ground from the first frames on
        ids = [ctx.create_body(handles[k % len(handles)], (8.0 * k, 0.0, 2.0), scenes.random_quaternion(rng), params)
               for k in range(LARGE)]
        rest = ctx.create_settings(small, schedule)
        for k in range(SMALL):
            ctx.create_body(rest, (8.0 * k, 20.0, 1.0), scenes.random_quaternion(rng), params)
        for _ in range(2):
            ctx.update(1.0 / 60.0, 2, 20)
        return {ctx.placement(i)[0] for i in ids}, [ctx.read(i) for i in ids]
    finally:
        ctx.close()


@pytest.mark.parametrize("schedule", ["coloured", "exact"])
def test_teams_beside_a_batch_equal_one_workgroup(settings, schedule):
    kinds, got = _run(settings, schedule, 2)
    assert kinds == {"team"}
    print(f"{schedule}: teams done", flush=True)
    kinds, want = _run(settings, schedule, 0)
    assert kinds == {"streamed"}
    for k, (g, w) in enumerate(zip(got, want)):
        for key in ("pos", "vel", "body_pos"):
            assert np.array_equal(np.asarray(g[key]), np.asarray(w[key])), f"body {k}: {key}"
