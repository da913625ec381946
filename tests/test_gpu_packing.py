"""How bodies share workgroups: none do while the chip runs a workgroup of each at once (512), beyond
that as many workgroups as it runs at once, never more; a body's floats do not depend on it."""
import numpy as np
import pytest

from joltphysics_amd import scenes
from joltphysics_amd.records import BodyParams
from joltphysics_amd.xpbd import Context, build_settings

pytestmark = pytest.mark.gpu

AT_ONCE = 512


@pytest.fixture(scope="module")
def settings():
    def cloth(n):
        v, f = scenes.cloth(n, 0.05, 100.0, jitter=0.005, seed=n)
        return build_settings(scenes.MeshSpec(vertices=v, faces=f, attrs=scenes.attrs(1e-4, 1e-4, 1e-3)))
    return {n: cloth(n) for n in (5, 9, 17, 31)}


def _run(settings, sizes, iterations=2):
    ctx = Context(0)
    try:
        ctx.set_gravity((0.0, 0.0, -9.81))
        handles = {n: ctx.create_settings(s) for n, s in settings.items()}
        ids = [ctx.create_body(handles[n], (3.0 * k, 0.0, 1.0), (0.0, 0.6, 0.0, 0.8),
                               BodyParams(num_iterations=iterations + (k % 7 == 3), allow_sleeping=False))
               for k, n in enumerate(sizes)]
        ctx.update(1 / 60, 1, 2)
        places = [ctx.placement(i) for i in ids]
        assert all(p[0] == "bundle" for p in places)
        return len({p[2] for p in places}), {p[1] for p in places}, [ctx.read(ids[k])["pos"] for k in range(0, len(ids), 37)]
    finally:
        ctx.close()


@pytest.mark.parametrize("sizes", [
    [5] * 512, [5, 9, 17, 31] * 100,                        # a workgroup each
    [5] * 513, [9] * 1023, [5, 9, 17, 31] * 200, [5] * 3000,  # at most 512, two iteration counts among them
], ids=lambda s: f"{len(s)}x{max(s)}")
def test_workgroups_and_results(settings, sizes):
    count, _, got = _run(settings, sizes)
    print(f"{len(sizes)} bodies: {count} workgroups", flush=True)
    if len(sizes) <= AT_ONCE:
        assert count == len(sizes)
    else:
        assert count <= AT_ONCE
    alone = {}
    for k, g in zip(range(0, len(sizes), 37), got):
        key = (sizes[k], k % 7 == 3)
        if key not in alone:
            alone[key] = _run(settings, [sizes[k]], 2 + key[1])[2][0]
        assert np.array_equal(g, alone[key]), f"body {k}"


@pytest.mark.parametrize("sizes, threads", [([17], {512}), ([17] * 256, {512}), ([31], {1024}), ([5] + [31] * 255, {1024}),
                                            ([31] * 257, {512})], ids=lambda v: str(len(v)))
def test_threads(settings, sizes, threads):
    """Where a body has more than 512 vertices, workgroups have 1024 threads while each has a CU to itself."""
    workgroups, used, got = _run(settings, sizes)
    assert workgroups == len(sizes) and used == threads
    for k, g in zip(range(0, len(sizes), 37), got):
        want = _run(settings, [sizes[k]], 2 + (k % 7 == 3))[2][0]
        assert np.array_equal(g, want), f"body {k}"


def test_layout_costs_less_than_the_bodies(settings):
    """Laying out many small bodies, a workgroup each, takes less than creating them."""
    import time
    create = layout = 1e9
    for _ in range(4):
        ctx = Context(0)
        st = ctx.create_settings(settings[17])
        t0 = time.perf_counter()
        for k in range(400):
            ctx.create_body(st, (2.0 * k, 0.0, 1.0), (0.0, 0.0, 0.0, 1.0), BodyParams(allow_sleeping=False))
        t1 = time.perf_counter()
        ctx.update(1 / 60, 1, 1)
        ctx.synchronize()
        create, layout = min(create, t1 - t0), min(layout, time.perf_counter() - t1)
        ctx.close()
    print(f"400 bodies: created in {1e3 * create:.1f} ms, first update {1e3 * layout:.1f} ms", flush=True)
    # 25 against 37 ms; 55 with eleven allocations, four uploads and a program built for every workgroup
    assert layout < create
