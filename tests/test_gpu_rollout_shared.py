"""Bodies of a rollout that have the same settings share its programs, wherever they stand in the list:
each body's result and gradients are those of a rollout of its own, and more of them cost little."""
import time

import numpy as np
import pytest

from joltphysics_amd import scenes
from joltphysics_amd.xpbd import Context, build_settings

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

FRAMES, ITERATIONS = 6, 4


def _pass(ctx, handles, comp, vel, seed):
    """Final positions in float and double, and the gradients, body by body."""
    from joltphysics_amd.autograd import rollout
    r = ctx.create_rollout(handles, num_iterations=ITERATIONS, frames=FRAMES, checkpoint_interval=4)
    c = torch.from_numpy(np.concatenate(comp)).cuda().requires_grad_(True)
    v = torch.from_numpy(np.concatenate(vel).reshape(-1)).cuda().requires_grad_(True)
    x = rollout(c, v, r)
    g = torch.from_numpy(np.concatenate(seed)).cuda()
    gc, gv = torch.autograd.grad(x, (c, v), g)
    c64, v64 = c.detach().double(), v.detach().double()
    x64 = torch.empty((r.num_vertices, 3), dtype=torch.float64, device="cuda")
    r.forward_f64(c64.data_ptr(), v64.data_ptr(), x64.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    out, at_v, at_e = [], 0, 0
    for ck, vk in zip(comp, vel):
        nv, ne = len(vk), len(ck)
        out.append([a.cpu().numpy() for a in (x.detach()[at_v:at_v + nv], x64[at_v:at_v + nv], gc[at_e:at_e + ne],
                                              gv.view(-1, 3)[at_v:at_v + nv])])
        at_v, at_e = at_v + nv, at_e + ne
    r.close()
    return out


def test_alternating_settings_match_separate_rollouts():
    rng = np.random.default_rng(9)
    cloth = build_settings(scenes.config4_rollout(num_bodies=1, n=9, frames=FRAMES).mesh)
    tets = build_settings(scenes.rollout_tet_block(1, 3, frames=FRAMES).mesh)
    ctx = Context(0)
    handles = {id(s): ctx.create_settings(s) for s in (cloth, tets)}
    bodies = [cloth, tets, cloth, cloth, tets, cloth]
    comp = [rng.uniform(1e-4, 1e-2, len(s.edges)).astype(np.float32) for s in bodies]
    vel = [rng.uniform(-0.1, 0.1, (len(s.vertices), 3)).astype(np.float32) for s in bodies]
    seed = [rng.standard_normal((len(s.vertices), 3)).astype(np.float32) for s in bodies]
    got = _pass(ctx, [handles[id(s)] for s in bodies], comp, vel, seed)
    for k, s in enumerate(bodies):
        want = _pass(ctx, [handles[id(s)]], comp[k:k + 1], vel[k:k + 1], seed[k:k + 1])[0]
        for g, w, what in zip(got[k], want, ("positions", "positions in double", "compliance", "velocity")):
            assert np.isfinite(w).all() and np.array_equal(g, w), f"body {k}: {what}"
    ctx.close()


def test_bodies_of_one_settings_cost_little():
    s = build_settings(scenes.config4_rollout(num_bodies=1, n=64, frames=2).mesh)

    def create(count):
        best = 1e9
        for _ in range(6):
            ctx = Context(0)
            st = ctx.create_settings(s)
            t = time.perf_counter()
            r = ctx.create_rollout([st] * count, frames=2, checkpoint_interval=1)
            best = min(best, time.perf_counter() - t)
            r.close()
            ctx.close()
        return best

    one, many = create(1), create(64)
    print(f"one body {1e3 * one:.2f} ms, 64 bodies {1e3 * many:.2f} ms", flush=True)
    # about 4 times; 47 with a level program for every body and its records made on the host
    assert many < 12 * one
