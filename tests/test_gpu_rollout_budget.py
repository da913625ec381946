"""Where the segment tape of a rollout's adjoint does not fit: what the context's other rollouts hold
and what is free on the card leave it one sub-step's tape, never a refused rollout, and the gradients
stay the same bit for bit, whatever the constraints."""
import numpy as np
import pytest

from joltphysics_amd import scenes
from joltphysics_amd.xpbd import Context, build_settings

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

BUDGET = 8 << 30        # of a context's segment tapes


def _cloth(n=64):
    v, f = scenes.cloth(n, 0.05, 100.0)
    return build_settings(scenes.MeshSpec(vertices=v, faces=f, attrs=scenes.attrs(1e-3, 1e-3, 0.0), bend_type=scenes.BEND_NONE))


def _fill(ctx):
    """Rollouts whose segment tapes leave less than one sub-step of one 64 x 64 cloth of the budget."""
    s = _cloth()
    st = ctx.create_settings(s)
    per_body = 16 * (len(s.edges) + 1)      # bytes of a sub-step
    left, out = BUDGET, []
    for bodies in (32, 1):
        subs = left // (bodies * per_body)
        if subs > 1:
            out.append(ctx.create_rollout([st] * bodies, num_iterations=1, frames=subs, checkpoint_interval=subs))
            left -= subs * bodies * per_body
    assert 0 <= left < 2 * per_body
    return out


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _case(kind):
    if kind == "tets":
        return scenes.rollout_tet_block(3, 4, frames=20)
    if kind == "balloon":
        return scenes.rollout_balloon(4, 3, frames=20)
    return scenes.config4_rollout(num_bodies=3, n=20, frames=20, lra=True, bends=kind == "bends_lra")


@pytest.mark.parametrize("kind", ["edges_lra", "bends_lra", "tets", "balloon"])
def test_one_substep_tape_gives_the_same_gradients(kind):
    from joltphysics_amd.autograd import rollout
    case = _case(kind)
    s = build_settings(case.mesh)
    results, taken = [], []
    for filled in (False, True):
        ctx = Context(0)
        ctx.set_gravity(case.gravity)
        fillers = _fill(ctx) if filled else []
        st = ctx.create_settings(s)
        before = _free()
        r = ctx.create_rollout([st] * case.num_bodies, num_iterations=case.iterations, dt=case.dt, frames=case.frames,
                               checkpoint_interval=case.frames, pressure=case.pressure)
        taken.append(before - _free())
        comp = torch.from_numpy(case.compliance).cuda().requires_grad_(True)
        vel = torch.from_numpy(case.velocity.reshape(-1)).cuda().requires_grad_(True)
        x = rollout(comp, vel, r)
        seed = torch.from_numpy(np.random.default_rng(3).standard_normal(tuple(x.shape)).astype(np.float32)).cuda()
        results.append([g.cpu().numpy() for g in (x.detach(), *torch.autograd.grad(x, (comp, vel), seed))])
        torch.cuda.synchronize()
        r.close()
        if filled:      # the budget is given back with the rollouts that held it
            for f in fillers:
                f.close()
            before = _free()
            r = ctx.create_rollout([st] * case.num_bodies, num_iterations=case.iterations, dt=case.dt, frames=case.frames,
                                   checkpoint_interval=case.frames, pressure=case.pressure)
            taken.append(before - _free())
            r.close()
        ctx.close()
    print(f"{kind}: {taken} bytes taken", flush=True)
    assert taken[1] < taken[0] and taken[1] < taken[2]
    for k, (whole, sub) in enumerate(zip(*results)):
        assert np.isfinite(whole).all()
        # faces that share a vertex, and the LRAs of one anchor, add to its adjoint in any order: 32-bit
        # sums taken in another order
        assert np.linalg.norm(sub - whole) <= 1e-5 * np.linalg.norm(whole)
        if kind != "balloon":
            # an anchor's adjoint reaches nothing but the gradient by its own velocity
            moving = np.tile(s.vertices["inv_mass"] > 0, case.num_bodies) if k == 2 else slice(None)
            per = (-1, 3) if k == 2 else whole.shape
            assert np.array_equal(sub.reshape(per)[moving], whole.reshape(per)[moving])


def test_rollout_on_a_full_card():
    """A rollout whose segment tape is more than what is free is created and runs."""
    ctx = Context(0)
    s = _cloth()
    st = ctx.create_settings(s)
    subs = BUDGET // (32 * 16 * (len(s.edges) + 1))
    # positions, velocities and checkpoints of the sub-steps: 32 bytes a vertex each
    rest = 32 * 4096 * 32 * (subs + 8)
    hold = torch.empty(_free() - rest - (3 << 30), dtype=torch.uint8, device="cuda")
    assert _free() < BUDGET + rest
    r = ctx.create_rollout([st] * 32, num_iterations=1, frames=subs, checkpoint_interval=subs)
    assert _free() > 1 << 30
    del hold
    torch.cuda.empty_cache()
    r.close()
    ctx.close()
