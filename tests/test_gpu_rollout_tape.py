"""The rollout adjoint's two ways to its tape: a whole segment's, kept while the segment is
recomputed, and one sub-step's, filled by running the sub-step again (segments whose tape exceeds
the budget).  Checkpoints change no value, so both give the same gradients bit for bit."""
import numpy as np
import pytest

from joltphysics_amd import scenes
from joltphysics_amd.xpbd import Context, build_settings

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _gradients(case, s, interval):
    from joltphysics_amd.autograd import rollout
    ctx = Context(0)
    ctx.set_gravity(case.gravity)
    st = ctx.create_settings(s)
    r = ctx.create_rollout([st] * case.num_bodies, num_iterations=case.iterations, dt=case.dt, frames=case.frames,
                           checkpoint_interval=interval)
    comp = torch.from_numpy(case.compliance).cuda().requires_grad_(True)
    vel = torch.from_numpy(case.velocity.reshape(-1)).cuda().requires_grad_(True)
    x = rollout(comp, vel, r)
    seed = torch.from_numpy(np.random.default_rng(3).standard_normal(tuple(x.shape)).astype(np.float32)).cuda()
    out = [g.cpu().numpy() for g in (x.detach(), *torch.autograd.grad(x, (comp, vel), seed))]
    torch.cuda.synchronize()
    r.close()
    ctx.close()
    return out


# segments: shorter than the rollout, the whole rollout, longer than it; 32 x 220 frames of a
# 64 x 64 cloth in one segment exceed the tape budget (8 GiB)
@pytest.mark.parametrize("n,bodies,frames,intervals", [(9, 3, 7, (1, 3, 7, 50)), (64, 32, 220, (10, 220))])
def test_segment_length_changes_nothing(n, bodies, frames, intervals):
    case = scenes.config4_rollout(num_bodies=bodies, n=n, frames=frames)
    s = build_settings(case.mesh)
    want = _gradients(case, s, intervals[0])
    assert all(np.isfinite(w).all() for w in want)
    for interval in intervals[1:]:
        for g, w in zip(_gradients(case, s, interval), want):
            assert np.array_equal(g, w)
