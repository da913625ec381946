"""Wide task programs at the ends of the float range: the coloured schedule's levels hold hundreds of
constraints, which run a lane each with shared divisions, and the quotients that these do not cover
(denormal results, infinities) fall back to the plain divisions.  Bit-exact against the
restatement (FP32) on the recoloured settings."""
import numpy as np
import pytest

from helpers import float_equal, recoloured_settings, run_gpu, run_restatement
from joltphysics_amd import scenes
from joltphysics_amd.records import BodyParams
from joltphysics_amd.xpbd import build_settings, host_schedule

pytestmark = pytest.mark.gpu

BEND, EDGE, SECOND_HALF, NOP = 1, 2, 1 << 15, 0xFFFFFFFF


def _widest(s, kind):
    h = host_schedule(s, "coloured")
    r, b = h["identity_recs"], h["identity_level_begin"]
    own = (r[:, 0] != NOP) & (((r[:, 0] >> 14) & 3) == kind)
    if kind == BEND:
        own &= (r[:, 1] & SECOND_HALF) == 0
    return max(int(own[b[k]:b[k + 1]].sum()) for k in range(len(b) - 1))


def _check(s, gravity=0.0, frames=(1, 3)):
    # four lanes each, n bends take n / 16 tasks of about 215 instructions on four SIMDs, a lane each one
    # task of 290: more than about 100 run a lane each, edges (48 and 70) more than about 110
    assert _widest(s, BEND) > 128 and _widest(s, EDGE) > 128
    body = scenes.BodySpec(None, (0.0, 0.0, 0.0), (0.0, 0.0, 0.0, 1.0),
                           BodyParams(num_iterations=3, allow_sleeping=False, max_linear_velocity=1e30))
    sc = scenes.Scene("wide", [body], [], gravity=(0.0, 0.0, gravity), collision_steps=1)
    got = run_gpu(sc, [s], frames_to_keep=frames, schedule="coloured")
    want = run_restatement(sc, [recoloured_settings(s)[0]], [], frames_to_keep=frames)
    for f in frames:
        for k in ("pos", "vel"):
            assert np.isfinite(want[f][0][k]).all() and float_equal(got[f][0][k], want[f][0][k]), f"frame {f} {k}"
    return want


@pytest.mark.parametrize("scale", [1e-22, 1e-12, 1e-6, 1.0, 1e6, 1e10])
@pytest.mark.parametrize("shape", ["cloth", "sphere"])
def test_ends_of_the_float_range(shape, scale):
    if shape == "cloth":
        v, f = scenes.cloth(48, 0.05 * scale, 100.0, jitter=0.005 * scale, seed=3, nz=40)
    else:
        v, f = scenes.icosphere(4, radius=scale)
    v["vel"] = np.random.default_rng(5).uniform(-scale, scale, (len(v), 3)).astype(np.float32)
    s = build_settings(scenes.MeshSpec(vertices=v, faces=f, attrs=scenes.attrs(1e-4, 1e-4, 1e-3)))
    _check(s, gravity=-9.81 * scale)


@pytest.mark.parametrize("kick", [1e-38, 1e-40, 3e-36])
def test_denormal_quotients(kick):
    """A flat sheet whose vertices leave it by denormal steps: normals, and so a bend's and an edge's
    quotients, have denormal components beside ordinary ones, in some lanes of a level."""
    v, f = scenes.cloth(40, 1.0, 1.0)
    some = np.random.default_rng(2).random(len(v)) < 0.3
    v["vel"][some, 2] = np.random.default_rng(7).uniform(-1, 1, int(some.sum())) * kick
    s = build_settings(scenes.MeshSpec(vertices=v, faces=f, attrs=scenes.attrs(0.0, 0.0, 0.0)))
    want = _check(s)
    z = np.abs(want[1][0]["pos"][:, 2])
    assert (z[z > 0] < np.finfo(np.float32).tiny * 1e3).all() and (z > 0).any()
