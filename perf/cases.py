"""Performance cases: the work a user of the soft-body update has it do.

A case is a set of soft bodies in a world (`kind` "scene"), advanced by
``Context.update`` and read back with ``Context.read``, or a differentiable rollout
(`kind` "rollout"), run through ``autograd.rollout`` with or without its backward pass.

Scene fields: `shape` (cloth, cube, sphere or mixed), `n` (vertices along a cloth's side,
cells along a cube's side, subdivisions of a sphere, largest cloth side of a mixed batch),
`m` (a cloth's other side), `bodies`, `steps` (collision steps), `iterations`, `frames`
(frames of one pass), `schedule` (exact, or the throughput schedule coloured), `pinned`
(two corners of a cloth, the top layer of a cube and its long-range attachments), `colliders`
(plane, box, spheres, boxes).  Rollout fields: `shape` (cloth: edges only, bends: a cloth with
dihedral bends and long-range attachments, tets: a block with volumes), `n`, `bodies`, `frames`,
`iterations`, `backward`.
"""
from __future__ import annotations

import random

import numpy as np
import torch

from joltphysics_amd import scenes
from joltphysics_amd.autograd import rollout
from joltphysics_amd.records import (BEND_DIHEDRAL, BEND_NONE, LRA, LRA_EUCLIDEAN, LRA_NONE, SHAPE_BOX, SHAPE_PLANE,
                                     SHAPE_SPHERE, BodyParams, Collider)
from joltphysics_amd.xpbd import Context, build_settings

DT = 1.0 / 60.0
GRAVITY = (0.0, 0.0, -9.81)


def _scene(name, shape, n, m=0, bodies=1, steps=1, iterations=5, frames=1, schedule="exact", pinned=False,
           colliders="plane"):
    return {"name": name, "kind": "scene", "shape": shape, "n": n, "m": m, "bodies": bodies, "steps": steps,
            "iterations": iterations, "frames": frames, "schedule": schedule, "pinned": pinned, "colliders": colliders}


def _rollout(name, shape, n, bodies, frames, iterations=5, backward=True):
    return {"name": name, "kind": "rollout", "shape": shape, "n": n, "bodies": bodies, "frames": frames,
            "iterations": iterations, "backward": backward}


def listed():
    return [
        # the smallest call: a flag in a game, one frame, positions read back for rendering
        _scene("flag_8x8", "cloth", 8, 8, pinned=True),
        # one ordinary cloth over a box, frame by frame
        _scene("cloth_32x32_box", "cloth", 32, 32, pinned=True, colliders="box"),
        # a handful of pressurised balls: ApplyPressure's volume sum and face impulses
        _scene("balls_x6", "sphere", 3, bodies=6, steps=2),
        # one tetrahedral body: edges and volumes, no bends
        _scene("cube_16", "cube", 16, steps=2),
        # a game frame with a crowd of small uneven bodies, every one read back
        _scene("crowd_x48", "mixed", 40, bodies=48),
        # the batched uneven workload in the reference's constraint order, several frames per call
        _scene("batch_x2048", "mixed", 128, bodies=2048, steps=2, frames=20),
        # the same batch under the throughput schedule
        _scene("batch_x2048_coloured", "mixed", 128, bodies=2048, steps=2, frames=20, schedule="coloured"),
        # one cloth too large for a workgroup's LDS, odd sides
        _scene("cloth_127x113", "cloth", 127, 113, steps=2, pinned=True),
        # a large cloth among spheres: a team of workgroups, exact order
        _scene("cloth_384x384_spheres", "cloth", 384, 384, steps=2, iterations=8, colliders="spheres"),
        # a large block with volumes and long-range attachments among boxes, throughput schedule
        _scene("block_40_coloured", "cube", 40, steps=4, iterations=10, schedule="coloured", pinned=True, colliders="boxes"),
        # fitting the compliance of 64 cloths: forward and adjoint
        _rollout("rollout_cloth64_x64", "cloth", 64, 64, 60),
        # a small fit over a body with volumes
        _rollout("rollout_tets4_x3", "tets", 4, 3, 10),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    kind = rng.choice(("cloth", "cloth", "cube", "sphere", "mixed", "mixed", "large", "rollout", "rollout"))
    schedule = rng.choice(("exact", "exact", "coloured"))
    steps, iterations = rng.choice((1, 1, 2, 4)), rng.choice((3, 4, 5, 5, 8, 10))
    if kind == "cloth":
        return _drawn(_scene("", "cloth", log_int(8, 140), log_int(8, 140), bodies=log_int(1, 12), steps=steps,
                             iterations=iterations, schedule=schedule, pinned=rng.random() < 0.5,
                             colliders=rng.choice(("plane", "box", "spheres"))))
    if kind == "cube":
        return _drawn(_scene("", "cube", log_int(3, 19), bodies=log_int(1, 16), steps=steps, iterations=iterations,
                             schedule=schedule, pinned=rng.random() < 0.4, colliders=rng.choice(("plane", "boxes"))))
    if kind == "sphere":
        return _drawn(_scene("", "sphere", rng.randint(2, 4), bodies=log_int(1, 40), steps=steps, iterations=iterations,
                             schedule=schedule))
    if kind == "mixed":
        return _drawn(_scene("", "mixed", log_int(16, 128), bodies=log_int(8, 1024), steps=rng.choice((1, 2)),
                             iterations=5, frames=log_int(1, 12), schedule=schedule))
    if kind == "large":
        if rng.random() < 0.5:
            return _drawn(_scene("", "cloth", log_int(160, 384), log_int(160, 384), steps=rng.choice((1, 2)),
                                 iterations=rng.choice((4, 5, 8)), schedule=schedule,
                                 colliders=rng.choice(("plane", "spheres"))))
        return _drawn(_scene("", "cube", log_int(24, 44), steps=rng.choice((1, 2)), iterations=rng.choice((4, 5, 8)),
                             schedule=schedule, pinned=rng.random() < 0.5, colliders=rng.choice(("plane", "boxes"))))
    shape = rng.choice(("cloth", "cloth", "bends", "tets"))
    n = {"cloth": log_int(8, 72), "bends": log_int(6, 24), "tets": log_int(2, 7)}[shape]
    bodies = log_int(1, 64) if shape == "cloth" else log_int(1, 16)
    frames = log_int(4, 60) if shape == "cloth" else log_int(3, 12)
    return _drawn(_rollout("", shape, n, bodies, frames, iterations=rng.choice((3, 5, 5)), backward=rng.random() < 0.75))


def _drawn(case):
    del case["name"]
    return case


# ------------------------------------------------------------------ inputs
def _log_uniform(rng, lo, hi, size=None):
    return np.exp(rng.uniform(np.log(lo), np.log(hi), size=size)).astype(np.float32)


def _shapes(case):
    """(shape, n, m) of every body: the sizes belong to the case, not to the seed."""
    if case["shape"] != "mixed":
        return [(case["shape"], case["n"], case["m"])] * case["bodies"]
    r = random.Random("%d of up to %d" % (case["bodies"], case["n"]))
    out = []
    for _ in range(case["bodies"]):
        u = r.random()
        if u < 0.6:
            n = int(round(8.0 * (case["n"] / 8.0) ** r.random()))
            out.append(("cloth", n, n))
        elif u < 0.9:
            out.append(("cube", r.randint(4, max(5, min(16, case["n"] // 8))), 0))
        else:
            out.append(("sphere", r.randint(2, 3 if case["n"] < 64 else 4), 0))
    return out


def _mesh(shape, n, m, pinned, rng):
    """MeshSpec of one shape: wrinkled cloths (no hinge starts flat), 5-tet cubes, spheres."""
    if shape == "cloth":
        pins = ((m - 1) * n, m * n - 1) if pinned else ()
        v, f = scenes.cloth(n, 0.05, 100.0, pinned=pins, jitter=0.005, seed=int(rng.integers(1 << 30)), nz=m)
        v["vel"] = rng.uniform(-0.1, 0.1, (len(v), 3)).astype(np.float32)
        return scenes.MeshSpec(vertices=v, faces=f, attrs=scenes.attrs(1e-4, 1e-4, 1e-3), bend_type=BEND_DIHEDRAL)
    if shape == "sphere":
        v, f = scenes.icosphere(n, radius=1.0, inv_mass=1.0)
        v["vel"] = rng.uniform(-0.1, 0.1, (len(v), 3)).astype(np.float32)
        return scenes.MeshSpec(vertices=v, faces=f, attrs=scenes.attrs(1e-4, 1e-4, 1e-3), bend_type=BEND_DIHEDRAL)
    v, e, t = scenes.tet_cube(n, 0.1, inv_mass=1.0, compliance=1e-5, jitter=0.002, seed=int(rng.integers(1 << 30)))
    v["vel"] = rng.uniform(-0.1, 0.1, (len(v), 3)).astype(np.float32)
    flags = scenes.CALC_EDGE_LENGTHS | scenes.CALC_VOLUMES | scenes.OPTIMIZE
    if not pinned:
        return scenes.MeshSpec(vertices=v, edges=e, volumes=t, flags=flags)
    g = n + 1
    top = n * g * g
    v["inv_mass"][top:] = 0.0
    v["vel"][top:] = 0.0
    lra = np.zeros(top, LRA)
    lra["v"][:, 0] = top + np.arange(top) % (g * g)
    lra["v"][:, 1] = np.arange(top)
    return scenes.MeshSpec(vertices=v, edges=e, volumes=t, lras=lra, flags=flags | scenes.CALC_LRA_LENGTHS)


def _bodies(case, seed):
    """[(settings index, position, rotation, parameters)] and the distinct settings arrays."""
    rng = np.random.default_rng([seed, case["bodies"], case["n"]])
    settings, index, bodies = [], {}, []
    shapes = _shapes(case)
    side = max(1, int(np.ceil(len(shapes) ** 0.5)))
    for k, key in enumerate(shapes):
        if key not in index:
            s = build_settings(_mesh(*key, case["pinned"], rng))
            for array in (s.edges, s.bends, s.volumes):
                array["compliance"] = _log_uniform(rng, 1e-6, 1e-3)
            index[key] = len(settings)
            settings.append(s)
        shape, n, m = key
        extent = {"cloth": 0.05 * max(n, m), "cube": 0.1 * n, "sphere": 2.0}[shape]
        height = 1.2 if shape == "sphere" else 0.6 * extent + 0.1
        pos = (8.0 * (k % side), 8.0 * (k // side), height + float(rng.uniform(0.0, 0.2)))
        rot = (0.0, 0.0, 0.0, 1.0) if case["pinned"] or len(shapes) == 1 else scenes.random_quaternion(rng)
        params = BodyParams(num_iterations=case["iterations"], allow_sleeping=False,
                            pressure=float(rng.uniform(500, 2000)) if shape == "sphere" else 0.0)
        bodies.append((index[key], pos, rot, params))
    return settings, bodies


def _colliders(case, seed):
    rng = np.random.default_rng([seed, 77])
    half = {"cloth": 0.025 * case["n"], "cube": 0.05 * case["n"]}.get(case["shape"], 1.0)
    out = []
    if case["colliders"] == "box":
        out.append(Collider(SHAPE_BOX, (0.5, 0.5, 0.1), pos=(0.0, 0.0, -0.6)))
    else:
        out.append(Collider(SHAPE_PLANE, (0.0, 0.0, 1.0, 0.0, 1000.0)))
    if case["colliders"] == "spheres":
        # below the cloth's start, so that it falls onto them
        for _ in range(64):
            p = rng.uniform(-half, half, 2)
            r = float(rng.uniform(0.1, 0.4))
            out.append(Collider(SHAPE_SPHERE, (r,), pos=(float(p[0]), float(p[1]), 1.2 * half - r - float(rng.uniform(0.0, 0.3)))))
    if case["colliders"] == "boxes":
        # around the block, touching its sides as it swings
        for _ in range(256):
            he = tuple(float(x) for x in rng.uniform(0.1, 0.5, 3))
            angle = float(rng.uniform(0.0, 2.0 * np.pi))
            r = half + float(np.linalg.norm(he)) + float(rng.uniform(0.0, 3.0))
            d = max(abs(np.cos(angle)), abs(np.sin(angle)))
            out.append(Collider(SHAPE_BOX, he, pos=(float(r * np.cos(angle) / d), float(r * np.sin(angle) / d), float(rng.uniform(0.0, 2.4 * half))),
                                rot=scenes.random_quaternion(rng)))
    for c in out:
        c.bounds = scenes.collider_world_bounds(c)
    return out


def _rollout_case(case, seed):
    if case["shape"] == "tets":
        return scenes.rollout_tet_block(case["bodies"], case["n"], frames=case["frames"], seed=seed)
    n = case["n"]
    bends = case["shape"] == "bends"
    v, f = scenes.cloth(n, 0.05, 100.0, pinned=((n - 1) * n, n * n - 1), jitter=0.01 if bends else 0.0, seed=seed)
    mesh = scenes.MeshSpec(vertices=v, faces=f, bend_type=BEND_DIHEDRAL if bends else BEND_NONE,
                           attrs=scenes.attrs(1e-3, 1e-3, 1e-3 if bends else 0.0, lra_type=LRA_EUCLIDEAN if bends else LRA_NONE))
    rng = np.random.default_rng([seed, n])
    edges = len(build_settings(mesh).edges)
    comp = (1e-3 * rng.uniform(0.5, 2.0, case["bodies"] * edges)).astype(np.float32)
    vel = rng.uniform(-0.1, 0.1, (case["bodies"] * n * n, 3)).astype(np.float32)
    return scenes.RolloutCase("rollout", mesh, case["bodies"], case["frames"], case["iterations"], DT, GRAVITY, comp, vel,
                              np.ones_like(comp))


def prepare(case, seed):
    ctx = Context(0)
    ctx.set_gravity(GRAVITY)
    if case["kind"] == "rollout":
        rc = _rollout_case(case, seed)
        st = ctx.create_settings(build_settings(rc.mesh))
        r = ctx.create_rollout([st] * case["bodies"], num_iterations=case["iterations"], dt=DT, frames=case["frames"])
        rng = np.random.default_rng([seed, 5])
        device = torch.device("cuda")
        comp = torch.from_numpy(rc.compliance).to(device).requires_grad_(case["backward"])
        vel = torch.from_numpy(np.ascontiguousarray(rc.velocity.reshape(-1))).to(device).requires_grad_(case["backward"])
        grad = torch.from_numpy(rng.standard_normal((r.num_vertices, 3)).astype(np.float32)).to(device)
        return {"case": case, "ctx": ctx, "rollout": r, "compliance": comp, "velocity": vel, "grad": grad}
    settings, bodies = _bodies(case, seed)
    ctx.set_colliders(_colliders(case, seed))
    handles = [ctx.create_settings(s, case["schedule"]) for s in settings]
    ids = []
    for k, pos, rot, params in bodies:
        body = ctx.create_body(handles[k], pos, rot, params)
        if case["schedule"] == "coloured" and len(settings[k].vertices) > 40000:
            ctx.set_tail_mode(body, True)       # a team colours its last group too
        ids.append(body)
    # a running simulation: the first frame has laid the bodies out on the device
    ctx.update(DT, case["steps"], 1)
    ctx.synchronize()
    return {"case": case, "ctx": ctx, "ids": ids}


def run(state):
    case = state["case"]
    if case["kind"] == "rollout":
        if not case["backward"]:
            with torch.no_grad():
                return {"x": rollout(state["compliance"], state["velocity"], state["rollout"])}
        x = rollout(state["compliance"], state["velocity"], state["rollout"])
        dc, dv = torch.autograd.grad(x, (state["compliance"], state["velocity"]), state["grad"])
        return {"x": x.detach(), "grad_compliance": dc, "grad_velocity": dv}
    ctx = state["ctx"]
    ctx.update(DT, case["steps"], case["frames"])
    got = [ctx.read(b) for b in state["ids"]]
    if len(got) == 1:
        return {k: got[0][k] for k in ("pos", "vel", "body_pos")}
    return {k: np.concatenate([g[k] for g in got]) for k in ("pos", "vel", "body_pos")}


# ------------------------------------------------------------------ what a pass needs
def _counts(shape, n, m, pinned):
    """(vertices, edges, bends, volumes, long-range attachments), closed forms."""
    if shape == "cloth":
        quads = (n - 1) * (m - 1)
        # structural edges and one diagonal per quad; a wrinkled sheet has part of the other
        # diagonals too (a flat one all of them), which are left out here
        return n * m, n * (m - 1) + m * (n - 1) + quads, 3 * quads - n - m + 2, 0, 0
    if shape == "sphere":
        faces = 20 * 4 ** n
        return faces // 2 + 2, 3 * faces // 2, 3 * faces // 2, 0, 0
    edges = 3 * n * (n + 1) ** 2 + 3 * n * n * (n + 1)
    return (n + 1) ** 3, edges, 0, 5 * n ** 3, n * (n + 1) ** 2 if pinned else 0


def work(case):
    # each body's state in and out once per pass (position, velocity, inverse mass), its
    # constraint records once; 40 operations per edge, 190 per bend, 110 per volume, 20 per
    # attachment, 40 per vertex and sub-step (twice that and a second sweep for an adjoint)
    if case["kind"] == "rollout":
        n = case["n"]
        if case["shape"] == "tets":
            v, e, b, t, a = _counts("cube", n, 0, False)
        else:
            v, e, b, t, a = _counts("cloth", n, n, True)
            if case["shape"] == "cloth":
                b = 0
            else:
                a = n * n - 2
        subs = case["bodies"] * case["frames"] * case["iterations"] * (3 if case["backward"] else 1)
        state = v * (12 + 12 + 4) + e * 4
        return {"bytes": case["bodies"] * (state * (2 if case["backward"] else 1) + 12 * v),
                "flops": subs * (40 * e + 190 * b + 110 * t + 20 * a + 40 * v)}
    total = {"bytes": 0, "flops": 0}
    subs = case["frames"] * case["steps"] * case["iterations"]
    for shape, n, m in _shapes(case):
        v, e, b, t, a = _counts(shape, n, m, case["pinned"])
        total["bytes"] += v * (28 + 24) + 16 * e + 24 * (b + t) + 12 * a
        total["flops"] += subs * (40 * e + 190 * b + 110 * t + 20 * a + 40 * v)
    return total


def tolerance(case):
    # the update restates the reference's float operations in its order, bit for bit, whatever
    # the schedule: any other result is another simulation.  A gradient's sums may be taken in
    # another order.
    if case["kind"] == "scene" or not case["backward"]:
        return "exact"
    return {"rel": 1e-5, "max": 1e-3}


# ------------------------------------------------------------------ the same in 64 bits
def _program(parts):
    """Levels of a body list's constraints: parts of (settings, first vertex, first edge).
    Within a body the update groups run one after the other, each its volumes, bends, edges and
    attachments; a constraint waits for the ones before it that share a vertex either writes."""
    levels = []
    for s, voff, eoff in parts:
        wrote, read = [0] * len(s.vertices), [0] * len(s.vertices)
        begin = {"volume": 0, "bend": 0, "edge": 0, "lra": 0}
        arrays = {"volume": s.volumes, "bend": s.bends, "edge": s.edges, "lra": s.lras}
        lists = {k: a["v"].tolist() for k, a in arrays.items()}
        for g in s.groups:
            for kind in ("volume", "bend", "edge", "lra"):
                end = int(g[kind + "_end"])
                for c in range(begin[kind], end):
                    v = lists[kind][c]
                    w = v[1:] if kind == "lra" else v
                    lv = max(max(wrote[i] for i in v), max(read[i] for i in w))
                    if lv >= len(levels):
                        levels.append({})
                    levels[lv].setdefault((kind, id(s), voff, eoff), (s, []))[1].append(c)
                    for i in v:
                        read[i] = max(read[i], lv + 1)
                    for i in w:
                        wrote[i] = max(wrote[i], lv + 1)
                begin[kind] = end
    out = []
    for level in levels:
        merged = {}
        for (kind, _, voff, eoff), (s, rows) in level.items():
            a = {"volume": s.volumes, "bend": s.bends, "edge": s.edges, "lra": s.lras}[kind][rows]
            p = {"volume": ("six_rest_volume", "compliance"), "bend": ("compliance", "initial_angle"),
                 "edge": ("rest", "compliance"), "lra": ("max_distance", "max_distance")}[kind]
            merged.setdefault(kind, []).append((a["v"].astype(np.int64) + voff, np.stack([a[p[0]], a[p[1]]]).astype(np.float64),
                                                np.array(rows, np.int64) + eoff))
        out.append([(k, torch.from_numpy(np.concatenate([r[0] for r in rows])),
                     torch.from_numpy(np.concatenate([r[1] for r in rows], axis=1)),
                     torch.from_numpy(np.concatenate([r[2] for r in rows]))) for k, rows in merged.items()])
    return out


def _project(x, w, kind, idx, par, compliance, inv_dt_sq):
    """Positions of one level's vertices after its constraints (XPBD, zero accumulated lambda)."""
    p = [x[idx[:, k]] for k in range(idx.shape[1])]
    ww = [w[idx[:, k], None] for k in range(idx.shape[1])]

    def dot(a, b):
        return (a * b).sum(1, keepdim=True)

    if kind == "lra":
        d = p[1] - p[0]
        length = dot(d, d).sqrt()
        far = length > par[0][:, None]
        return x.index_put((idx[:, 1],), torch.where(far, p[0] + d * par[0][:, None] / torch.where(far, length, 1.0), p[1]))
    if kind == "edge":
        d = p[1] - p[0]
        length = dot(d, d).sqrt()
        denom = length * (ww[0] + ww[1] + compliance * inv_dt_sq)
        c = d * (length - par[0][:, None]) / denom
        grads, lam = [c, -c], -1.0
    elif kind == "volume":
        a, b, c = p[1] - p[0], p[2] - p[0], p[3] - p[0]
        violation = dot(torch.linalg.cross(a, b), c).abs() - par[0][:, None]
        grads = [torch.linalg.cross(p[3] - p[1], p[2] - p[1]), torch.linalg.cross(b, c), torch.linalg.cross(c, a), torch.linalg.cross(a, b)]
        lam = violation / (sum(wk * dot(g, g) for wk, g in zip(ww, grads)) + compliance * inv_dt_sq)
    else:
        e = p[1] - p[0]
        el = dot(e, e).sqrt()
        a, b = p[2] - p[1], p[3] - p[1]
        n1, n2 = torch.linalg.cross(p[2] - p[0], a), torch.linalg.cross(b, p[3] - p[0])
        s1, s2 = dot(n1, n1), dot(n2, n2)
        sign = torch.where(dot(torch.linalg.cross(n2, n1), e) < 0, -1.0, 1.0)
        d = dot(n1, n2) / (s1 * s2).sqrt()
        ax = d.abs().clamp(max=1.0)
        angle = (1.0 - ax).sqrt() * (np.pi / 2 - 0.175394 * ax)
        angle = torch.where(d < 0, np.pi - angle, angle)
        c = sign * angle - par[1][:, None]
        c = torch.where(c > np.pi, c - 2 * np.pi, torch.where(c < -np.pi, c + 2 * np.pi, c))
        n1, n2 = n1 / s1, n2 / s2
        g0 = (dot(a, e) * n1 + dot(b, e) * n2) / el
        g2, g3 = el * n1, el * n2
        grads = [g0, -g0 - g2 - g3, g2, g3]
        lam = c / (sum(wk * dot(g, g) for wk, g in zip(ww, grads)) + compliance * inv_dt_sq)
    return x.index_put((idx.reshape(-1),), torch.stack([pk - lam * wk * g for pk, wk, g in zip(p, ww, grads)], 1).reshape(-1, 3))


def exact(case, seed):
    most = 3e7 if case["kind"] == "rollout" else 1.2e8     # what plain torch takes in 20 seconds
    if work(case)["flops"] > most or case["kind"] == "scene" and (
            case["schedule"] != "exact" or case["colliders"] in ("spheres", "boxes")):
        return None
    if case["kind"] == "rollout":
        return _exact_rollout(case, seed)
    settings, bodies = _bodies(case, seed)
    parts, voff = [], 0
    x, v, w, start, count = [], [], [], [], []
    for k, pos, rot, _ in bodies:
        s = settings[k]
        r = torch.from_numpy(scenes._rot_matrix(np.float64(np.float32(rot))))
        parts.append((s, voff, 0))
        x.append(torch.from_numpy(s.vertices["pos"].astype(np.float64)) @ r.T)
        v.append(torch.from_numpy(s.vertices["vel"].astype(np.float64)) @ r.T)
        w.append(torch.from_numpy(s.vertices["inv_mass"].astype(np.float64)))
        start.append(np.float64(np.float32(pos)))
        count.append(len(s.vertices))
        voff += count[-1]
    x, v, w = torch.cat(x), torch.cat(v), torch.cat(w)
    body = torch.repeat_interleave(torch.arange(len(bodies)), torch.tensor(count))
    at = torch.from_numpy(np.array(start))
    program = _program(parts)
    its = case["iterations"]
    h = DT / case["steps"] / its
    move = (w > 0)[:, None]
    g = torch.tensor(GRAVITY, dtype=torch.float64)
    faces = [(torch.from_numpy(settings[k].faces["v"].astype(np.int64)) + p[1], prm.pressure)
             for (k, _, _, prm), p in zip(bodies, parts) if prm.pressure > 0]
    friction, touch = 0.2, case["colliders"] == "plane"
    for _ in range((1 + case["frames"]) * case["steps"]):
        for _ in range(its):
            for f, pressure in faces:
                a, b, c = x[f[:, 0]], x[f[:, 1]], x[f[:, 2]]
                six = (torch.linalg.cross(a, b) * c).sum()
                if six > 0:
                    imp = pressure * h / six * torch.linalg.cross(b - a, c - a)
                    for k in range(3):
                        v = v.index_add(0, f[:, k], imp * w[f[:, k], None])
            v = torch.where(move, (v + g * h) * (1.0 - 0.1 * h), v)
            before = x
            x = x + v * h
            for level in program:
                for kind, idx, par, _ in level:
                    c = par[0 if kind == "bend" else 1][:, None]
                    x = _project(x, w, kind, idx, par, c, 1.0 / (h * h))
            v = torch.where(move, (x - before) / h, v)
            if touch:       # the ground plane z = 0: push out, friction, no bounce
                depth = -(x[:, 2] + at[body, 2])
                hit = (depth > 0) & (w > 0)
                vt = v.clone()
                vt[:, 2] = 0
                speed = vt.norm(dim=1)
                f = (friction * depth / (speed.clamp(min=1e-300) * h)).clamp(max=1.0)
                slow = vt * (1.0 - f)[:, None]
                x = torch.where(hit[:, None], x + depth[:, None] * torch.tensor([0.0, 0.0, 1.0], dtype=torch.float64), x)
                v = torch.where(hit[:, None], slow, v)
        for k in range(len(bodies)):
            sel = slice(parts[k][1], parts[k][1] + count[k])
            d = 0.5 * (x[sel].min(0).values + x[sel].max(0).values)
            x[sel] -= d
            at[k] += d
    return {"pos": x.numpy(), "vel": v.numpy(), "body_pos": at.numpy().reshape(-1)}


def _exact_rollout(case, seed):
    rc = _rollout_case(case, seed)
    s = build_settings(rc.mesh)
    nv, ne = len(s.vertices), len(s.edges)
    parts = [(s, k * nv, k * ne) for k in range(case["bodies"])]
    program = _program(parts)
    x = torch.from_numpy(np.tile(s.vertices["pos"].astype(np.float64), (case["bodies"], 1)))
    w = torch.from_numpy(np.tile(s.vertices["inv_mass"].astype(np.float64), case["bodies"]))
    comp = torch.from_numpy(rc.compliance.astype(np.float64)).requires_grad_(case["backward"])
    vel = torch.from_numpy(rc.velocity.astype(np.float64).reshape(-1)).requires_grad_(case["backward"])
    v = vel.reshape(-1, 3)
    h = DT / case["iterations"]
    move = (w > 0)[:, None]
    g = torch.tensor(GRAVITY, dtype=torch.float64)
    for _ in range(case["frames"] * case["iterations"]):
        v = torch.where(move, (v + g * h) * (1.0 - 0.1 * h), v)
        before = x
        x = x + v * h
        for level in program:
            for kind, idx, par, edge in level:
                c = comp[edge][:, None] if kind == "edge" else par[0 if kind == "bend" else 1][:, None]
                x = _project(x, w, kind, idx, par, c, 1.0 / (h * h))
        v = torch.where(move, (x - before) / h, v)
    if not case["backward"]:
        return {"x": x.numpy()}
    rng = np.random.default_rng([seed, 5])
    grad = torch.from_numpy(rng.standard_normal(tuple(x.shape)).astype(np.float32).astype(np.float64))
    dc, dv = torch.autograd.grad(x, (comp, vel), grad)
    return {"x": x.detach().numpy(), "grad_compliance": dc.numpy(), "grad_velocity": dv.numpy()}
