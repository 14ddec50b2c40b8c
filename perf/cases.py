"""What the framework's speed is measured on: calls of its public entry points at the sizes they are
used at, from one falling box to a field of 393,216 bodies.

A case is a dict of plain values. Its "kind" names the call:

  frame    one step of a small world and its body states, the loop of a game or a viewer
  rollout  a world put back to a saved state, stepped "steps" times, and its body states read: what
           a planner, a search or a parameter sweep does
  pile     "steps" steps of a heap that has come to rest against its container, and its states
  grad     autograd.Rollout forward and backward: final states, dL/d state0, dL/d friction
  collide  the stateless narrowphase over fixture pairs
  pairs    the stateless pair search over fat AABBs

`listed()` holds twelve of them, `draw(rng)` gives more over the same ranges. Scenes are those of
b2g.scenes (the sizes of its benchmark and tests) with the case's seed.
"""
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "box2d-rs_amd"))

import b2g  # noqa: E402
from b2g import autograd, scenes  # noqa: E402

DT = 1.0 / 60.0
POLYGON_RADIUS = 0.01  # B2_POLYGON_RADIUS


def listed():
    return [
        # The smallest world there is: one box on the ground, stepped once a frame with the settings
        # of B2world::new but for sleeping (asleep it would not be solved at all). Latency and
        # launches are all there is.
        {"name": "frame_box", "kind": "frame", "scene": "box", "n": 1, "continuous": True},
        # The testbed's 20-row pyramid, 210 boxes: an ordinary game frame, two-point contacts.
        {"name": "frame_pyramid", "kind": "frame", "scene": "pyramid", "n": 20, "continuous": True},
        # Stacks of boxes with every default on (sleeping, continuous physics): a level loaded from
        # its saved state and run until the stacks fall asleep (half a second, 30 steps).
        {"name": "stacks_1531", "kind": "rollout", "scene": "stacks", "n": 1531, "steps": 40, "warm": 5,
         "sleep": True, "continuous": True},
        # The benchmark's window: 65,536 mixed bodies in free fall, steps 6 to 25.
        {"name": "field_65536", "kind": "rollout", "scene": "field", "n": 65536, "steps": 20, "warm": 5,
         "sleep": False, "continuous": False},
        # The same field six times as large: the throughput end.
        {"name": "field_393216", "kind": "rollout", "scene": "field", "n": 393216, "steps": 20, "warm": 5,
         "sleep": False, "continuous": False},
        # A settled heap: one island of tens of thousands of contacts, the dense solve.
        {"name": "pile_32768", "kind": "pile", "scene": "heap", "n": 32768, "steps": 10, "warm": 300},
        # The field landing with continuous physics on (the reference's default): hundreds of times
        # of impact a step.
        {"name": "landing_65536", "kind": "rollout", "scene": "landing", "n": 65536, "steps": 4, "warm": 215,
         "sleep": False, "continuous": True},
        # Many worlds of 16 to 1024 bodies stepped together: training of a policy, a sweep.
        {"name": "batch_1024", "kind": "pile", "scene": "batch", "n": 1024, "steps": 10, "warm": 150},
        # Hanging chains of revolute joints swinging down.
        {"name": "chains_1024", "kind": "rollout", "scene": "chains", "n": 1024, "steps": 20, "warm": 10,
         "sleep": False, "continuous": False},
        # Gradients through 30 steps of 192 worlds of 64 bodies.
        {"name": "grad_192x64", "kind": "grad", "n": 192, "bodies": 64, "steps": 30},
        # 60,000 shape pairs near contact (the no-allocation entry point's range is up to 65,536).
        {"name": "collide_60000", "kind": "collide", "n": 60000},
        # Pair search over the fat AABBs of 50,003 proxies.
        {"name": "pairs_50003", "kind": "pairs", "n": 50003},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["frame", "stacks", "field", "heap", "landing", "batch", "chains", "grad", "collide", "pairs"])
    if kind == "frame":
        return {"kind": "frame", "scene": "pyramid", "n": rng.randint(2, 24), "continuous": rng.random() < 0.5}
    if kind == "stacks":
        return {"kind": "rollout", "scene": "stacks", "n": _log(rng, 20, 6000), "steps": rng.randint(35, 45), "warm": 5,
                "sleep": True, "continuous": rng.random() < 0.7}
    if kind == "field":
        return {"kind": "rollout", "scene": "field", "n": _log(rng, 300, 300000), "steps": rng.randint(10, 25),
                "warm": 5, "sleep": rng.random() < 0.3, "continuous": False}
    if kind == "heap":
        return {"kind": "pile", "scene": "heap", "n": _log(rng, 200, 32000), "steps": rng.randint(5, 12), "warm": 300}
    if kind == "landing":
        return {"kind": "rollout", "scene": "landing", "n": _log(rng, 2000, 60000), "steps": rng.randint(2, 4),
                "warm": rng.randint(205, 215), "sleep": False, "continuous": True}
    if kind == "batch":
        return {"kind": "pile", "scene": "batch", "n": _log(rng, 20, 1024), "steps": rng.randint(5, 12), "warm": 150}
    if kind == "chains":
        return {"kind": "rollout", "scene": "chains", "n": _log(rng, 8, 1024), "steps": rng.randint(10, 25), "warm": 10,
                "sleep": False, "continuous": False}
    if kind == "grad":
        return {"kind": "grad", "n": _log(rng, 4, 192), "bodies": rng.randint(5, 64), "steps": rng.randint(10, 30)}
    if kind == "collide":
        return {"kind": "collide", "n": _log(rng, 100, 65536)}
    return {"kind": "pairs", "n": _log(rng, 500, 60000)}


# ---- worlds ----------------------------------------------------------------------------------
def _scene(case, seed):
    """(scene, batched, joints) of a case."""
    kind, n = case["scene"], case["n"]
    rng = np.random.default_rng(seed)
    if kind == "box":
        sc = scenes.hello_world()
        sc.body_defs["position"][1] += rng.uniform(-0.5, 0.5, 2).astype(np.float32)
        return sc, False, None
    if kind == "pyramid":
        sc = scenes.pyramid(rows=n)
        k = len(sc.body_defs) - 1
        sc.body_defs["position"][1:, 0] += rng.uniform(-0.01, 0.01, k).astype(np.float32)
        return sc, False, None
    if kind == "stacks":
        sc = scenes.stack_world(n, seed)
        sc.body_defs["linear_velocity"][1:, 0] += rng.uniform(-0.02, 0.02, n).astype(np.float32)
        return sc, False, None
    if kind == "field":
        # the grid of the benchmark's world in a box that leaves the same gap around it
        return scenes.large_world(n, seed=seed, half_extent=0.6 * np.ceil(np.sqrt(n)) + 46.4), False, None
    if kind == "landing":
        # the lowest row reaches the floor 182 steps after the start
        return scenes.large_world(n, seed=seed, half_extent=0.6 * np.ceil(np.sqrt(n)) + 46.4), False, None
    if kind == "heap":
        # a little over twice as wide as high
        return scenes.heap_world(n, seed, half_extent=max(4.0, 0.9 * np.sqrt(n))), False, None
    if kind == "batch":
        return _batch(n, seed), True, None
    sc, joints = scenes.chains(n, 16)
    sc.body_defs["linear_velocity"][1 + n:] = rng.uniform(-0.5, 0.5, (16 * n, 2))
    return sc, False, joints


def _batch(n, seed):
    """The worlds of scenes.batched_worlds (16 to 1024 bodies, heaps and stacks by turns) with the same
    sizes for every seed, spread evenly over their logarithm."""
    u = np.random.default_rng(9).permutation(n) + 0.5
    sizes = np.round(16.0 * 64.0 ** (u / n)).astype(int)
    parts, worlds = [], []
    for i, k in enumerate(sizes):
        make = scenes.stack_world if i % 2 else scenes.heap_world
        sc = make(int(k), scenes.world_seed(seed & 0x7FFFFFFF, i), half_extent=20.0)
        parts.append(sc[:4])
        worlds.append(np.full(len(sc.body_defs), i, np.int32))
    bd, fb, sd, fd = scenes.concat(*parts)
    return scenes.BatchScene(bd, np.concatenate(worlds), fb, sd, fd, {})


def _world(case, seed):
    sc, batched, joints = _scene(case, seed)
    w = b2g.World()
    w.set_flags(warm_starting=True, allow_sleep=bool(case.get("sleep", False)), continuous=False, block_solve=True)
    if batched:
        w.add_batched(sc.body_defs, sc.body_world, sc.fixture_body, sc.shape_defs, sc.fixture_defs)
    else:
        w.add(sc.body_defs, sc.fixture_body, sc.shape_defs, sc.fixture_defs)
    if joints is not None:
        w.add_joints(joints)
    return w


def _states(st):
    """The columns of the body-state records: pose (m_xf, sweep centre and angle), velocity, sleep."""
    f = st.view(np.float32).reshape(len(st), 16)
    return {"pose": f[:, 0:7], "velocity": f[:, 7:10], "sleep": f[:, 13:15]}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "collide":
        return _prepare_collide(case, seed)
    if kind == "pairs":
        return _prepare_pairs(case, seed)
    if kind == "grad":
        return _prepare_grad(case, seed)
    w = _world(case, seed)
    on = dict(warm_starting=True, allow_sleep=bool(case.get("sleep", False)),
              continuous=bool(case.get("continuous", False)), block_solve=True)
    if kind == "frame":
        w.set_flags(**on)
        for _ in range(90):  # the bodies come to rest
            w.step(DT, 8, 3)
        w.body_states()
        return {"kind": kind, "world": w, "steps": 1}
    before = 175 if case["scene"] == "landing" else case["warm"]  # free fall: nothing to hit yet
    for _ in range(before):
        w.step(DT, 8, 3)
    w.set_flags(**on)
    for _ in range(case["warm"] - before):
        w.step(DT, 8, 3)
    s = {"kind": kind, "world": w, "steps": case["steps"]}
    st = w.body_states()
    if kind == "rollout":
        s["states"], s["fat"] = st, w.fat_aabbs()
    return s


def run(s):
    kind, w = s["kind"], s["world"]
    if kind in ("frame", "rollout", "pile"):
        if kind == "rollout":
            w.set_body_states(s["states"])
            w.set_fat_aabbs(s["fat"])
        for _ in range(s["steps"]):
            w.step(DT, 8, 3)
        return _states(w.body_states())
    if kind == "grad":
        state0, friction = s["state0"], s["friction"]
        final = autograd.Rollout.apply(w, state0, friction, s["steps"])
        loss = ((final[s["body0"], 0:2] - s["goal"]) ** 2).sum()
        gs, gf = torch.autograd.grad(loss, (state0, friction))
        return {"final": final.detach(), "grad_state": gs, "grad_friction": gf}
    if kind == "collide":
        m = w.collide_pairs(s["pairs"], s["xa"], s["xb"])
        return {"type": m["type"], "count": m["point_count"], "normal": m["local_normal"], "point": m["local_point"],
                "points": m["points"]["local_point"], "id": m["points"]["id"].view(np.int32)}
    return {"pairs": w.broadphase_pairs(s["fat"])}


def _prepare_grad(case, seed):
    n, bodies = case["n"], case["bodies"]
    b = scenes.differentiable_worlds(n, bodies, config=seed & 0x7FFFFFFF)
    w = b2g.World()
    w.set_flags(warm_starting=True, allow_sleep=False, continuous=False, block_solve=True)  # a tape needs these
    w.add_batched(b.body_defs, b.body_world, b.fixture_body, b.shape_defs, b.fixture_defs)
    for _ in range(60):  # the bodies have dropped onto each other
        w.step(DT, 8, 3)
    dev = torch.device("cuda")
    state0 = torch.from_numpy(autograd.state6(w.body_states())).to(dev).requires_grad_(True)
    friction = torch.from_numpy(b.fixture_defs["friction"].copy()).to(dev).requires_grad_(True)
    return {"kind": "grad", "world": w, "steps": case["steps"], "state0": state0, "friction": friction,
            "body0": torch.from_numpy(b.meta["body0"]).to(dev),
            "goal": torch.from_numpy(b.meta["goal"].astype(np.float32)).to(dev)}


# ---- the stateless entry points -----------------------------------------------------------------
def _shapes(n, rng):
    """The mix of the large world: half circles (radius 0.25 to 0.5), three tenths boxes (half
    extents 0.25 to 0.5), the rest convex polygons of 3 to 8 vertices. Vertices in float32, the rows
    of the shorter polygons filled up with their last vertex."""
    kind = rng.choice(3, n, p=[0.5, 0.3, 0.2])  # circle, box, polygon
    radius = rng.uniform(0.25, 0.5, n).astype(np.float32)
    h = rng.uniform(0.25, 0.5, (n, 2)).astype(np.float32)
    nv = np.where(kind == 1, 4, rng.integers(3, 9, n))
    k = np.minimum(np.arange(8)[None, :], nv[:, None] - 1)
    jitter = np.take_along_axis(rng.uniform(-0.25, 0.25, (n, 8)), k, 1)
    ang = 2.0 * np.pi * (k + jitter) / nv[:, None]
    v = np.stack([radius[:, None] * np.cos(ang), radius[:, None] * np.sin(ang)], 2).astype(np.float32)
    corner = np.array([[-1, -1], [1, -1], [1, 1], [-1, 1]], np.float32)[np.minimum(np.arange(8), 3)]
    v[kind == 1] = corner[None] * h[kind == 1][:, None, :]
    return kind, radius, h, nv, v


def _collide_inputs(case, seed):
    """Shapes, pairs (the polygon first) and transforms of pairs at 0.5 to 1.05 of touching distance."""
    n = case["n"]
    rng = np.random.default_rng([7, seed])
    nf = max(4, n // 3)
    shapes = _shapes(nf, rng)
    kind, radius, v = shapes[0], shapes[1], shapes[4]
    pairs = rng.integers(0, nf, (n, 2)).astype(np.int32)
    pairs[:, 1] = np.where(pairs[:, 0] == pairs[:, 1], (pairs[:, 1] + 1) % nf, pairs[:, 1])
    swap = (kind[pairs[:, 0]] == 0) & (kind[pairs[:, 1]] != 0)
    pairs[swap] = pairs[swap][:, ::-1]
    reach = np.where(kind == 0, radius, 0.85 * np.hypot(v[..., 0], v[..., 1]).max(1))
    xf = []
    for c in range(2):
        a = rng.uniform(-np.pi, np.pi, n)
        p = rng.uniform(-50.0, 50.0, (n, 2)) if c == 0 else xf[0][:, :2].astype(np.float64)
        if c == 1:
            d = rng.uniform(0.5, 1.05, n) * (reach[pairs[:, 0]] + reach[pairs[:, 1]])
            t = rng.uniform(0.0, 2.0 * np.pi, n)
            p = p + np.stack([d * np.cos(t), d * np.sin(t)], 1)
        xf.append(np.concatenate([p, np.sin(a)[:, None], np.cos(a)[:, None]], 1).astype(np.float32))
    return shapes, pairs, xf[0], xf[1]


def _prepare_collide(case, seed):
    (kind, radius, h, nv, v), pairs, xa, xb = _collide_inputs(case, seed)
    n = len(kind)
    sd = np.zeros(n, b2g.SHAPE_DEF)
    sd["type"] = np.choose(kind, [b2g.SHAPE_CIRCLE, b2g.SHAPE_BOX, b2g.SHAPE_POLYGON])
    sd["radius"] = np.where(kind == 0, radius, 0.0)
    sd["count"] = np.where(kind == 2, nv, 0)
    sd["params"][kind == 1, :2] = h[kind == 1]
    sd["params"][kind == 2, :16] = v[kind == 2].reshape(-1, 16)
    w = _loose_world(n, sd)
    return {"kind": "collide", "world": w, "pairs": pairs, "xa": xa, "xb": xb}


def _loose_world(n, sd):
    """A world of n dynamic bodies with one fixture each, on the GPU."""
    bd = np.zeros(n, b2g.BODY_DEF)
    bd["type"] = b2g.B2_DYNAMIC_BODY
    bd["awake"] = 1
    bd["gravity_scale"] = 1.0
    bd["position"][:, 0] = np.arange(n)
    fd = np.zeros(n, b2g.FIXTURE_DEF)
    fd["density"], fd["category"], fd["mask"] = 1.0, 1, 0xFFFF
    w = b2g.World()
    w.add(bd, np.arange(n, dtype=np.int32), sd, fd)
    w.body_states()
    return w


def _prepare_pairs(case, seed):
    """Circles, and fat AABBs (0.7 to 1.2 m) spread so that a proxy meets about three others. The seed
    deals the boxes out to the proxies, so every seed has as many pairs."""
    n = case["n"]
    rng = np.random.default_rng(8)
    sd = np.zeros(n, b2g.SHAPE_DEF)
    sd["radius"] = 0.4
    w = _loose_world(n, sd)
    side = np.sqrt(n) * 0.75
    c = rng.uniform(-side, side, (n, 2)) * np.array([1.0, 0.8])
    h = rng.uniform(0.35, 0.6, (n, 2))
    fat = np.concatenate([c - h, c + h], 1).astype(np.float32)
    fat = fat[np.random.default_rng([8, seed]).permutation(n)]
    return {"kind": "pairs", "world": w, "fat": fat}


# ---- what a pass cannot do without ------------------------------------------------------------------
# Bytes and operations of one step per body, per candidate pair and per touching contact: body state
# (position, velocity, sweep start, transform) read and written, mass, shape and both boxes read and
# the boxes written; a pair's two ids and its manifold (60 bytes) read and written; a contact's
# velocity iteration is about 170 operations, its position iteration about 150, its set-up about 200,
# a manifold about 400, two transforms and a body's integration about 150. Pairs and contacts per body
# are those of the scene (a field in free fall, a settled heap).
_PER_BODY = {"box": (1, 1), "pyramid": (2.8, 1.9), "stacks": (1.1, 1.0), "field": (1.2, 0.2), "landing": (2.0, 0.6),
             "heap": (6.0, 2.1), "batch": (3.5, 1.4), "chains": (1.0, 0.0), "grad": (2.5, 0.9)}


def _step_work(bodies, scene, joints=0):
    pairs, touching = (bodies * x for x in _PER_BODY[scene])
    nbytes = bodies * (2 * 64 + 32 + 80 + 48) + pairs * (8 + 2 * 60) + joints * 2 * 100
    flops = bodies * 150 + pairs * 400 + touching * (8 * 170 + 3 * 150 + 200) + joints * (8 * 150 + 3 * 150 + 200)
    return nbytes, flops


def _bodies(case):
    scene = case.get("scene", "grad")
    if scene == "pyramid":
        return case["n"] * (case["n"] + 1) // 2
    if scene == "batch":
        return int(case["n"] * 243)  # the mean of sizes spread evenly over their logarithm, 16 to 1024
    if scene == "chains":
        return case["n"] * 16
    if scene == "grad":
        return case["n"] * case["bodies"]
    return case["n"]


def work(case):
    kind, n = case["kind"], case["n"]
    if kind == "collide":
        return {"bytes": n * (8 + 32 + 72) + (n // 3) * 100, "flops": 400 * n}
    if kind == "pairs":
        return {"bytes": n * 16 + 3 * n * 8, "flops": 60 * n}
    bodies = _bodies(case)
    scene = case.get("scene", "grad")
    b, f = _step_work(bodies, scene, bodies if scene == "chains" else 0)
    steps = case.get("steps", 1)
    if kind == "grad":
        # the steps forward, and each step's reverse: about three times its operations and twice its bytes
        return {"bytes": 3 * b * steps + 4 * 24 * bodies, "flops": 4 * f * steps}
    moved = {"frame": 64, "pile": 64, "rollout": 64 + 64 + 16}[kind]
    return {"bytes": b * steps + moved * bodies, "flops": f * steps}


def tolerance(case):
    kind = case["kind"]
    if kind == "pairs":
        return "exact"
    if kind == "collide":
        # one manifold from its inputs, a few float32 roundings at coordinates of up to 50 m: 3.5e-6 from
        # the value in 64 bits over 20,000 pairs, with the same features in all of them
        return {"rel": 2e-5, "max": 0.99, "differ": 1e-4}
    # Steps that follow one another enlarge a rounding: these are four times (where that is over 0.03, that)
    # what the outputs moved by when every start velocity was moved by one or two units in its last place.
    # The largest is the relative error of the velocities of bodies at rest or being hit; single bodies
    # move by their whole value.
    if kind == "grad":
        return {"rel": 0.02, "max": 0.99}
    scene = case["scene"]
    if scene in ("box", "pyramid"):
        return {"rel": 2e-5, "max": 1e-3}
    if scene == "stacks":
        return {"rel": 1e-4, "max": 5e-3}
    return {"rel": 5e-3 if scene == "field" else 0.03, "max": 0.99}


# ---- 64 bits -----------------------------------------------------------------------------------------
def exact(case, seed):
    """The manifolds of the collide case in 64 bits. A world's step has no such value: the order in
    which its contacts are solved is the implementation's own and Gauss-Seidel's iterates depend on
    it, and whether two shapes touch at all is decided anew in every step."""
    if case["kind"] != "collide":
        return None
    (kind, radius, _, nv, v), pairs, xa, xb = _collide_inputs(case, seed)
    n = len(pairs)
    out = {"type": None, "count": None, "id": None, "normal": np.zeros((n, 2)), "point": np.zeros((n, 2)),
           "points": np.zeros((n, 2, 2))}
    xa, xb = xa.astype(np.float64), xb.astype(np.float64)
    a, b = pairs[:, 0], pairs[:, 1]
    r = radius.astype(np.float64)
    v = v.astype(np.float64)
    for f, rows in ((_circles, (kind[a] == 0) & (kind[b] == 0)), (_polygon_circle, (kind[a] != 0) & (kind[b] == 0)),
                    (_polygons, (kind[a] != 0) & (kind[b] != 0))):
        i = np.nonzero(rows)[0]
        if len(i):
            hit, normal, point, pts = f(v[a[i]], nv[a[i]], v[b[i]], nv[b[i]], r[a[i]], r[b[i]], xa[i], xb[i])
            out["normal"][i] = np.where(hit[:, None], normal, 0.0)
            out["point"][i] = np.where(hit[:, None], point, 0.0)
            out["points"][i] = np.where(hit[:, None, None], pts, 0.0)
    return out


def _rot(x, p):
    s, c = x[..., 2], x[..., 3]
    while s.ndim < p.ndim - 1:
        s, c = s[..., None], c[..., None]
    return np.stack([c * p[..., 0] - s * p[..., 1], s * p[..., 0] + c * p[..., 1]], -1)


def _rot_t(x, p):
    return _rot(np.concatenate([x[:, :2], -x[:, 2:3], x[:, 3:4]], 1), p)


def _to_world(x, p):
    t = x[:, :2]
    return _rot(x, p) + (t if p.ndim == 2 else t[:, None, :])


def _to_local(x, p):
    t = x[:, :2]
    return _rot_t(x, p - (t if p.ndim == 2 else t[:, None, :]))


def _edges(v, nv):
    """Edge vectors' unit normals and each vertex's successor, for rows filled up with the last vertex."""
    k = np.arange(8)[None, :]
    last = k >= nv[:, None] - 1
    nxt = np.where(last[..., None], v[:, :1], np.roll(v, -1, 1))
    e = nxt - v
    e = e / np.maximum(np.hypot(e[..., 0], e[..., 1]), 1e-300)[..., None]
    return np.stack([e[..., 1], -e[..., 0]], -1), nxt, k < nv[:, None]


def _circles(va, na, vb, nb, ra, rb, xa, xb):
    n = len(xa)
    d = xb[:, :2] - xa[:, :2]
    hit = (d * d).sum(1) <= (ra + rb) ** 2
    z = np.zeros((n, 2))
    return hit, z, z, np.zeros((n, 2, 2))


def _polygon_circle(va, na, vb, nb, ra, rb, xa, xb):
    n = len(xa)
    c = _to_local(xa, xb[:, :2])
    normals, nxt, real = _edges(va, na)
    sep = np.where(real, (normals * (c[:, None] - va)).sum(-1), -np.inf)
    i = np.arange(n)
    best = sep.argmax(1)
    s = sep[i, best]
    radius = POLYGON_RADIUS + rb
    v1, v2, nm = va[i, best], nxt[i, best], normals[i, best]
    u1 = ((c - v1) * (v2 - v1)).sum(1)
    u2 = ((c - v2) * (v1 - v2)).sum(1)
    near1, near2 = c - v1, c - v2
    l1, l2 = np.hypot(near1[:, 0], near1[:, 1]), np.hypot(near2[:, 0], near2[:, 1])
    inside = s < np.finfo(np.float32).eps
    mid = inside | ((u1 > 0.0) & (u2 > 0.0))
    at1 = ~inside & (u1 <= 0.0)
    at2 = ~inside & (u1 > 0.0) & (u2 <= 0.0)
    dist = np.where(at1, l1, np.where(at2, l2, s))
    hit = (s <= radius) & (dist <= radius)
    normal = np.where(at1[:, None], near1 / np.maximum(l1, 1e-300)[:, None],
                      np.where(at2[:, None], near2 / np.maximum(l2, 1e-300)[:, None], nm))
    point = np.where(at1[:, None], v1, np.where(at2[:, None], v2, 0.5 * (v1 + v2)))
    assert np.all(mid | at1 | at2)
    return hit, normal, point, np.zeros((n, 2, 2))


def _best_axis(v1, n1, x1, v2, n2, x2):
    """The edge of polygon 1 with the largest separation from polygon 2, and that separation."""
    normals, _, real = _edges(v1, n1)
    w2 = _to_local(x1, _to_world(x2, v2))
    s = ((w2[:, None, :, :] - v1[:, :, None, :]) * normals[:, :, None, :]).sum(-1).min(2)
    s = np.where(real, s, -np.inf)
    best = s.argmax(1)
    return best, s[np.arange(len(s)), best]


def _clip(p, q, normal, offset):
    """The segment p q cut to normal . x <= offset; whether two points are left."""
    d0, d1 = (normal * p).sum(1) - offset, (normal * q).sum(1) - offset
    cut = d0 * d1 < 0.0
    m = p + (np.where(cut, d0 / np.where(cut, d0 - d1, 1.0), 0.0))[:, None] * (q - p)
    first = np.where((d0 <= 0.0)[:, None], p, q)
    second = np.where(cut[:, None], m, q)
    return first, second, (d0 <= 0.0) & (d1 <= 0.0) | cut


def _polygons(va, na, vb, nb, ra, rb, xa, xb):
    n = len(xa)
    total = 2.0 * POLYGON_RADIUS
    ea, sa = _best_axis(va, na, xa, vb, nb, xb)
    eb, sb = _best_axis(vb, nb, xb, va, na, xa)
    flip = sb > sa + 0.1 * 0.005
    hit = (sa <= total) & (sb <= total)
    f2, f3 = flip[:, None], flip[:, None, None]
    v1, n1, x1 = np.where(f3, vb, va), np.where(flip, nb, na), np.where(f2, xb, xa)
    v2, n2, x2 = np.where(f3, va, vb), np.where(flip, na, nb), np.where(f2, xa, xb)
    edge = np.where(flip, eb, ea)
    i = np.arange(n)
    normals1, next1, _ = _edges(v1, n1)
    normals2, next2, real2 = _edges(v2, n2)
    against = (normals2 * _rot_t(x2, _rot(x1, normals1[i, edge]))[:, None]).sum(-1)
    j = np.where(real2, against, np.inf).argmin(1)
    p, q = _to_world(x2, v2[i, j]), _to_world(x2, next2[i, j])
    a, b = v1[i, edge], next1[i, edge]
    t = (b - a) / np.hypot(*(b - a).T)[:, None]
    normal = np.stack([t[:, 1], -t[:, 0]], 1)
    tw = _rot(x1, t)
    nw = np.stack([tw[:, 1], -tw[:, 0]], 1)
    aw, bw = _to_world(x1, a), _to_world(x1, b)
    p, q, two = _clip(p, q, -tw, -(tw * aw).sum(1) + total)
    hit &= two
    p, q, two = _clip(p, q, tw, (tw * bw).sum(1) + total)
    hit &= two
    front = (nw * aw).sum(1)
    k0, k1 = (nw * p).sum(1) - front <= total, (nw * q).sum(1) - front <= total
    hit &= k0 | k1
    lp, lq = _to_local(x2, p), _to_local(x2, q)
    pts = np.zeros((n, 2, 2))
    pts[:, 0] = np.where(k0[:, None], lp, lq)
    pts[:, 1] = np.where((k0 & k1)[:, None], lq, 0.0)
    return hit, normal, 0.5 * (a + b), pts
