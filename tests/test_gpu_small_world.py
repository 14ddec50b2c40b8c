"""Small worlds (k_small_solve, k_small_build, k_small_pairs: a step's solve and its pair search in one workgroup
each) against the launches they replace, which a timed kernel keeps: the constraints, colours, operations
and orders are the same, so states, boxes, contacts with their manifolds, colours and the solver's state agree
bit for bit, step by step.

Worlds at the edges of the kernels' limits: one body, a wave and a workgroup of bodies and one more, the most
bodies and one more, no pair at all; a heap that forms one large island; sleeping on; continuous collision with its
rebuilds; a world whose pairs outgrow their arrays (fixtures in one place); one with more touching
contacts than the workgroup takes and one with a body of more than 127 contacts, which the kernels hand back to
the launches untouched.
"""
import numpy as np
import pytest

import b2g
from b2g import scenes

from test_gpu_hub import hub_scene

pytestmark = pytest.mark.gpu

DT = np.float32(1.0 / 60.0)


def _pile(n, cols, seed=0, gap=0.52, spin=0.0):
    """n boxes and circles in columns of touching bodies on a ground box."""
    rng = np.random.default_rng(seed)
    bd = np.zeros(n + 1, b2g.BODY_DEF)
    bd["gravity_scale"], bd["awake"], bd["allow_sleep"] = 1.0, 1, 1
    bd[1:]["type"] = 2
    i = np.arange(n)
    bd["position"][1:] = np.stack([(i % cols - 0.5 * cols) * gap, 0.76 + (i // cols) * 0.51], 1)
    bd["angular_velocity"][1:] = rng.uniform(-spin, spin, n)
    bd[3::7]["type"] = 1  # some kinematic ones
    bd["linear_velocity"][3::7] = (0.3, 0.1)
    sd = np.zeros(n + 1, b2g.SHAPE_DEF)
    sd["type"] = b2g.SHAPE_BOX
    sd["params"][:, :2] = 0.25
    sd[0]["params"][:2] = (2.0 * cols + 5.0, 0.5)
    circles = 2 + 3 * np.arange((n - 1) // 3)
    sd["type"][circles] = b2g.SHAPE_CIRCLE
    sd["radius"][circles] = 0.25
    sd["params"][circles] = 0.0
    fd = np.zeros(n + 1, b2g.FIXTURE_DEF)
    fd["friction"], fd["density"], fd["restitution_threshold"] = 0.5, 1.0, 1.0
    fd["category"], fd["mask"] = 1, 0xFFFF
    fd["is_sensor"][5::11] = 1
    return scenes.Scene(bd, np.arange(n + 1, dtype=np.int32), sd, fd, {"name": "pile"})


def _same_place(n):
    """n proxies of a body each in one place: n (n - 1) / 2 pairs, more than their arrays hold at first."""
    sc = _pile(n, 1)
    sc.body_defs["position"][1:] = (0.0, 3.0)
    sc.body_defs["type"][1:] = 2
    sc.fixture_defs["is_sensor"] = 1
    return sc


def _scene(kind):
    if kind.startswith("pile"):
        n = int(kind[4:])
        return _pile(n, max(1, int(round(n ** 0.5)) * 2), seed=n, spin=2.0)
    if kind == "dense":  # more touching contacts than the workgroup takes
        return _pile(1300, 40, gap=0.49)
    if kind == "apart":
        return scenes.large_world(n=300, seed=3, half_extent=400.0)
    if kind == "heap":
        return scenes.heap_world(600, seed=11, half_extent=10.0)
    if kind == "hub":
        return hub_scene()
    return _same_place(int(kind[5:]))


def _run(sc, steps, sleep, continuous, iters, launches):
    w = b2g.World()
    w.set_flags(warm_starting=True, allow_sleep=sleep, continuous=continuous, block_solve=True)
    w.add(sc.body_defs, sc.fixture_body, sc.shape_defs, sc.fixture_defs)
    if launches:
        w.time_kernel("traverse")
    out, touching = [], 0
    for _ in range(steps):
        w.step(DT, *iters)
        p = w.profile()
        touching = max(touching, p["touching"])
        fab, flags, man = w.contacts()
        out.append((p["touching"], w.body_states().tobytes(), w.fat_aabbs().tobytes(), fab.tobytes(), flags.tobytes(),
                    man.tobytes(), np.asarray(w.contact_colours()).tobytes(), str(w.solver_state())))
    w.close()
    return out, touching


@pytest.mark.parametrize("kind,sleep,continuous", [
    ("pile1", False, False), ("pile63", True, True), ("pile64", False, False), ("pile65", False, True),
    ("pile511", True, False), ("pile1023", False, False), ("pile1024", True, False), ("pile2047", False, False),
    ("pile2048", False, False), ("apart", True, True), ("heap", True, True), ("heap", False, False),
    ("place80", False, False), ("dense", False, False), ("hub", False, True), ("hub", True, False)])
def test_small_world_kernels_match_the_launches(kind, sleep, continuous):
    sc = _scene(kind)
    steps = 40 if len(sc.body_defs) > 1000 else 90
    # (the launches solve a hub's last colour serially, in an order that varies from run to run: no iterations)
    iters = {"pile65": (1, 0), "hub": (0, 0)}.get(kind, (8, 3))
    ref, touching = _run(sc, steps, sleep, continuous, iters, True)
    got, _ = _run(sc, steps, sleep, continuous, iters, False)
    print("%s: up to %d touching contacts" % (kind, touching), flush=True)
    assert touching >= (0 if kind in ("apart", "place80") else 1)
    if kind == "dense":
        assert touching > 2048
    for step, (x, y) in enumerate(zip(ref, got)):
        for name, u, v in zip(("touching", "states", "boxes", "contacts", "flags", "manifolds", "colours", "solver"),
                              x, y):
            assert u == v, "step %d: %s differ" % (step, name)
