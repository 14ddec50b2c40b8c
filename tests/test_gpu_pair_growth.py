"""A contact set that outgrows its arrays (more than eight pairs per proxy), with and without proxies of more
pairs than a walk's slots hold: the pairs equal those of the fat boxes on the host at every step, and a
contact that persists keeps its predecessor (its impulses warm-start the next step: the states repeat from run
to run and differ from those without warm starting).
"""
import numpy as np
import pytest

import b2g

pytestmark = pytest.mark.gpu

DT = np.float32(1.0 / 60.0)


def _world(clusters, per, sensors):
    """clusters of `per` small boxes in one place each, over a ground box."""
    n = clusters * per
    bd = np.zeros(n + 1, b2g.BODY_DEF)
    bd["gravity_scale"], bd["awake"], bd["allow_sleep"] = 1.0, 1, 1
    bd[1:]["type"] = 2
    i = np.arange(n) // per
    side = int(np.ceil(np.sqrt(clusters)))
    jitter = np.random.default_rng(3).uniform(-0.01, 0.01, (n, 2))
    bd["position"][1:] = np.stack([(i % side) * 3.0, 2.0 + (i // side) * 3.0], 1) + jitter
    bd["linear_velocity"][1:] = 100.0 * jitter  # (they push each other: impulses)
    sd = np.zeros(n + 1, b2g.SHAPE_DEF)
    sd["type"] = b2g.SHAPE_BOX
    sd["params"][:, :2] = 0.25
    sd[0]["params"][:2] = (4.0 * side + 5.0, 0.5)
    fd = np.zeros(n + 1, b2g.FIXTURE_DEF)
    fd["friction"], fd["density"], fd["restitution_threshold"] = 0.5, 1.0, 1.0
    fd["category"], fd["mask"] = 1, 0xFFFF
    fd["is_sensor"][1:] = sensors
    w = b2g.World()
    w.add(bd, np.arange(n + 1, dtype=np.int32), sd, fd)
    return w, bd


def _host_pairs(w):
    fat = w.fat_aabbs()
    got = w.contacts()[0]
    order = np.argsort(fat[:, 0], kind="stable")
    out = []
    for a, i in enumerate(order):
        j = order[a + 1:a + 1 + np.searchsorted(fat[order[a + 1:], 0], fat[i, 2], side="right")]
        hit = j[(fat[j, 1] <= fat[i, 3]) & (fat[i, 1] <= fat[j, 3])]
        out.append(np.stack([np.minimum(i, hit), np.maximum(i, hit)], 1))
    want = np.concatenate(out)
    got = np.sort(np.asarray(got).reshape(-1, 2), 1)
    return want[np.lexsort((want[:, 1], want[:, 0]))], got[np.lexsort((got[:, 1], got[:, 0]))]


@pytest.mark.parametrize("clusters,per", [(100, 30), (40, 70), (30, 90)])
def test_growing_contact_set(clusters, per):
    w, bd = _world(clusters, per, 1)
    w.set_flags(warm_starting=True, allow_sleep=False, continuous=False, block_solve=True)
    for step in range(3):
        w.step(DT, 8, 3)
        want, got = _host_pairs(w)
        assert len(want) > 8 * len(bd)
        assert np.array_equal(want, got), "step %d" % step
    w.close()


def test_persisting_contacts_keep_their_impulses():
    out = []
    for warm in (True, True, False):
        w, bd = _world(90, 24, 0)
        w.set_flags(warm_starting=warm, allow_sleep=False, continuous=False, block_solve=True)
        for _ in range(4):
            w.step(DT, 8, 3)
        assert w.contact_count > 8 * len(bd)
        out.append(w.body_states().tobytes())
        w.close()
    assert out[0] == out[1]
    assert out[0] != out[2]
