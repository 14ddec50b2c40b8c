"""The adjoint's group kernels (a workgroup per bin of islands or per world, a constraint per thread)
against its per-colour launches on the same recorded run.

Whether a recorded step is replayed and reversed by groups follows the forward solve's grouping, which
changes no result: with the island and the per-world solve switched off the same steps are recorded
ungrouped. The frozen replay then agrees bit for bit, and the gradients to the order of their atomic sums:
12 steps of float32 sums of up to 30 terms, 12 * 30 * 2^-24 = 2e-5 of the largest entry where a rounding
grows as the gradient does, and ten times that where it grows faster than the entries around it: 2e-4
(the same backward run twice differs by up to 3e-6). Group sizes on both sides of
each workgroup size (64, 128, 256, 512 constraints), beyond the largest, and steps with no contact at all.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = np.float32(1.0 / 60.0)


def _grad(batch, grouped, warm_steps, steps, block=True):
    import b2g
    w = b2g.World()
    w.set_flags(warm_starting=True, allow_sleep=False, continuous=False, block_solve=block)
    if not grouped:
        w.tune(b2g.TUNE_WORLD_SOLVE, 0)
        w.tune(b2g.TUNE_ISLAND_SOLVE, 0)
    w.add_batched(batch.body_defs, batch.body_world, batch.fixture_body, batch.shape_defs, batch.fixture_defs)
    for _ in range(warm_steps):
        w.step(DT, 8, 3)
    w.tape_begin(5)
    for _ in range(steps):
        w.step(DT, 8, 3)
    w.tape_end()
    final = w.body_states()
    touching = w.profile()["touching"]
    replay = w.tape_replay()
    cot = np.random.default_rng(3).normal(size=(len(final), 6)).astype(np.float32)
    g, gf = w.tape_backward(cot)
    again, _ = w.tape_backward(cot)  # the kept working memory carries nothing over
    w.close()
    return final.tobytes(), replay.tobytes(), g, gf, again, touching


def _close(a, b):
    assert np.abs(a - b).max() <= 2e-4 * np.abs(b).max(), np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("worlds,n,warm,block", [(1, 12, 90, True), (3, 40, 90, True), (20, 24, 90, True),
                                                 (17, 60, 90, False), (16, 100, 90, True), (16, 200, 110, True),
                                                 (16, 420, 130, True), (2, 5, 0, True)])
def test_groups_match_per_colour_launches(worlds, n, warm, block):
    from b2g import scenes
    batch = scenes.differentiable_worlds(worlds, n)
    a = _grad(batch, True, warm, 12, block)
    b = _grad(batch, False, warm, 12, block)
    assert a[0] == b[0], "forward runs differ"
    assert a[1] == b[1], "frozen replays differ"
    assert warm == 0 or a[5] > n // 2
    for x in (a, b):
        assert np.isfinite(x[2]).all() and np.isfinite(x[3]).all()
        _close(x[4], x[2])
    _close(a[2], b[2])
    if np.abs(b[3]).max() > 0:
        _close(a[3], b[3])
