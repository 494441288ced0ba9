"""Worlds of one device stepped from several threads at once.  A step's colouring, sorts and sweeps
wait for workgroups of their own grids, and a sweep's workgroup takes a whole CU, so two worlds'
grids on the chip together could hold what the other waits for; the worlds' steps take turns.
Bar: every world ends bit for bit where it ends alone, by eager steps, replayed steps and with the
broadphase and narrowphase called in between, and no step times out.  Worlds may also be created,
captured, read and closed in threads: a capture is not broken by another thread's copies."""
import threading

import numpy as np
import pytest

from helpers import seed

pytestmark = pytest.mark.gpu

DT = 1.0 / 120.0
# a large island each (register sweep), islands of every class, sorts in several workgroups
SCENES = [(1, 6000, 0, 20, 1e-4), (1, 9000, 0, 20, 0.0), (3, 0, 64, 10, 1e-4), (0, 20000, 0, 10, 0.0)]


def _world(axm, k):
    config, n, worlds, sweeps, tol = SCENES[k]
    b, d = axm.scene(config, seed(config), n, worlds)
    if tol > 0.0:
        d.residual_tol, d.max_iterations = tol, 60
    w = axm.World(d)
    w.set_bodies(b)
    w.run(DT, sweeps, 100, graph=True)
    return w


def _passes(axm, w, k):
    sweeps = SCENES[k][3]
    for _ in range(6):
        w.step(DT, sweeps)
    for _ in range(3):
        w.run(DT, sweeps, 12, graph=True)
        w.broadphase()
        w.collide()
    w.run(DT, sweeps, 6, graph=False)
    g = w.get_bodies()
    return [g.pos.copy(), g.quat.copy(), g.lin_vel.copy(), g.ang_vel.copy()]


def _life(axm, config, n, worlds, sweeps):
    """A world created, captured, read and closed, a few times over; pairs and a network beside it."""
    b, d = axm.scene(config, seed(config), n, worlds)
    rng = np.random.default_rng(n)
    X = rng.normal(size=(500, axm.MLP_INPUTS)).astype(np.float32)
    one = np.ones(300, np.uint32)
    half = np.full((300, 3), 0.5, np.float32)
    x = rng.uniform(-0.5, 0.5, (2, 300, 3)).astype(np.float32)
    q = np.tile(np.array([0, 0, 0, 1], np.float32), (300, 1))
    out = []
    for _ in range(3):
        w = axm.World(d)
        w.set_bodies(b)
        w.run(DT, sweeps, 20, graph=True)
        w.step(DT, sweeps, axm.STEP_RESIDUAL)
        m = w.manifolds()
        g = w.get_bodies()
        out = [g.pos.copy(), g.lin_vel.copy(), m["pos"].copy(), w.impulses()[1]]
        w.close()
        p = axm.collide_pairs(one, half, x[0], q, one, half, x[1], q, noalloc=True)
        assert p["status"] == 0
        net = axm.Mlp(0, seed=3)
        out += [p["pos"], net.forward(X)]
    return out


def test_whole_lives_in_threads(axm, gpu):
    jobs = [(0, 300, 0, 10), (1, 6000, 0, 20), (3, 0, 32, 10), (2, 70000, 0, 10), (1, 3000, 0, 20), (0, 9000, 0, 10)]
    ref = [_life(axm, *j) for j in jobs]
    got, err = [None] * len(jobs), []

    def work(k):
        try:
            got[k] = _life(axm, *jobs[k])
        except Exception as e:  # noqa: BLE001 (reported below)
            err.append((k, e))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(len(jobs))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not err, err
    for r, g in zip(ref, got):
        for x, y in zip(r, g):
            assert np.array_equal(x, y)


def test_worlds_in_threads_end_as_alone(axm, gpu):
    ref = []
    for k in range(len(SCENES)):
        w = _world(axm, k)
        ref.append(_passes(axm, w, k))
        w.close()
    worlds = [_world(axm, k) for k in range(len(SCENES))]
    got, err = [None] * len(SCENES), []
    start = threading.Barrier(len(SCENES))

    def work(k):
        start.wait()
        try:
            got[k] = _passes(axm, worlds[k], k)
        except Exception as e:  # noqa: BLE001 (reported below)
            err.append((k, e))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(len(SCENES))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for w in worlds:
        w.close()
    assert not err, err
    for r, g in zip(ref, got):
        for x, y in zip(r, g):
            assert np.array_equal(x, y)
