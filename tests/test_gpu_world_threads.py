"""Worlds of one device stepped from several threads at once.  A step's colouring, sorts and sweeps
wait for workgroups of their own grids, and a sweep's workgroup takes a whole CU, so two worlds'
grids on the chip together could hold what the other waits for; the worlds' steps take turns.
Bar: every world ends bit for bit where it ends alone, by eager steps, replayed steps and with the
broadphase and narrowphase called in between, and no step times out."""
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
