"""Solves of more than two seconds: a bounded wait of the sweeps gives up after two seconds without
progress, not after two seconds of work, so islands of 257 to 4096 manifolds may take as many sweeps
as they are given, alone or in several rounds of the register sweep (whose later pieces first wait
for the earlier ones).  Bar: the same bits as with the large islands swept in a launch per colour,
where each of these islands is solved by a workgroup of its own without a wait."""
import time

import numpy as np
import pytest

from test_gpu_island_classes import _scene

pytestmark = pytest.mark.gpu

DT = 1.0 / 120.0


def _run(axm, b, mode, sweeps):
    d = axm.default_desc(num_planes=0, island_solve=1)
    d.solver_mode = mode
    for k in range(3):
        d.gravity[k], d.origin[k] = 0.0, -4.0
    w = axm.World(d)
    w.set_bodies(b)
    w.step(DT, 1)
    t = time.perf_counter()
    st = w.step(DT, sweeps)
    t = time.perf_counter() - t
    g = w.get_bodies()
    out = [g.pos.copy(), g.lin_vel.copy(), g.ang_vel.copy()] + list(w.impulses())
    w.close()
    print("mode %d: %d sweeps %.2f s" % (mode, sweeps, t), flush=True)
    return out, st, t


@pytest.mark.parametrize("sizes,sweeps", [([300], 450000), ([3900] * 18, 230000)])
def test_long_solve_ends(axm, gpu, sizes, sweeps):
    b = _scene(axm, sizes, 23, False)
    one, st, took = _run(axm, b, 0, sweeps)
    assert st.iterations == sweeps
    ref, _, _ = _run(axm, b, 1, sweeps)
    for x, y in zip(one, ref):
        assert np.array_equal(x, y)
    assert took > 2.2, "too short to tell"
