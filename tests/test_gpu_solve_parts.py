"""The solver's sweeps in one launch (large islands beside the others) and in launches of their own
(as they run while timed): the same bits, with and without a tolerance, on a pile (one large island
and many small ones), a batch of worlds (islands of every class) and a scene without large islands."""
import numpy as np
import pytest

from helpers import seed

pytestmark = pytest.mark.gpu

DT = 1.0 / 120.0


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("config,n,worlds,settle,tol", [(1, 9000, 0, 80, 0.0), (1, 6000, 0, 200, 1e-4), (3, 0, 48, 240, 1e-4),
                                                         (0, 300, 0, 120, 0.0)])
def test_one_launch_matches_two(axm, gpu, config, n, worlds, settle, tol, graph):
    b, d = axm.scene(config, seed(config), n, worlds)
    if tol > 0.0:
        d.residual_tol = tol
        d.max_iterations = 300
    out = []
    for timed in (False, True):
        w = axm.World(d)
        w.set_bodies(b)
        w.run(DT, 10, settle, graph=True)
        w.totals(reset=True)
        if timed:
            w.profile(True)
        st = w.run(DT, 300 if tol > 0.0 else 10, 6, graph=graph)
        g = w.get_bodies()
        t = w.totals()
        out.append((g.pos, g.quat, g.lin_vel, g.ang_vel, st.residual, t.sweeps, t.steps_at_tol, t.contact_sweeps))
        w.close()
    for x, y in zip(*out):
        assert np.array_equal(x, y)
    assert out[0][5] > 0
