"""Residual stops with islands of every kind in one launch: large islands that check every
residual_every sweeps, islands of 257 to 4096 manifolds that check after each of theirs, in one round
of the register sweep or several, and smaller ones.  Bar: the same sweeps, residual and bits as with
the large islands swept in a launch per colour, where every other island is solved by a workgroup or a
wave of its own."""
import numpy as np
import pytest

from test_gpu_island_classes import _scene

pytestmark = pytest.mark.gpu

DT = 1.0 / 120.0


def _run(axm, b, mode, tol, every, most):
    d = axm.default_desc(num_planes=0, island_solve=1)
    d.solver_mode = mode
    d.residual_tol, d.residual_every, d.max_iterations = tol, every, most
    for k in range(3):
        d.gravity[k], d.origin[k] = 0.0, -4.0
    w = axm.World(d)
    w.set_bodies(b)
    w.totals(reset=True)
    seen = []
    for _ in range(3):
        st = w.step(DT, most, axm.STEP_RESIDUAL)
        seen.append((st.iterations, st.residual, st.manifolds))
    g, t = w.get_bodies(), w.totals()
    out = [g.pos.copy(), g.quat.copy(), g.lin_vel.copy(), g.ang_vel.copy()] + list(w.impulses())
    w.close()
    return seen, out, (t.sweeps, t.steps_at_tol, t.contact_sweeps, t.local_contact_sweeps)


@pytest.mark.parametrize("tol,every,most", [(1e-3, 1, 60), (1e-3, 3, 60), (1e-2, 4, 30), (1e-9, 4, 10), (10.0, 2, 5)])
@pytest.mark.parametrize("sizes", [
    [5000, 300, 1200, 40, 5],
    [4500, 4200, 257, 4000, 100, 9, 3],
    [5000] + [3900] * 17,  # several rounds of the register sweep
    [3900] * 18,           # and no large island
])
def test_stops_equal_colour_launches(axm, gpu, sizes, tol, every, most):
    # spheres where the sizes have to be exact: boxes also touch across their corners
    b = _scene(axm, sizes, 29, len(sizes) < 10)
    one = _run(axm, b, 0, tol, every, most)
    ref = _run(axm, b, 1, tol, every, most)
    assert one[0] == ref[0]
    assert one[2] == ref[2]
    assert (one[2][3] < one[2][2]) == (max(sizes) > 4096)
    for x, y in zip(one[1], ref[1]):
        assert np.array_equal(x, y)
