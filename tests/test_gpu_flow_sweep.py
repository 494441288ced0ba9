"""The large islands' sweep (island_solve off: every manifold takes it) against one launch per colour
and sweep, through the C ABI: up to 256 x the CUs' count of slots it runs with one slot per pair of
lanes, above that in the staged sweep.

Bar: both see every body's visits in the same order and stop at the same check of the same residual,
so sweep counts, residuals, positions, velocities and impulses are equal."""
import numpy as np
import pytest

from helpers import seed
from test_gpu_island_classes import _scene

pytestmark = pytest.mark.gpu

DT = 1.0 / 120.0


def _run(axm, b, d, mode, tol, every, sweeps, steps):
    d.island_solve, d.solver_mode = 0, mode
    d.residual_tol, d.residual_every, d.max_iterations = tol, every, sweeps
    w = axm.World(d)
    w.set_bodies(b)
    its = []
    for _ in range(steps):
        st = w.step(DT, sweeps, axm.STEP_RESIDUAL)
        its.append((st.iterations, st.residual))
    g = w.get_bodies()
    out = [g.pos.copy(), g.quat.copy(), g.lin_vel.copy(), g.ang_vel.copy()] + list(w.impulses())
    m = st.manifolds
    w.close()
    return its, out, m


def _equal(axm, b, d, tol, every, sweeps, steps):
    a = _run(axm, b, axm.WorldDesc.from_buffer_copy(d), 0, tol, every, sweeps, steps)
    c = _run(axm, b, axm.WorldDesc.from_buffer_copy(d), 1, tol, every, sweeps, steps)
    assert a[0] == c[0]
    for x, y in zip(a[1], c[1]):
        assert np.array_equal(x, y)
    return a


@pytest.mark.parametrize("tol,every,sweeps", [(0.0, 1, 1), (0.0, 1, 8), (1e-3, 1, 60), (1e-3, 3, 60), (1e-2, 2, 7),
                                              (1e-9, 4, 10), (10.0, 1, 5)])
@pytest.mark.parametrize("sizes", [[1], [31], [32], [33], [63, 65], [7, 300, 1200]])
def test_register_sweep_equals_colour_launches(axm, gpu, sizes, tol, every, sweeps):
    b = _scene(axm, sizes, 5, True)
    d = axm.default_desc(num_planes=0)
    for k in range(3):
        d.gravity[k], d.origin[k] = 0.0, -4.0
    its, _, m = _equal(axm, b, d, tol, every, sweeps, 3)
    if not any(s > 300 for s in sizes) and tol == 10.0:
        assert all(i == 1 for i, _ in its)  # the first check stops: the visits run ahead are taken back


@pytest.mark.parametrize("tol,every,sweeps", [(0.0, 1, 6), (0.3, 2, 30)])
def test_staged_sweep_equals_colour_launches(axm, gpu, tol, every, sweeps):
    """More slots than pairs of lanes: a settling batch of worlds swept jointly."""
    b, d = axm.scene(3, seed(3), 0, 256)
    w = axm.World(d)
    w.set_bodies(b)
    w.run(DT, 10, 240, graph=True)
    g = w.get_bodies()
    b.pos, b.quat, b.lin_vel, b.ang_vel = g.pos, g.quat, g.lin_vel, g.ang_vel
    w.close()
    _, _, m = _equal(axm, b, d, tol, every, sweeps, 2)
    assert m > 65536
