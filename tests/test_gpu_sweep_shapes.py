"""Launch shapes of the staged sweep, on the only steps that run it (large islands of more than 65536
manifolds: a settled batch swept jointly): every shape and poll policy gives the default's bits, with
and without residual checks, and the autotuner picks one of its candidates.  On a step that it does
not run the autotuner keeps the shape the world has."""
import numpy as np
import pytest

from helpers import seed

pytestmark = pytest.mark.gpu

DT = 1.0 / 120.0
SHAPES = [(0, 0, 0x12), (512, 64, 0x12), (1024, 32, 0x12), (100, 48, 0x12), (256, 16, 0x00), (0, 0, 0x76)]


@pytest.fixture(scope="module")
def batch(axm, gpu):
    b, d = axm.scene(3, seed(3), 0, 256)
    w = axm.World(d)
    w.set_bodies(b)
    w.run(DT, 10, 240, graph=True)
    g = w.get_bodies()
    b.pos, b.quat, b.lin_vel, b.ang_vel = g.pos, g.quat, g.lin_vel, g.ang_vel
    w.close()
    return b


def _desc(axm, tol):
    d = axm.scene(3, seed(3), 0, 256)[1]
    d.island_solve = 0
    d.residual_tol, d.residual_every, d.max_iterations = tol, 2, 30
    return d


@pytest.mark.parametrize("tol", [0.0, 0.3])
def test_shapes_give_the_same_bits(axm, gpu, batch, tol):
    out = []
    for groups, kib, policy in SHAPES:
        print("shape", groups, kib, hex(policy), flush=True)
        w = axm.World(_desc(axm, tol))
        w.set_bodies(batch)
        w.set_sweep_config(groups, kib, policy)
        for _ in range(2):
            st = w.step(DT, 6, axm.STEP_RESIDUAL)
        assert st.manifolds > 65536
        g = w.get_bodies()
        out.append([g.pos.copy(), g.quat.copy(), g.lin_vel.copy(), g.ang_vel.copy(), st.iterations, st.residual]
                   + list(w.impulses()))
        w.close()
    for o in out[1:]:
        for x, y in zip(out[0], o):
            assert np.array_equal(x, y)


def test_autotune_picks_where_the_sweep_runs(axm, gpu, batch):
    w = axm.World(_desc(axm, 0.0))
    w.set_bodies(batch)
    w.step(DT, 6)
    w.set_sweep_config(100, 48, 0x22)
    groups, kib, policy, ms = w.autotune(DT, 6, 2)
    assert (groups, kib) in ((256, 160), (512, 80), (1024, 32)) and policy == 0x12 and ms > 0
    w.close()


@pytest.mark.parametrize("config,n,worlds", [(3, 0, 64), (1, 6000, 0)])
def test_autotune_keeps_the_shape_elsewhere(axm, gpu, config, n, worlds):
    b, d = axm.scene(config, seed(config), n, worlds)
    w = axm.World(d)
    w.set_bodies(b)
    w.run(DT, 10, 60, graph=True)
    for shape in ((100, 48, 0x22), (512, 64, 0x12)):
        w.set_sweep_config(*shape)
        got = w.autotune(DT, 10, 2)
        assert got[:3] == shape and got[3] > 0
    w.close()
