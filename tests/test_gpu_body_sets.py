"""Body sets through axm_world_set_bodies / axm_world_get_bodies: poses and velocities come back bit
for bit at sizes around a workgroup and beyond the pinned staging (several pieces), also when only
some fields are asked for; of several faulty bodies the first one's code is returned, in the order
the faults are looked for; a set of the same shape put into a world with captured steps runs like a
new world; world ids may have gaps and are refused above the limit."""
import ctypes as C

import numpy as np
import pytest

from helpers import seed

pytestmark = pytest.mark.gpu

DT = 1.0 / 120.0


def _bodies(axm, n, s):
    rng = np.random.default_rng(s)
    b = axm.Bodies(n)
    b.pos[:] = rng.uniform(-50, 50, (n, 3))
    q = rng.normal(size=(n, 4))
    b.quat[:] = q / np.linalg.norm(q, axis=1, keepdims=True)
    b.lin_vel[:] = rng.normal(size=(n, 3))
    b.ang_vel[:] = rng.normal(size=(n, 3))
    b.inv_mass[:] = rng.uniform(0.5, 2, n)
    b.inv_inertia[:] = rng.uniform(0.5, 2, (n, 3))
    b.shape_type[:] = rng.integers(0, 3, n)
    b.shape_params[:] = rng.uniform(0.1, 0.4, (n, 3))
    return b


@pytest.mark.parametrize("n", [1, 63, 255, 257, 4099, 74899, 250001])
def test_round_trip(axm, gpu, n):
    b = _bodies(axm, n, n)
    w = axm.World(axm.default_desc())
    w.set_bodies(b)
    for _ in range(2):
        g = w.get_bodies()
        for f in ("pos", "quat", "lin_vel", "ang_vel"):
            assert np.array_equal(getattr(g, f), getattr(b, f)), f
    part = axm.Bodies(n)
    s = axm.BodySoA()
    s.quat = part.quat.ctypes.data_as(C.POINTER(C.c_float))
    s.ang_vel = part.ang_vel.ctypes.data_as(C.POINTER(C.c_float))
    assert axm.lib().axm_world_get_bodies(w._h, C.byref(s)) == 0
    assert np.array_equal(part.quat, b.quat) and np.array_equal(part.ang_vel, b.ang_vel)
    assert not part.pos.any() and not part.lin_vel.any()
    w.close()


def _spoil(b, kind, i):
    if kind == "body":
        b.lin_vel[i, 2] = np.inf
    elif kind == "norm":
        b.quat[i] = 0.1
    elif kind == "shape":
        b.shape_type[i] = 3
    elif kind == "size":
        b.shape_params[i, 0] = 0.0
    elif kind == "world":
        b.world[i - 1] = 7
    elif kind == "material":
        b.material[i, 0] = -1.0
    else:
        b.flags[i] = 1


@pytest.mark.parametrize("n", [300, 100003])
@pytest.mark.parametrize("first,second,code", [
    ("body", "shape", 400), ("shape", "body", None), ("size", "norm", None), ("norm", "size", 400),
    ("world", "body", -1), ("material", "shape", 400), ("kinematic", "shape", 400)])
def test_first_faulty_body_decides(axm, gpu, n, first, second, code):
    b = _bodies(axm, n, 5)
    b.material = np.tile(np.array([0.4, 0.1, 0.01, 0.02], np.float32), (n, 1))
    b.flags = np.zeros(n, np.uint32)
    w = axm.World(axm.default_desc())
    w.set_bodies(b)

    def refused(kinds):
        c = b.copy()
        for kind, i in kinds:
            _spoil(c, kind, i)
        with pytest.raises(axm.AxmError) as e:
            w.set_bodies(c)
        return e.value.code

    alone = refused([(first, n // 3)])
    if code == 400:
        assert alone == 400
    if code == -1:
        assert alone == axm.INVALID_PARAMETER
    assert alone != refused([(second, n // 3)])
    assert refused([(first, n // 3), (second, n - 1)]) == alone
    assert refused([(first, n // 3), (second, n // 3 + 1)]) == alone
    assert refused([(first, n - 1), (second, 0)]) == refused([(second, 0)])
    assert np.array_equal(w.get_bodies().pos, b.pos)
    w.close()


def test_same_sized_set_keeps_captured_steps(axm, gpu):
    b, d = axm.scene(0, seed(0), 400)
    c = b.copy()
    c.lin_vel = c.lin_vel + np.float32(0.25) * (c.inv_mass > 0)[:, None].astype(np.float32)
    w = axm.World(d)
    w.set_bodies(b)
    w.run(DT, 10, 30, graph=True)
    w.set_bodies(c)
    w.run(DT, 10, 30, graph=True)
    got = w.get_bodies()
    w.close()
    w = axm.World(d)
    w.set_bodies(c)
    w.run(DT, 10, 30, graph=False)
    ref = w.get_bodies()
    w.close()
    for f in ("pos", "quat", "lin_vel", "ang_vel"):
        assert np.array_equal(getattr(got, f), getattr(ref, f)), f


def test_world_ids_with_gaps(axm, gpu):
    b = _bodies(axm, 64, 9)
    b.pos[:] = (b.pos * np.float32(0.02)).astype(np.float32)  # within 2 m: pairs within each world
    b.inv_inertia[:] = 1.0
    out = []
    for ids in ((0, 1), (3, 70000)):
        c = b.copy()
        c.world[:32], c.world[32:] = ids
        w = axm.World(axm.default_desc())
        w.set_bodies(c)
        w.run(DT, 10, 10, graph=False)
        out.append(w.get_bodies())
        w.close()
    for f in ("pos", "quat", "lin_vel", "ang_vel"):
        assert np.array_equal(getattr(out[0], f), getattr(out[1], f)), f
    for top in (1 << 22, 0xFFFFFFFF):
        c = b.copy()
        c.world[63] = top
        w = axm.World(axm.default_desc())
        with pytest.raises(axm.AxmError) as e:
            w.set_bodies(c)
        assert e.value.code == axm.OUT_OF_RANGE
        w.close()
