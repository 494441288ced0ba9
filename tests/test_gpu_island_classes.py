"""The small islands' kernel at the edges of its size classes, through the C ABI: islands of at
most 8 manifolds share waves by window, those up to 16, 32 and 64 take blocks of a wave's lanes,
up to 256 a workgroup with two lanes per manifold, up to 4096 the large islands' register sweep
or, when they are many, a workgroup with the rows in memory; above that the large islands'
sweep takes over.

Bar: with a fixed sweep count the split into islands changes no result (islands share no dynamic
body and every body sees the same visits in the same order), so positions, rotations, velocities
and impulses with and without island_solve are equal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = 1.0 / 120.0


def _sheet(m):
    """Lattice cells whose neighbour contacts number exactly m: a w x w sheet and a tail."""
    w = 1
    while 2 * (w + 1) * w <= m:
        w += 1
    cells = [(x, y) for y in range(w) for x in range(w)]
    return cells + [(w + k, 0) for k in range(m - 2 * w * (w - 1))]


def _scene(axm, sizes, seed, boxes):
    """One island per size: a sheet of touching bodies (spheres, or boxes and spheres mixed) whose
    first body rests on a static sphere; sheets stand 4 m apart."""
    rng = np.random.default_rng(seed)
    pos, typ, static = [], [], []
    for k, m in enumerate(sizes):
        z = 4.0 * k
        pos.append((0.0, 0.0, z))
        typ.append(axm.SHAPE_SPHERE)
        static.append(True)
        for x, y in _sheet(m - 1):
            pos.append((0.99 * x, 0.99 + 0.99 * y, z))
            typ.append(axm.SHAPE_BOX if boxes and (x + y // 2) % 3 else axm.SHAPE_SPHERE)
            static.append(False)
    n = len(pos)
    b = axm.Bodies(n)
    b.pos[:] = np.array(pos, np.float32)
    b.shape_type[:] = typ
    b.shape_params[:] = 0.5
    for i in range(n):
        if not static[i]:
            b.inv_mass[i], b.inv_inertia[i] = axm.mass_properties(typ[i], b.shape_params[i])
    move = ~np.array(static)
    b.lin_vel[move] = rng.normal(scale=0.3, size=(n, 3)).astype(np.float32)[move]
    b.ang_vel[move] = rng.normal(scale=0.3, size=(n, 3)).astype(np.float32)[move]
    return b


def _run(axm, b, split, sweeps, steps):
    d = axm.default_desc(num_planes=0, island_solve=split)
    for k in range(3):
        d.gravity[k] = 0.0
        d.origin[k] = -4.0
    w = axm.World(d)
    w.set_bodies(b)
    for _ in range(steps):
        st = w.step(DT, sweeps, axm.STEP_RESIDUAL)
    g, m, lab = w.get_bodies(), w.manifolds(), w.islands()[0]
    out = [g.pos.copy(), g.quat.copy(), g.lin_vel.copy(), g.ang_vel.copy(), w.impulses()[1], np.float32(st.residual)]
    dyn = np.where(b.inv_mass[m["a"]] > 0, m["a"], m["b"])
    _, count = np.unique(lab[dyn], return_counts=True)
    w.close()
    return out, sorted(count.tolist()), st


@pytest.mark.parametrize("boxes", [False, True])
@pytest.mark.parametrize("sizes", [
    [1, 2, 7, 8, 8, 8, 8, 8, 8, 8, 9, 9, 9, 9, 9, 15, 16],
    [16, 17, 17, 17, 31, 32, 33, 33, 63, 64, 65],
    [64, 65, 128, 255, 256, 257],
    [255, 257, 511, 512, 513, 1025],
    [4095, 4096, 4097],
    [3900] * 18,  # the largest class in several rounds of the register sweep
    [300] * 230,  # and one workgroup per island
])
def test_island_classes_equal_the_joint_sweep(axm, gpu, sizes, boxes):
    b = _scene(axm, sizes, 17 + len(sizes), boxes)
    one, count, _ = _run(axm, b, 1, 9, 1)
    if not boxes:  # boxes also touch across their corners: somewhat larger islands
        assert count == sorted(sizes)
    for steps in (1, 3):
        one, _, _ = _run(axm, b, 1, 9, steps)
        joint, _, _ = _run(axm, b, 0, 9, steps)
        for x, y in zip(one, joint):
            assert np.array_equal(x, y)


def test_more_colours_than_a_mask_holds(axm, gpu):
    """A hub sphere with 80 small ones around it needs more than 64 colours: its island takes the
    path without colour masks, beside small islands that do not need them."""
    rng = np.random.default_rng(3)
    v = rng.normal(size=(4000, 3))
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    spots = []
    for p in v:  # well-separated directions
        if all(np.dot(p, q) < 0.966 for q in spots):
            spots.append(p)
    spots = spots[:80]
    assert len(spots) > 64
    n = 1 + len(spots) + 4
    b = axm.Bodies(n)
    b.shape_params[:, 0] = 0.12
    b.shape_params[0, 0] = 1.0
    b.pos[1:1 + len(spots)] = np.array(spots, np.float32) * 1.11
    b.pos[1 + len(spots):] = [[8.0, 0.0, 0.23 * k] for k in range(4)]
    for i in range(n):
        b.inv_mass[i], b.inv_inertia[i] = axm.mass_properties(axm.SHAPE_SPHERE, b.shape_params[i])
    b.lin_vel[:] = rng.normal(scale=0.2, size=(n, 3))
    one, _, st = _run(axm, b, 1, 7, 2)
    joint, _, _ = _run(axm, b, 0, 7, 2)
    assert st.colours > 64
    for x, y in zip(one, joint):
        assert np.array_equal(x, y)
