"""The solve order's sort where a workgroup takes several tiles (more than 128 x 2048 manifolds), with
a last tile that is not full and a last workgroup with fewer tiles than the others: by island and
colour (several passes) and by colour alone (one), against numpy's stable sort."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = 1.0 / 120.0
TILE, GROUPS = 2048, 128


def _rows(axm, n):
    """n spheres: three sheets of 48 x 48, more than 4096 manifolds each, and rows of 1 to 20; returns
    the bodies and how many touch."""
    rng = np.random.default_rng(n)
    sheet = np.stack(np.meshgrid(np.arange(48), np.arange(48), indexing="ij"), -1).reshape(-1, 2) * 0.98
    parts = [np.column_stack([sheet, np.full(len(sheet), -5.0 * k)]) for k in (1, 2, 3)]
    touching, left = 3 * 2 * 48 * 47, n - 3 * len(sheet)
    lens = []
    while left > 0:
        lens.append(min(int(rng.integers(1, 21)), left))
        left -= lens[-1]
    side = int(np.ceil(np.sqrt(len(lens))))
    for k, m in enumerate(lens):
        parts.append(np.stack([0.98 * np.arange(m), np.full(m, 1.5 * (k // side)), np.full(m, 1.5 * (k % side))], 1))
    b = axm.Bodies(n)
    # an island's bodies and manifolds lie apart in memory
    b.pos[rng.permutation(n)] = np.concatenate(parts).astype(np.float32)
    b.inv_mass[:] = 1.0
    b.inv_inertia[:] = 2.5
    b.shape_params[:, 0] = 0.5
    return b, touching + sum(lens) - len(lens)


@pytest.mark.parametrize("n", [300007, 700001])
def test_solve_order_over_several_tiles(axm, gpu, n):
    b, m = _rows(axm, n)
    tiles = -(-m // TILE)
    run = -(-tiles // GROUPS)
    assert m > GROUPS * TILE and m % TILE and tiles % run, "the case this is about"
    for split in (1, 0):
        d = axm.default_desc(num_planes=0, island_solve=split)
        for k in range(3):
            d.gravity[k], d.origin[k] = 0.0, -60.0
        w = axm.World(d)
        w.set_bodies(b)
        st = w.step(DT, 1)
        assert st.overflow == 0 and st.manifolds == m
        a = w.manifolds()["a"].astype(np.int64)
        col, order, *_ = w.colours()
        key = col.astype(np.int64)
        if split:
            root = w.islands()[0][a].astype(np.int64)
            local = np.bincount(root, minlength=n)[root] <= 4096
            assert local.any() and not local.all()
            key = np.where(local, (1 << 31) | root << 8, 0) | key
        assert np.array_equal(order, np.argsort(key, kind="stable"))
        w.close()
