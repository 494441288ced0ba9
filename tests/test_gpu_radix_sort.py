"""The step's sorts at the edges of their tiles, in one workgroup and in several: bodies by cell key
(through the broadphase's pairs) and manifolds by solve order, against numpy's stable sort."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = 1.0 / 120.0


def _towers(axm, n, s):
    """n spheres, a fifth of them in touching pairs, scattered over a wide floor of cells."""
    rng = np.random.default_rng(s)
    b = axm.Bodies(n)
    side = int(np.ceil(n ** (1 / 3))) + 1
    cell = rng.permutation(side ** 3)[:n]
    p = np.stack([cell // side ** 2, cell // side % side, cell % side], 1).astype(np.float32) * 2.0
    touch = rng.permutation(n - 1)[:n // 5] if n > 1 else np.zeros(0, int)
    p[touch + 1] = p[touch] + np.array([0.98, 0.0, 0.0], np.float32)
    b.pos[:] = p
    b.inv_mass[:] = 1.0
    b.inv_inertia[:] = 2.5
    b.shape_params[:, 0] = 0.5
    return b


def _check(axm, w, n, s, worlds=1):
    b = _towers(axm, n, s)
    if worlds > 1:
        b.world[:] = np.arange(n) * worlds // n
    w.set_bodies(b)
    st = w.step(DT, 2)
    assert st.overflow == 0
    m = w.manifolds()
    a, o = m["a"].astype(np.int64), m["b"].astype(np.int64)
    # every touching pair is found, each once
    d = b.pos[a[o < n]] - b.pos[o[o < n]]
    assert len(np.unique(a * (n + 1) + np.minimum(o, n))) == len(a)
    assert (np.linalg.norm(d, axis=1) < 1.1).all() and len(a) >= n // 8
    col, order, *_ = w.colours()
    lab, _, _ = w.islands()
    root = lab[a]
    size = np.bincount(root, minlength=n)
    local = size[root] <= 4096
    key = np.where(local, (1 << 31) | root.astype(np.int64) << 8, 0) | col.astype(np.int64)
    assert np.array_equal(order, np.argsort(key, kind="stable"))


@pytest.mark.parametrize("sizes", [(1, 2, 4095, 4096, 4097, 300), (9001,), (12288, 12289), (70001,)])
def test_sorts(axm, gpu, sizes):
    d = axm.default_desc()
    d.gravity[0] = d.gravity[1] = d.gravity[2] = 0.0
    w = axm.World(d)
    for k, n in enumerate(sizes):
        _check(axm, w, n, k)
    w.close()


def test_sort_arrays_end_at_a_page(axm, gpu):
    """524288 bodies: the arrays of a word per body are whole pages, so a word written past one of
    them (the total of the cell ranks' scan was) would be in a page of something else or of nothing."""
    d = axm.default_desc()
    d.gravity[0] = d.gravity[1] = d.gravity[2] = 0.0
    w = axm.World(d)
    _check(axm, w, 524288, 4)
    w.close()


@pytest.mark.parametrize("n, worlds", [(131072, 1), (131073, 1), (135168, 1), (140001, 1), (131073, 2), (139264, 700)])
def test_sort_by_passes(axm, gpu, n, worlds):
    """Either side of the count above which bodies are sorted pass by pass: a last tile of one key, whole
    tiles, and keys with the world above the cell (31 and 40 bits, in four passes)."""
    d = axm.default_desc()
    d.gravity[0] = d.gravity[1] = d.gravity[2] = 0.0
    w = axm.World(d)
    _check(axm, w, n, 5, worlds)
    w.close()
