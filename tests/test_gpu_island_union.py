"""The islands of a step on both sides of the body count where their union moves from LDS to memory,
against a plain search over the same manifolds: labels are the smallest body index of the component,
with long chains (a row of touching spheres), many components and bodies in any order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = 1.0 / 120.0


def _rows(axm, n, length, s):
    """n spheres in rows of `length` touching ones, body numbers shuffled, no gravity."""
    rng = np.random.default_rng(s)
    b = axm.Bodies(n)
    i = np.arange(n)
    row, col = i // length, i % length
    p = np.zeros((n, 3), np.float32)
    p[:, 0] = col * 0.999
    p[:, 1] = (row % 181) * 3.0
    p[:, 2] = (row // 181) * 3.0
    order = rng.permutation(n)
    b.pos[:] = p[order]
    b.inv_mass[:] = 1.0
    b.inv_inertia[:] = 2.5
    b.shape_type[:] = 0
    b.shape_params[:, 0] = 0.5
    b.inv_mass[order[:n // 50]] = 0.0  # static bodies cut some rows
    b.inv_inertia[b.inv_mass == 0] = 0.0
    return b


def _components(n, a, b):
    par = np.arange(n)

    def find(x):
        while par[x] != x:
            par[x] = par[par[x]]
            x = par[x]
        return x

    for x, y in zip(a.tolist(), b.tolist()):
        x, y = find(x), find(y)
        if x != y:
            par[max(x, y)] = min(x, y)
    return np.array([find(x) for x in range(n)])


@pytest.mark.parametrize("n,length", [(1, 1), (700, 700), (1025, 5), (36864, 300), (36865, 300)])
def test_labels_are_components(axm, gpu, n, length):
    b = _rows(axm, n, length, n)
    d = axm.default_desc()
    d.gravity[0] = d.gravity[1] = d.gravity[2] = 0.0
    w = axm.World(d)
    w.set_bodies(b)
    st = w.step(DT, 2)
    m = w.manifolds()
    dyn = b.inv_mass > 0
    both = np.array([y < n and dyn[x] and dyn[y] for x, y in zip(m["a"].tolist(), m["b"].tolist())], bool)
    want = _components(n, m["a"][both], m["b"][both])
    lab, _, _ = w.islands()
    assert np.array_equal(lab[dyn], want[dyn])
    assert st.islands == len(np.unique(want[dyn]))
    w.close()
