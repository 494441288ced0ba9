"""The network's kernels at the edges of their tiles: rows are independent in the forward pass (a
prefix gives the same bits as the whole), gradients of few and of odd row counts match the CPU
oracle, and a training run is, bit for bit, its batches' gradients and Adam steps one by one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _net(axm, s):
    net = axm.Mlp(0)
    net.init(s)
    return net


def test_forward_rows_are_independent(axm, gpu):
    rng = np.random.default_rng(1)
    net = _net(axm, 3)
    X = rng.normal(size=(70001, 24)).astype(np.float32)
    whole = net.forward(X)
    for n in (1, 15, 16, 17, 31, 32, 33, 255, 257, 8191, 65535, 65537):
        assert np.array_equal(net.forward(X[:n]), whole[:n]), n
    # rows that begin in the middle of a tile
    assert np.array_equal(net.forward(X[13:1000]), whole[13:1000])


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 129, 16385])
def test_gradient_at_tile_edges(axm, orc, gpu, n):
    rng = np.random.default_rng(n)
    net = _net(axm, 4)
    X = rng.normal(size=(n, 24)).astype(np.float32)
    Y = rng.normal(size=(n, 3)).astype(np.float32)
    loss, g = net.loss_grad(X, Y)
    lo, go = orc.mlp_grad(net.params, X, Y, emu=True, fp64=False)
    go = go.astype(np.float64)
    # the oracle sums in another order: a bf16 tie that falls the other way moves a hidden value by
    # 2^-8, and with it one row's output error; more than one per cent of the whole it cannot be
    assert abs(loss - lo) <= 1e-2 * max(1.0, lo)
    assert np.linalg.norm(g - go) <= 1e-2 * np.linalg.norm(go)


@pytest.mark.parametrize("n,batch", [(1, 1), (200, 64), (5000, 1777), (40000, 17000)])
def test_training_is_its_steps(axm, gpu, n, batch):
    rng = np.random.default_rng(n)
    X = rng.normal(size=(n, 24)).astype(np.float32)
    Y = rng.normal(size=(n, 3)).astype(np.float32)
    a, b = _net(axm, 5), _net(axm, 5)
    a.train(X, Y, 2, batch, 1e-3)
    for _ in range(2):
        for r in range(0, n, batch):
            _, g = b.loss_grad(X[r:r + batch], Y[r:r + batch])
            b.adam_step(g, lr=1e-3)
    assert np.array_equal(a.params, b.params)
    assert np.array_equal(a.forward(X[:64]), b.forward(X[:64]))  # the bf16 copies follow the parameters
