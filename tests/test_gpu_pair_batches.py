"""Batches of shape pairs: a pair's result is the pair's own, whatever its place and the batch's size
(tiles of 64 to 1024 pairs, expansion of deep pairs by waves of a queue); deep pairs of every kind
expand as the CPU oracle does; calls from several threads at once keep to their own results."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _args(n, s, spread=0.6, planes=True):
    rng = np.random.default_rng(s)
    ta = rng.integers(0, 3, n).astype(np.uint32)
    tb = rng.integers(0, 4 if planes else 3, n).astype(np.uint32)
    pa, pb = (rng.uniform(0.25, 0.75, (n, 3)).astype(np.float32) for _ in range(2))
    xa = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    xb = (xa + spread * rng.normal(size=(n, 3))).astype(np.float32)
    q = rng.normal(size=(2, n, 4))
    qa, qb = (q / np.linalg.norm(q, axis=2, keepdims=True)).astype(np.float32)
    up = rng.normal(size=(n, 3))
    up /= np.linalg.norm(up, axis=1, keepdims=True)
    pb[tb == 3] = up[tb == 3]
    xb[tb == 3] = 0.0
    return ta, pa, xa, qa, tb, pb, xb, qb


FIELDS = ("npts", "pos", "normal", "depth", "feature")


@pytest.mark.parametrize("n", [1, 63, 65, 16384, 16385, 32769, 262145])
def test_results_do_not_depend_on_the_batch(axm, gpu, n):
    whole = _args(n, 3)
    out = axm.collide_pairs(*whole)
    g = _args(n, 4, planes=False)
    o, st = axm.gjk_epa_pairs(*g)
    assert (st == 1).sum() * 8 > n or n < 64
    rng = np.random.default_rng(n)
    for lo, k in {(0, min(n, 40)), (max(0, n - 61), min(n, 61)), (int(rng.integers(n)), 1), (n // 3, min(100, n - n // 3))}:
        part = axm.collide_pairs(*[a[lo:lo + k] for a in whole])
        for f in FIELDS:
            assert np.array_equal(part[f], out[f][lo:lo + k]), (f, lo, k)
        po, ps = axm.gjk_epa_pairs(*[a[lo:lo + k] for a in g])
        assert np.array_equal(po, o[lo:lo + k]) and np.array_equal(ps, st[lo:lo + k])


@pytest.mark.parametrize("spread", [0.3, 0.02])
def test_expansion_matches_oracle(axm, orc, gpu, spread):
    n = 600
    ta, pa, xa, qa, tb, pb, xb, qb = _args(n, 11, spread, planes=False)
    out, st = axm.gjk_epa_pairs(ta, pa, xa, qa, tb, pb, xb, qb)
    deep = 0
    for i in range(n):
        o, s = orc.gjk_epa(int(ta[i]), pa[i], xa[i], qa[i], int(tb[i]), pb[i], xb[i], qb[i])
        assert st[i] == s, i
        # the same operations in the same order
        assert np.array_equal(out[i], np.asarray(o[:10], np.float32)), i
        deep += s == 1
    assert deep > n // 10


def test_calls_from_threads(axm, gpu):
    jobs = [_args(n, 20 + k) for k, n in enumerate((5000, 300, 20000, 64))]
    want = [axm.collide_pairs(*j) for j in jobs]
    bad = []

    def work(k):
        for _ in range(5):
            got = axm.collide_pairs(*jobs[k])
            if not all(np.array_equal(got[f], want[k][f]) for f in FIELDS):
                bad.append(k)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(len(jobs))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
