"""axm_collide_pairs_noalloc from several threads at once: the calls share one staging buffer per
device, its queue of deep pairs included, and take turns on it, so each returns what it returns
alone."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _deep(n, s):
    """Boxes and capsules whose cores intersect: every pair goes through the queue."""
    rng = np.random.default_rng(s)
    q = rng.normal(size=(2, n, 4))
    q = (q / np.linalg.norm(q, axis=2, keepdims=True)).astype(np.float32)
    x = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    box = rng.uniform(0.4, 0.8, (n, 3)).astype(np.float32)
    cap = np.tile(np.array([0.3, 0.6, 0.0], np.float32), (n, 1))
    off = rng.uniform(-0.1, 0.1, (n, 3)).astype(np.float32)
    return np.full(n, 1, np.uint32), box, x, q[0], np.full(n, 2, np.uint32), cap, x + off, q[1]


@pytest.mark.parametrize("n", [1, 700, 16384])
def test_overlapping_calls_answer_as_alone(axm, gpu, n):
    threads, calls = 4, 6
    args = [_deep(n, 10 * n + t) for t in range(threads)]
    ref = [axm.collide_pairs(*a) for a in args]
    got = [[] for _ in range(threads)]
    start = threading.Barrier(threads)

    def work(t):
        start.wait()
        for _ in range(calls):
            got[t].append(axm.collide_pairs(*args[t], noalloc=True))

    ts = [threading.Thread(target=work, args=(t,)) for t in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for t in range(threads):
        assert len(got[t]) == calls and ref[t]["npts"].all()
        for g in got[t]:
            assert g["status"] == ref[t]["status"] == 0
            for k in ("npts", "pos", "normal", "depth", "feature"):
                assert np.array_equal(g[k], ref[t][k]), k
