"""EPA on a box and a capsule whose polytope expansion meets a face without area: the pair ends
with EPAFailedToConverge and a contact, and that contact depends on the pair alone, not on what
earlier pairs left in the expansion's work area."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BOX = ([0.29069840908050537, 0.7301080226898193, 0.3185819089412689], [1.489362359046936, 384.7976989746094, 7.49639368057251],
       [0.31333789229393005, 0.2771002948284149, 0.7784448266029358, -0.46803683042526245])
CAPSULE = ([0.3833067715167999, 0.9943984746932983, 0.0], [2.9931912422180176, 384.800537109375, 7.529688835144043],
           [0.6862992644309998, -0.6402513980865479, -0.3449994921684265, -0.0068524847738444805])


def _pairs(n, at, seed):
    """n overlapping box-capsule pairs, the degenerate one at index `at`."""
    rng = np.random.default_rng(seed)
    ta, tb = np.full(n, 1, np.uint32), np.full(n, 2, np.uint32)
    pa = rng.uniform(0.25, 0.75, (n, 3)).astype(np.float32)
    pb = rng.uniform(0.25, 0.75, (n, 3)).astype(np.float32)
    xa = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    xb = (xa + 0.2 * rng.normal(size=(n, 3))).astype(np.float32)
    q = rng.normal(size=(2, n, 4))
    qa, qb = (q / np.linalg.norm(q, axis=2, keepdims=True)).astype(np.float32)
    pa[at], xa[at], qa[at] = BOX
    pb[at], xb[at], qb[at] = CAPSULE
    return ta, pa, xa, qa, tb, pb, xb, qb


@pytest.mark.parametrize("n,at", [(1, 0), (64, 63), (640, 17)])
def test_degenerate_face_result_depends_on_the_pair_alone(axm, orc, gpu, n, at):
    seen = []
    for seed in range(4):
        args = _pairs(n, at, seed)
        out, status = axm.gjk_epa_pairs(*args)
        assert status[at] == 302 and np.isfinite(out[at]).all()
        seen.append(out[at])
        m = axm.collide_pairs(*args)
        assert m["status"] == 302 and m["npts"][at] == 1 and np.isfinite(m["pos"][at]).all()
    for o in seen[1:]:
        assert np.array_equal(o, seen[0])
    ref, rst = orc.gjk_epa(1, *BOX, 2, *CAPSULE)
    assert rst == 302
    assert np.allclose(seen[0], ref[:10], rtol=1e-5, atol=1e-4)
