"""What the two launches of timed sweeps are charged with: together every contact point's sweeps, each
in the launch it ran in.  Islands of 257 to 4096 manifolds are solved on their own, but swept beside
the large ones."""
import importlib.util
import os
import types

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DT = 1.0 / 120.0


def _bench():
    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


def test_bytes_follow_the_launches(axm):
    b = _bench()
    # 1000 point sweeps, 700 of them in islands solved on their own, 300 of these by workgroups and waves
    tot = types.SimpleNamespace(contact_sweeps=1000, local_contact_sweeps=700)
    prof = types.SimpleNamespace(bundle_point_sweeps=300, bundle_launches=2, bundle_ms=3.0, pgs_ms=5.0, pgs_launches=2)
    k = b.sweep_launches(tot, prof)
    assert k["k_pgs_solve (large islands)"][0] == 700 * b.B_SWEEP
    assert k["k_pgs_solve (other islands)"][0] == 300 * b.B_SWEEP
    assert sum(v[0] for v in k.values()) == tot.contact_sweeps * b.B_SWEEP


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,beside", [([300, 20, 5], 300), ([20, 200, 5], 0), ([5000, 600, 40], 600)])
def test_islands_are_counted_where_they_ran(axm, gpu, sizes, beside):
    from test_gpu_island_classes import _scene
    d = axm.default_desc(num_planes=0, island_solve=1)
    for k in range(3):
        d.gravity[k], d.origin[k] = 0.0, -4.0
    w = axm.World(d)
    w.set_bodies(_scene(axm, sizes, 3, False))  # spheres: one contact point per manifold
    w.totals(reset=True)
    w.profile(True)
    st = w.step(DT, 7)
    prof, tot = w.profile(False), w.totals()
    assert st.manifolds == st.contacts == sum(sizes)
    small = sum(s for s in sizes if s <= 4096)
    assert tot.contact_sweeps == 7 * sum(sizes) and tot.local_contact_sweeps == 7 * small
    assert prof.bundle_point_sweeps == 7 * (small - beside)
    assert np.isclose(sum(v[0] for v in _bench().sweep_launches(tot, prof).values()), 7 * sum(sizes) * 240.0)
    w.close()
