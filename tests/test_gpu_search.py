"""The queued FP64 searches (k_search64): lanes refilled from a queue, one lane
per entry on long queues, four on short ones.  Their results are those of the
single complete pass (gjk_sv, one lane per entry from start to end) bit for
bit: the same operations on the same values."""
import numpy as np
import pytest

from grains3dgpu_amd import _abi as A
from grains3dgpu_amd import scene as S
from tests.scenes import (dense_cylinders_cones, dense_spheres, dense_superquadrics, lattice_superquadrics, rel_err)

pytestmark = pytest.mark.gpu


def run(sc, passes, flags=0, precision=A.FP64, tol=1e-10, steps=2):
    from grains3dgpu_amd import engine
    e = S.load(engine.Engine(dt=sc.dt, precision=precision, flags=flags, gjk_rel_tol=tol, narrow_passes=passes,
                             max_neighbors=64), sc)
    e.step(steps)
    out = e.get_torce() + e.get_state() + (e.get_contact_count(),)
    st = e.get_stats()
    e.close()
    return out, st


@pytest.mark.parametrize("make", [
    lambda: lattice_superquadrics(n_side=2, seed=5),              # fewer entries than waves
    lambda: dense_superquadrics(n=700, seed=6, box_frac=0.3),     # overlapping cores, boxes
    lambda: dense_superquadrics(n=300, seed=8, n_rng=(2.0, 2.0)),  # ellipsoids
    lambda: dense_cylinders_cones(n=500, seed=9),
    lambda: dense_spheres(n=400, seed=10),                        # no search at all
    lambda: S.config2(n=1200, seed=3, phi=0.5, resolve=False),    # hulls
], ids=["few", "cores", "ellipsoids", "cylinders", "spheres", "hulls"])
@pytest.mark.parametrize("flags", [0, A.NESTEROV])
def test_short_queue_equals_single_pass(make, flags):
    sc = make()
    (a, sa), (b, sb) = run(sc, 1, flags), run(sc, 2, flags)
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)
    assert sa["contacts"] > 0
    for k in ("gjk_calls", "gjk_iterations", "gjk_max_iterations", "deep_contacts", "contacts"):
        assert sa[k] == sb[k], k


def test_long_queue():
    """More than 98,304 entries (the one-lane form).  FP64: equal to the
    single pass.  FP32-mixed with FP64 contact geometry: its re-runs and the
    FP64 path's searches stop at a relative gap of 1e-10 from different
    starts; a gap g pins a contact normal to sqrt(2 g) = 1.4e-5, so forces
    agree to 5e-5 of the largest."""
    sc = lattice_superquadrics(n_side=27, seed=12)
    (a, sa), (b, sb) = run(sc, 1, steps=1), run(sc, 2, steps=1)
    assert sb["narrow_deferred"] > 98304
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)
    assert sa["gjk_iterations"] == sb["gjk_iterations"]
    m, sm = run(sc, 2, flags=A.WARM_START | A.FP64_CONTACTS, precision=A.FP32_MIXED, tol=1e-6, steps=1)
    assert sm["fp64_refines"] > 98304
    np.testing.assert_array_equal(m[6], b[6])
    assert rel_err(m[0], b[0]) < 5e-5
