"""The reverse sweep takes its contacts' closest points from the step's
searches where the two-pass FP64 narrow phase leaves them, and searches again
otherwise; it takes the states between checkpoints from the log of the
recorded steps, and runs them again where the log does not stand (a state set
while recording).  All run the same arithmetic, so the gradients are equal bit for
bit: touching ellipsoids, spheres among ellipsoids, several checkpoint blocks."""
import numpy as np
import pytest

from grains3dgpu_amd import _abi as A
from grains3dgpu_amd import scene as S
from tests.scenes import lattice_superquadrics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which", ["ellipsoids", "mixed"])
def test_recorded_searches_give_the_same_gradients(which):
    from grains3dgpu_amd import engine
    if which == "ellipsoids":
        sc = lattice_superquadrics(n_side=7, n_rng=(2.0, 2.0))
    else:
        sc = S.config4(n=125, seed=5, vel=0.5, a_rng=(0.4e-3, 0.6e-3), jitter=0.05, layout="lattice")
    rng = np.random.default_rng(5)
    w = [rng.standard_normal((sc.n, k)) for k in (3, 4, 3, 3)]
    out = []
    for passes, log in ((1, True), (2, True), (2, False)):
        e = S.load(engine.Engine(dt=sc.dt, precision=A.FP64, gjk_rel_tol=1e-12, narrow_passes=passes), sc)
        e.adjoint_record(10)
        if not log:
            e.set_state(*e.get_state())
        e.step(42)
        assert e.get_stats()["contacts"] > 0
        g, g0 = e.adjoint(*w, want_state0=True)
        out.append([g, *g0])
    assert np.abs(out[0][0]).max() > 0
    for a, b, c in zip(*out):
        np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(a, c)


def test_passes_changed_between_two_sweeps():
    """The records are the step's own: a sweep in one pass, whose searches
    leave none, does not take those of the sweep before it in two."""
    from grains3dgpu_amd import engine
    sc = lattice_superquadrics(n_side=5, n_rng=(2.0, 2.0))
    rng = np.random.default_rng(6)
    w = [rng.standard_normal((sc.n, k)) for k in (3, 4, 3, 3)]
    e = S.load(engine.Engine(dt=sc.dt, precision=A.FP64, gjk_rel_tol=1e-12, narrow_passes=2), sc)
    e.adjoint_record(5)
    e.step(12)
    out = []
    for passes in (2, 1, 2, 1):
        e.set_narrow_passes(passes)
        g, g0 = e.adjoint(*w, want_state0=True)
        out.append([g, *g0])
    assert np.abs(out[0][0]).max() > 0
    for o in out[1:]:
        for a, b in zip(out[0], o):
            np.testing.assert_array_equal(a, b)
