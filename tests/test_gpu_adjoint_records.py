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


@pytest.mark.parametrize("graph", [False, True])
def test_checkpoint_that_finds_no_memory(graph, monkeypatch):
    """A step call that stops because a checkpoint finds no memory leaves the
    state of the steps it took, with their forces, counts and cell keys; a
    state set afterwards is the one the next steps start from."""
    from grains3dgpu_amd import engine
    from grains3dgpu_amd.engine import GrainsError
    sc = lattice_superquadrics(n_side=5, n_rng=(2.0, 2.0))

    def make():
        return S.load(engine.Engine(dt=sc.dt, precision=A.FP64, gjk_rel_tol=1e-12), sc)

    def result(e):
        return [*e.get_state(), *e.get_torce(), e.get_contact_count(), *e.get_cell_keys()]

    want, want0 = make(), make()
    want.step(10, graph=graph)
    want0.step(4, graph=graph)
    # room for the checkpoints of the start and of 5 steps, not of 10
    monkeypatch.setenv("GRAINS_ADJOINT_BYTES", str(3 * 104 * sc.n - 1))
    e = make()
    e.adjoint_record(5)
    with pytest.raises(GrainsError, match="GRAINS_ADJOINT_BYTES"):
        e.step(13, graph=graph)
    for a, b in zip(result(e), result(want)):
        np.testing.assert_array_equal(a, b)
    e.set_state(sc.pos, sc.quat, sc.vel, sc.omega)
    e.reset_contact_count()
    monkeypatch.delenv("GRAINS_ADJOINT_BYTES")
    e.set_sims(sc)  # (a new layout ends the recording)
    e.step(4, graph=graph)
    for a, b in zip(result(e), result(want0)):
        np.testing.assert_array_equal(a, b)


def test_state_set_after_a_step_call_that_stopped(monkeypatch):
    """As above, without a new layout between: the run that stopped left
    records ahead of the state's planes."""
    from grains3dgpu_amd import engine
    from grains3dgpu_amd.engine import GrainsError
    sc = lattice_superquadrics(n_side=5, n_rng=(2.0, 2.0))
    monkeypatch.setenv("GRAINS_ADJOINT_BYTES", str(2 * 104 * sc.n - 1))
    e = S.load(engine.Engine(dt=sc.dt, precision=A.FP64, gjk_rel_tol=1e-12), sc)
    want = S.load(engine.Engine(dt=sc.dt, precision=A.FP64, gjk_rel_tol=1e-12), sc)
    want.step(3)
    e.adjoint_record(5)
    with pytest.raises(GrainsError, match="GRAINS_ADJOINT_BYTES"):
        e.step(8)
    e.set_state(sc.pos, sc.quat, sc.vel, sc.omega)
    e.step(3)
    for a, b in zip(e.get_state(), want.get_state()):
        np.testing.assert_array_equal(a, b)


def test_log_gives_way_to_checkpoints_and_sweep(monkeypatch):
    """The logged states are kept where there is memory to spare: with room for
    the checkpoints, or for them, the sweep's buffers and a block run again,
    but not for the log as well, recording and sweep go on without it.  Bytes a
    particle: a state 104, ten steps to a block, five checkpoints; the sweep
    364, 244 for each of max_neighbors, 36 for each of six walls."""
    from grains3dgpu_amd import engine
    sc = lattice_superquadrics(n_side=5, n_rng=(2.0, 2.0))
    rng = np.random.default_rng(7)
    w = [rng.standard_normal((sc.n, k)) for k in (3, 4, 3, 3)]
    K = 16
    sweep = 364 + 244 * K + 36 * 6

    def run(per_particle):
        monkeypatch.setenv("GRAINS_ADJOINT_BYTES", str(per_particle * sc.n))
        e = S.load(engine.Engine(dt=sc.dt, precision=A.FP64, gjk_rel_tol=1e-12, max_neighbors=K), sc)
        e.adjoint_record(10)
        e.step(42)
        return e

    want = run(0)
    # two blocks logged and two checkpoints, but not the third checkpoint
    short = run(2 * 11 * 104 + 52)
    for a, b in zip(short.get_state(), want.get_state()):
        np.testing.assert_array_equal(a, b)
    # all of the recording, but not the sweep beside it (1 %: allocations rounded up)
    tight = run(int(1.01 * (15 * 104 + sweep)) + 100)
    g, g0 = want.adjoint(*w, want_state0=True)
    h, h0 = tight.adjoint(*w, want_state0=True)
    assert np.abs(g).max() > 0
    for a, b in zip([g, *g0], [h, *h0]):
        np.testing.assert_array_equal(a, b)
