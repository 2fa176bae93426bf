"""Neighbour lists kept over several steps.  A run that keeps its lists equals
one whose lists are built anew for every step (the state set between steps:
positions and orientations unchanged, so the next step starts from the same
bits), bit for bit: state, forces, contact counts, cell keys, pair lists and
counters."""
import numpy as np
import pytest

from grains3dgpu_amd import _abi as A
from grains3dgpu_amd import scene as S
from tests.scenes import bimodal_spheres, dense_cylinders_cones, dense_spheres, dense_superquadrics

pytestmark = pytest.mark.gpu


def two_beds():
    a = dense_spheres(n=300, seed=3, vel=4.0, periodic=0b011)
    b = dense_spheres(n=500, seed=4, vel=0.5, periodic=0)
    n = len(a.pos)
    return S.Scene(shapes=a.shapes, tables=a.tables, n_materials=1, sims=[a.sims[0], b.sims[0]],
                   particle_shape=np.r_[a.particle_shape, b.particle_shape],
                   particle_sim=np.r_[np.zeros(n, np.uint32), np.ones(len(b.pos), np.uint32)],
                   pos=np.r_[a.pos, b.pos], quat=np.r_[a.quat, b.quat], vel=np.r_[a.vel, b.vel],
                   omega=np.r_[a.omega, b.omega], dt=1e-6)


def small_cells():
    # cells of 0.7 of the largest diameter: pairs in reach but not in
    # neighbouring cells are no candidates
    sc = dense_spheres(n=600, seed=5, vel=6.0)
    sc.sims[0]["cell_size"] = 0.7e-3
    return sc


def outside():
    # centres beyond periodic and open sides
    sc = dense_spheres(n=500, seed=6, vel=3.0, periodic=0b001)
    sc.pos[::7] += sc.sims[0]["domain_max"][0] * 0.3 * np.random.default_rng(1).uniform(-1, 1, sc.pos[::7].shape)
    return sc


SCENES = {
    "fast": lambda: dense_spheres(n=700, seed=2, vel=8.0, periodic=0b011),
    "slow": lambda: dense_spheres(n=400, seed=7, vel=0.01, walls=True),
    "two_beds": two_beds,
    "small_cells": small_cells,
    "wide_cells": lambda: _factor(dense_spheres(n=800, seed=8, vel=5.0), 1.6),
    "outside": outside,
    "superquadrics": lambda: dense_superquadrics(n=300, seed=9, vel=4.0),
    "cylinders": lambda: dense_cylinders_cones(n=300, seed=10, vel=4.0),
    "bimodal": lambda: bimodal_spheres(n_small=4000),
    "few_cells": lambda: dense_spheres(n=60, seed=11, vel=3.0, periodic=0b111),  # three or four cells a side
}


def _factor(sc, f):
    sc.sims[0]["cell_size_factor"] = f
    return sc


def result(e):
    return [*e.get_state(), *e.get_torce(), e.get_contact_count(), *e.get_cell_keys(),
            e.get_pairs(A.PAIRS_CANDIDATE), e.get_pairs(A.PAIRS_CONTACT)]


@pytest.mark.parametrize("name", SCENES)
@pytest.mark.parametrize("precision,flags,mode", [(A.FP64, 0, 0), (A.FP32_MIXED, 0, 3), (A.FP64, A.REF_QUIRKS, 2)])
def test_kept_lists_equal_fresh_ones(name, precision, flags, mode):
    from grains3dgpu_amd import engine
    sc = SCENES[name]()
    steps = 25

    def make():
        return S.load(engine.Engine(dt=sc.dt, precision=precision, flags=flags, max_neighbors=96,
                                    gjk_rel_tol=1e-6 if precision == A.FP32_MIXED else 0.0,
                                    candidate_staging=mode), sc)
    kept, fresh, graph = make(), make(), make()
    kept.step(steps)
    graph.step(steps, graph=True)
    cand = contacts = outside = 0
    for k in range(steps):
        if k:
            fresh.set_state(*fresh.get_state())
        fresh.step(1)
        st = fresh.get_stats()
        cand, contacts, outside = (cand + st["candidate_pairs"], contacts + st["contacts"],
                                   outside + st["out_of_domain"])
    want = result(fresh)
    for e in (kept, graph):
        for a, b in zip(result(e), want):
            np.testing.assert_array_equal(a, b)
        st = e.get_stats()
        assert (st["steps"], st["candidate_pairs"], st["contacts"], st["out_of_domain"]) == (steps, cand, contacts,
                                                                                           outside)
        # single steps go on from the same lists
        e.step(1)
        e.step(2)
    for a, b in zip(result(kept), result(graph)):
        np.testing.assert_array_equal(a, b)


def test_lists_too_long_with_the_skin():
    """max_neighbors holds every step's candidates but not the lists with
    their skin: the run goes on without one and equals one with room; one
    short of the candidates is an overflow, as before."""
    from grains3dgpu_amd import engine
    from grains3dgpu_amd.engine import GrainsError
    sc = dense_spheres(n=500, seed=12, vel=0.01)
    full = S.load(engine.Engine(dt=sc.dt, max_neighbors=96), sc)
    full.step(5)
    most = full.get_stats()["max_candidates"]
    tight = S.load(engine.Engine(dt=sc.dt, max_neighbors=most), sc)
    tight.step(5)
    for a, b in zip(result(tight), result(full)):
        np.testing.assert_array_equal(a, b)
    assert tight.get_stats()["max_candidates"] == most
    short = S.load(engine.Engine(dt=sc.dt, max_neighbors=most - 1), sc)
    with pytest.raises(GrainsError, match="max_neighbors"):
        short.step(5)


@pytest.mark.parametrize("scheme", [A.FIRST_ORDER_EXPLICIT, A.SECOND_ORDER_EXPLICIT, A.SECOND_ORDER_LEAPFROG,
                                    A.SECOND_ORDER_ADAMS_BASHFORTH])
@pytest.mark.parametrize("which", ["fast", "slow", "cylinders"])
def test_state_between_the_steps_of_a_run(which, scheme):
    """The steps of a run advance the records in list order; the state (and a
    two-step scheme's history) is written back at the run's end and before
    every build.  A run cut in two by a snapshot taken and put back, which
    builds anew from the state, and one cut into single steps equal it."""
    from grains3dgpu_amd import engine
    sc = SCENES[which]()

    def eng():
        return S.load(engine.Engine(dt=sc.dt, precision=A.FP64, integrator=scheme), sc)

    whole, cut, single = eng(), eng(), eng()
    whole.step(40)
    cut.step(13)
    cut.restore(cut.snapshot())
    cut.step(27)
    for _ in range(40):
        single.step(1)
    for a, b, c in zip(whole.get_state(), cut.get_state(), single.get_state()):
        np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(a, c)
    for a, b, c in zip(whole.get_torce(), cut.get_torce(), single.get_torce()):
        np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(a, c)


def test_lists_of_small_cells_hold_their_candidates_only():
    """Cells smaller than the grains: pairs that overlap beyond neighbouring
    cells are no candidates and take no room in max_neighbors (at most 8 of
    the 13 overlapping neighbours of a sphere here)."""
    from grains3dgpu_amd import engine
    sc = dense_spheres(n=600, seed=5, vel=0.01)
    sc.sims[0]["cell_size"] = 0.35e-3
    full = S.load(engine.Engine(dt=sc.dt, max_neighbors=96), sc)
    full.step(5)
    most = full.get_stats()["max_candidates"]
    assert most == 8
    tight = S.load(engine.Engine(dt=sc.dt, max_neighbors=most), sc)
    tight.step(5)
    for a, b in zip(result(tight), result(full)):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("mode", [0, 3])
def test_lists_that_outgrow_their_room_keep_the_warm_starts(mode):
    """A bed drawn together until its lists with the skin outgrow
    max_neighbors in the middle of a run: the directions its searches start
    from outlast the build that did not fit."""
    from grains3dgpu_amd import engine
    sc = dense_superquadrics(n=400, seed=9, phi=0.12, vel=0.0, periodic=0, walls=False)
    mid = 0.5 * np.asarray(sc.sims[0]["domain_max"])
    sc.vel = -4000.0 * (sc.pos - mid)

    def make(k):
        return S.load(engine.Engine(dt=sc.dt, precision=A.FP32_MIXED, flags=A.WARM_START | A.FP64_CONTACTS,
                                    max_neighbors=k, gjk_rel_tol=1e-6, candidate_staging=mode), sc)
    roomy = make(128)
    roomy.step(60)
    most = roomy.get_stats()["max_candidates"]
    tight = make(most)
    tight.step(60)
    assert tight.get_stats()["max_candidates"] == most
    for a, b in zip(result(tight), result(roomy)):
        np.testing.assert_array_equal(a, b)


def test_pairs_and_keys_of_a_new_layout_are_refused():
    """Pairs and cell keys are those of a step: none before a layout's first."""
    from grains3dgpu_amd import engine
    from grains3dgpu_amd.engine import GrainsError
    sc = dense_spheres(n=300, seed=14)
    e = S.load(engine.Engine(dt=sc.dt), sc)
    e.step(2)
    assert len(e.get_pairs(A.PAIRS_CANDIDATE))
    e.set_sims(sc)
    e.step(0)
    for read in (e.get_pairs, e.get_cell_keys):
        with pytest.raises(GrainsError, match="no step"):
            read()
    e.step(1)
    assert len(e.get_pairs(A.PAIRS_CANDIDATE))


@pytest.mark.parametrize("n", [1, 3, 300, 1025, 20000])
def test_key_order_is_stable(n):
    """The particles by (cell key, id), through one block or the radix passes,
    after a step that has changed cells."""
    import dataclasses
    from grains3dgpu_amd import engine
    sc = dense_spheres(n=max(n, 300), seed=15, vel=20.0, periodic=0b011)
    sc = dataclasses.replace(sc, **{k: getattr(sc, k)[:n] for k in ("pos", "quat", "vel", "omega", "particle_shape")})
    e = S.load(engine.Engine(dt=sc.dt, max_neighbors=64), sc)
    e.step(20)
    key, order = e.get_cell_keys()
    np.testing.assert_array_equal(order, np.argsort(key, kind="stable"))


@pytest.mark.parametrize("warm", [False, True])
def test_centres_outside_periodic_sides_as_the_oracle(warm, oracle_lib):
    """A run that starts with centres outside periodic sides: they take the
    neighbours of the border cell they are folded into, as in the reference's
    cells, until the step wraps them; then the run goes on as from there."""
    from grains3dgpu_amd import engine
    sc = dense_spheres(n=1500, seed=16, vel=0.5, periodic=0b011)
    sc.pos[::5, :2] -= 0.12 * np.asarray(sc.sims[0]["domain_max"])[:2]
    kw = dict(precision=A.FP32_MIXED, flags=A.WARM_START | A.FP64_CONTACTS, gjk_rel_tol=1e-6) if warm else {}
    e = S.load(engine.Engine(dt=sc.dt, max_neighbors=96, **kw), sc)
    o = S.load(oracle_lib.Oracle(dt=sc.dt), sc)
    o.step(1)
    e.step(1)
    assert e.get_stats()["out_of_domain"] > 0
    for which in (A.PAIRS_CANDIDATE, A.PAIRS_CONTACT):
        np.testing.assert_array_equal(e.get_pairs(which), o.get_pairs(which))
    # in one run, by graph, and cut after the first step by a state put back
    whole, cut = [S.load(engine.Engine(dt=sc.dt, max_neighbors=96, **kw), sc) for _ in range(2)]
    whole.step(12, graph=True)
    cut.step(1)
    cut.step(11)
    for a, b in zip(result(whole), result(cut)):
        np.testing.assert_array_equal(a, b)
