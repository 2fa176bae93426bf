"""The screening pass at the edges of its split: fewer entries than a wave or
than the dies share out, the smallest and largest launches, waves whose
entries belong to several sims.  It settles no pair that the complete pass
finds in contact and leaves out none, so two passes equal one bit for bit."""
import numpy as np
import pytest

from grains3dgpu_amd import _abi as A
from grains3dgpu_amd import scene as S
from tests.scenes import dense_cylinders_cones, dense_spheres, dense_superquadrics, lattice_superquadrics

pytestmark = pytest.mark.gpu

SCENES = {
    "pairs": lambda: dense_superquadrics(n=40, seed=31, phi=0.2, vel=0.5),
    "bed": lambda: dense_superquadrics(n=500, seed=32, phi=0.25, vel=0.5),
    "cylinders": lambda: dense_cylinders_cones(n=300, seed=33, vel=0.5),
    "sims": lambda: S.config3(n_sims=20, n_range=(200, 400), seed=34, phi=0.2),
}


@pytest.mark.parametrize("block,per_cu", [(64, 1), (256, 8), (128, 64)])
@pytest.mark.parametrize("which", sorted(SCENES))
def test_screen_settles_what_one_pass_does(which, block, per_cu):
    from grains3dgpu_amd import engine
    sc = SCENES[which]()
    out = []
    for passes in (1, 2):
        e = S.load(engine.Engine(dt=sc.dt, precision=A.FP64, gjk_rel_tol=1e-8, narrow_passes=passes, block_size=block,
                                 narrow_blocks_per_cu=per_cu), sc)
        e.step(5)
        out.append((e.get_state(), e.get_stats(), e.get_pairs(A.PAIRS_CONTACT)))
    one, two = out
    for a, b in zip(one[0], two[0]):
        np.testing.assert_array_equal(a, b)
    np.testing.assert_array_equal(one[2], two[2])
    for k in ("candidate_pairs", "gjk_calls", "contacts"):
        assert one[1][k] == two[1][k], k
    assert two[1]["candidate_pairs"] > 0


@pytest.mark.parametrize("block,per_cu", [(64, 1), (256, 8)])
@pytest.mark.parametrize("which", sorted(SCENES))
def test_reference_semantics_in_two_passes(which, block, per_cu):
    """REF_QUIRKS in FP64: the screen settles by spheres and OBB what one pass
    does; the rest are searched by two lanes each, with the same results."""
    from grains3dgpu_amd import engine
    sc = SCENES[which]()
    out = []
    for passes in (1, 2):
        e = S.load(engine.Engine(dt=sc.dt, precision=A.FP64, flags=A.REF_QUIRKS, narrow_passes=passes,
                                 block_size=block, narrow_blocks_per_cu=per_cu), sc)
        e.step(5)
        out.append((e.get_state(), e.get_stats(), e.get_pairs(A.PAIRS_CONTACT)))
    one, two = out
    for a, b in zip(one[0], two[0]):
        np.testing.assert_array_equal(a, b)
    np.testing.assert_array_equal(one[2], two[2])
    for k in ("candidate_pairs", "gjk_calls", "gjk_iterations", "contacts"):
        assert one[1][k] == two[1][k], k


@pytest.mark.parametrize("flags", [0, A.REF_QUIRKS])
@pytest.mark.parametrize("n", [2, 300, 17000])
def test_spheres_alone_equal_spheres_beside_a_box(n, flags):
    """A bed of spheres takes the pass without a search; one more particle, a
    box out of reach of all others, sends it through the general passes."""
    import dataclasses
    from grains3dgpu_amd import engine
    sc = dense_spheres(n=max(n, 300), seed=35, vel=0.5)
    if n < 300:
        sc = dataclasses.replace(sc, pos=sc.pos[:n], quat=sc.quat[:n], vel=sc.vel[:n], omega=sc.omega[:n],
                                 particle_shape=sc.particle_shape[:n])
    L = np.array(sc.sims[0]["domain_max"], float)
    sims = [dict(sc.sims[0], domain_max=tuple(L * [1, 1, 3]))]
    alone = dataclasses.replace(sc, sims=sims)
    box = [dict(kind=A.BOX, material=0, dims=(1e-4, 1e-4, 1e-4), density=2500.0)]
    beside = dataclasses.replace(
        sc, sims=sims, shapes=list(sc.shapes) + box, pos=np.r_[sc.pos, [L * [0.5, 0.5, 2.5]]],
        quat=np.r_[sc.quat, [[0, 0, 0, 1.0]]], vel=np.r_[sc.vel, [[0, 0, 0.0]]], omega=np.r_[sc.omega, [[0, 0, 0.0]]],
        particle_shape=np.r_[sc.particle_shape, len(sc.shapes)].astype(np.uint32))
    out = []
    for s in (alone, beside):
        e = S.load(engine.Engine(dt=s.dt, precision=A.FP64, flags=flags), s)
        e.step(8)
        out.append((e.get_state(), e.get_torce(), e.get_stats()["contacts"]))
    m = len(alone.pos)
    assert out[0][2] == out[1][2] and (n < 300 or out[0][2] > 0)
    for a, b in zip(out[0][0] + out[0][1], out[1][0] + out[1][1]):
        np.testing.assert_array_equal(a, b[:m])


@pytest.mark.parametrize("flags", [0, A.WARM_START | A.FP64_CONTACTS])
def test_complete_pass_by_one_lane_and_by_two(flags):
    """Launches whose lanes hold the queue (9,000 entries) twice over search
    each entry by two lanes, narrower ones by one: the same results."""
    from grains3dgpu_amd import engine
    sc = lattice_superquadrics(n_side=12, seed=36)
    out = []
    for block, per_cu in ((64, 1), (64, 8), (128, 2), (256, 8)):
        e = S.load(engine.Engine(dt=sc.dt, precision=A.FP32_MIXED, flags=flags, gjk_rel_tol=1e-6, block_size=block,
                                 narrow_blocks_per_cu=per_cu), sc)
        e.step(3)
        st = e.get_stats()
        assert 3 * 8192 < st["narrow_deferred"] < 3 * 16384
        out.append([*e.get_state(), e.get_pairs(A.PAIRS_CONTACT), np.array(st["contacts"])])
    for o in out[1:]:
        for a, b in zip(o, out[0]):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("block,per_cu", [(64, 1), (128, 2), (256, 8)])
def test_reference_semantics_in_one_packed_pass(block, per_cu):
    """REF_QUIRKS on a bed whose one pass packs its candidates from the lists
    (more than 10,000 grains), its waves taking shares of one to eight turns:
    FP64 equals two passes, FP32 itself in another launch and FP64's contacts."""
    from grains3dgpu_amd import engine
    sc = dense_superquadrics(n=11000, seed=37, phi=0.2, vel=0.5, box_frac=0.3)

    def run(precision, passes, **launch):
        e = S.load(engine.Engine(dt=sc.dt, precision=precision, flags=A.REF_QUIRKS, narrow_passes=passes, **launch), sc)
        e.step(3)
        st = e.get_stats()
        assert st["contacts"] > 0
        return [*e.get_state(), e.get_pairs(A.PAIRS_CONTACT),
                np.array([st[k] for k in ("candidate_pairs", "gjk_calls", "gjk_iterations", "contacts")])]

    launch = dict(block_size=block, narrow_blocks_per_cu=per_cu)
    for a, b in zip(run(A.FP64, 1, **launch), run(A.FP64, 2)):
        np.testing.assert_array_equal(a, b)
    one = run(A.FP32_MIXED, 1, **launch)
    for a, b in zip(one, run(A.FP32_MIXED, 1, block_size=64, narrow_blocks_per_cu=16)):
        np.testing.assert_array_equal(a, b)
