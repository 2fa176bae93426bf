"""The screening pass at the edges of its split: fewer entries than a wave or
than the dies share out, the smallest and largest launches, waves whose
entries belong to several sims.  It settles no pair that the complete pass
finds in contact and leaves out none, so two passes equal one bit for bit."""
import numpy as np
import pytest

from grains3dgpu_amd import _abi as A
from grains3dgpu_amd import scene as S
from tests.scenes import dense_cylinders_cones, dense_superquadrics

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
