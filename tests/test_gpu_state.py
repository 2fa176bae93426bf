"""grains_get_state returns every value that was set, at the edges of its
pinned buffers and of its threads' parts, and leaves out what is not asked for."""
import ctypes as C

import numpy as np
import pytest

from grains3dgpu_amd import _abi as A
from grains3dgpu_amd import scene as S
from tests.scenes import dense_spheres

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 257, 16383, 16385, 262144, 262145, 600001])
def test_state_round_trip(n):
    from grains3dgpu_amd import engine
    rng = np.random.default_rng(n)
    sh = np.zeros(1, S.SHAPE_DTYPE)
    sh["kind"], sh["density"] = A.SPHERE, 2500.0
    sh["dims"][0, 0] = 1e-3
    want = [rng.standard_normal((n, k)) for k in (3, 4, 3, 3)]
    sc = S.Scene(shapes=sh, tables=np.array([S.hooke_row(1e5, 0.8, 0.0, 0.3)]), n_materials=1,
                 sims=[dict(domain_min=(0, 0, 0), domain_max=(1, 1, 1))], particle_shape=np.zeros(n, np.uint32),
                 pos=want[0], quat=want[1], vel=want[2], omega=want[3], dt=1e-6)
    e = S.load(engine.Engine(dt=sc.dt), sc)
    for _ in range(2):
        for a, b in zip(e.get_state(), want):
            np.testing.assert_array_equal(a, b)
    v = np.zeros((n, 3))
    assert e.L.grains_get_state(e.h, None, None, A.dptr(v), None, C.c_uint64(n)) == 0
    np.testing.assert_array_equal(v, want[2])


def test_state_read_while_another_gpu_is_current():
    """A context's state is read whichever GPU the thread has set."""
    from grains3dgpu_amd import engine
    engine.lib()
    h = C.CDLL("libamdhip64.so.7")
    count = C.c_int()
    if h.hipGetDeviceCount(C.byref(count)) or count.value < 2:
        pytest.skip("needs two GPUs")
    sc = dense_spheres(n=500, seed=1)
    e = S.load(engine.Engine(dt=sc.dt), sc)
    assert h.hipSetDevice(1) == 0
    try:
        for a, b in zip(e.get_state(), (sc.pos, sc.quat, sc.vel, sc.omega)):
            np.testing.assert_array_equal(a, b)
    finally:
        h.hipSetDevice(0)
