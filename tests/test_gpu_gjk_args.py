"""The GJK batch with a shape set small enough for the kernel's arguments
equals the one that reads its tables from memory (one shape more than fits):
at the edges of a wave and of the rule, both precisions and semantics."""
import numpy as np
import pytest

from grains3dgpu_amd import _abi as A
from grains3dgpu_amd import scene as S
from tests.test_zz_no_alloc import _Dev, _pairs, _run

pytestmark = pytest.mark.gpu


def _scene(rng, n_shapes):
    sh = np.zeros(n_shapes, S.SHAPE_DTYPE)
    sh["kind"] = A.SUPERQUADRIC
    sh["dims"] = S.superquadric_params(rng, n_shapes)
    sh["kind"][0] = A.SPHERE
    sh["dims"][0, 0] = 7e-4
    sh["kind"][1] = A.BOX
    sh["dims"][1, :3] = (6e-4, 4e-4, 5e-4)
    sh["density"] = 2500.0
    return S.Scene(shapes=sh, tables=np.array([S.hooke_row(1e5, 0.8, 0.0, 0.3)]), n_materials=1,
                   sims=[dict(domain_min=(0, 0, 0), domain_max=(1, 1, 1))],
                   particle_shape=np.zeros(1, np.uint32), pos=np.zeros((1, 3)),
                   quat=np.array([[0, 0, 0, 1.0]]), vel=np.zeros((1, 3)), omega=np.zeros((1, 3)))


@pytest.mark.parametrize("flags", [0, A.REF_QUIRKS])
@pytest.mark.parametrize("precision", [A.FP64, A.FP32_MIXED], ids=["fp64", "fp32"])
@pytest.mark.parametrize("n", [1, 63, 65, 3000])
def test_shapes_in_arguments_equal_shapes_in_memory(n, precision, flags):
    from grains3dgpu_amd import engine
    rng = np.random.default_rng(n)
    sc = _scene(rng, 9)
    pairs = _pairs(rng, n, 8)  # the ninth shape, which the small set leaves out, is in no pair
    few = S.Scene(**{**sc.__dict__, "shapes": sc.shapes[:8]})
    dev = _Dev()
    out = []
    for s in (few, sc):
        e = engine.Engine(precision=precision, flags=flags, gjk_rel_tol=1e-10 if precision == A.FP64 else 1e-6)
        e.set_shapes(s)
        for fn in (e.L.grains_gjk_batch_device, e.L.grains_gjk_batch_device_noalloc):
            out.append(_run(e, dev, fn, *pairs)[:2])
    for a, b in ((0, 1), (2, 3)):  # both entry points, the same shape set
        np.testing.assert_array_equal(out[a][0], out[b][0])
        np.testing.assert_array_equal(out[a][1], out[b][1])
    if precision == A.FP64:
        np.testing.assert_array_equal(out[0][0], out[2][0])
        np.testing.assert_array_equal(out[0][1], out[2][1])
    else:
        # one arithmetic, contracted per kernel: the FP32 tolerance of the distances
        np.testing.assert_allclose(out[0][0], out[2][0], rtol=0, atol=1e-5 * 2e-3)


@pytest.mark.parametrize("n_shapes", [8, 9])
def test_batch_comes_after_the_default_stream(n_shapes):
    """Poses that copies on the default stream are still to bring: the call
    sees them, with the shapes in its arguments (8) as with them in memory (9)."""
    import ctypes as C
    from grains3dgpu_amd import engine
    rng = np.random.default_rng(3)
    e = engine.Engine(precision=A.FP64, gjk_rel_tol=1e-10)
    e.set_shapes(_scene(rng, n_shapes))
    n = 5000
    sa, sb, ta, tb = _pairs(rng, n, 8)
    dev = _Dev()
    want = _run(e, dev, e.L.grains_gjk_batch_device, sa, sb, ta, tb)[0]
    p = [dev.put(a) for a in (sa, sb, ta, ta, tb, np.zeros(n), np.zeros(n, np.int32))]
    big = 1 << 30
    work = [C.c_void_p(), C.c_void_p()]
    for w in work:
        assert dev.h.hipMalloc(C.byref(w), big) == 0
        dev.bufs.append(w)
    copy = dev.h.hipMemcpyAsync
    copy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int, C.c_void_p]
    for _ in range(30):  # some 10 ms of work
        assert copy(work[0], work[1], big, 3, None) == 0  # device to device
    assert copy(p[3], p[4], tb.nbytes, 3, None) == 0      # b's poses, in the place of a's
    assert e.L.grains_gjk_batch_device(e.h, p[0], p[1], p[2], p[3], n, p[5], p[6], None) == 0
    got = dev.get(p[5], want)
    dev.free()
    np.testing.assert_array_equal(got, want)
