"""Fields with edge bricks: groups of bricks per workgroup (one brick and
several, z bands of 1 to 16, bricks of one sample across), group spans that
share 16-byte and 32-bit words with their neighbours, q-outliers, and inverses
that quantize what they load (plane schedule; one and two fused dyadic levels):
archives and decodes bitwise against the oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")]

from fields import field  # noqa: E402


def check(oracle, shape, dtype, kind, bound):
    import waltz_amd
    x = field(shape, kind, dtype)
    want = oracle.compress(x, bound)
    a = waltz_amd.compress(torch.from_numpy(x).cuda(), abs_error=bound)
    assert a.cpu().numpy().tobytes() == want
    got = waltz_amd.decompress(a, shape=shape, dtype=torch.from_numpy(x).dtype).cpu().numpy()
    assert np.array_equal(got.view(np.uint8), oracle.decompress(want, shape, dtype).view(np.uint8))


@pytest.mark.parametrize("shape", [(1, 17, 33), (2, 50, 19), (11, 33, 47), (19, 33, 17), (36, 100, 52), (149, 35, 37),
                                   (9, 16, 17)], ids=str)
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_edges(oracle, shape, dtype):
    for kind, bound in (("smooth", 1e-3), ("outliers", 1e-2)):
        check(oracle, shape, dtype, kind, bound)


# (several bricks a workgroup: more than 2048 bricks)
@pytest.mark.parametrize("shape", [(40, 340, 500), (170, 300, 270)], ids=str)
def test_groups(oracle, shape):
    check(oracle, shape, np.float32, "smooth", 1e-3)


@pytest.mark.parametrize("fused", [1, 2])
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_requantizing_inverse(oracle, fused, dtype):
    from waltz_amd import stages
    shape, tdt = (81, 99, 122), torch.float32 if dtype == np.float32 else torch.float64
    try:
        stages.set_tuning(shape, tdt, True, fused, (32, 16, 16, 16, 16))
        for kind in ("smooth", "outliers"):
            check(oracle, shape, dtype, kind, 1e-2)
    finally:
        stages.clear_tuning()
