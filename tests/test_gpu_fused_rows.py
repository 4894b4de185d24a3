"""Forward fused levels with rows that are not 16-byte aligned (odd widths and
odd half widths, one sample past a tile, ragged rows and planes): archives
bitwise against the oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")]

from fields import field  # noqa: E402


@pytest.mark.parametrize("shape", [(80, 100, 129), (81, 97, 122), (79, 99, 191), (96, 96, 68)], ids=str)
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_unaligned_rows(oracle, shape, dtype):
    import waltz_amd
    from waltz_amd import stages
    tdt = torch.float32 if dtype == np.float32 else torch.float64
    assert oracle.geometry(*reversed(shape))[0] >= 2
    x = field(shape, "smooth", dtype) + field(shape, "noise", dtype, seed=5) / 16
    want = oracle.compress(x, 1e-3)
    try:
        stages.set_tuning(shape, tdt, False, 2, (32, 16, 16, 16, 16))
        got = waltz_amd.compress(torch.from_numpy(x).cuda(), abs_error=1e-3)
    finally:
        stages.clear_tuning()
    assert got.cpu().numpy().tobytes() == want
