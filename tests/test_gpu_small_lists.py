"""Side lists of small fields (placed with the payloads by a workgroup per chunk
of the stream): streams of 1, 2, 15 and 16 chunks, fewer and more record
segments than waves, many q-outliers and many repairs, bitwise against the
oracle; and an archive buffer that is too small at each section."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")]

SHAPES = [(9, 9, 9), (16, 16, 32), (16, 16, 33), (17, 20, 24), (32, 64, 64), (31, 65, 65), (17, 800, 9), (1, 256, 480),
          (4, 181, 181)]


def spikes(shape, dtype):
    rng = np.random.default_rng(9)
    v = rng.standard_normal(shape)
    return (v + (rng.random(shape) < 0.05) * 1e6).astype(dtype)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_bytes(oracle, shape, dtype):
    import waltz_amd
    x = spikes(shape, dtype)
    assert x.size <= 1 << 17
    for bound in (0.5, 0.01 if dtype == np.float64 else 0.25):
        want = oracle.compress(x, bound)
        assert int.from_bytes(want[24:28], "little") or int.from_bytes(want[28:32], "little")  # repairs or q-outliers
        got = waltz_amd.compress(torch.from_numpy(x).cuda(), abs_error=bound).cpu().numpy().tobytes()
        assert got == want


@pytest.mark.parametrize("shape", [(9, 9, 9), (17, 20, 24), (31, 65, 65)], ids=lambda s: "x".join(map(str, s)))
def test_capacity(oracle, shape):
    from waltz_amd import _lib
    x = spikes(shape, np.float32)
    want = oracle.compress(x, 0.5)
    dev, need = torch.from_numpy(x).cuda(), len(want)
    nz, ny, nx = shape
    for size in (need, need - 1, 3 * need // 4, need // 2, need // 8, 4 + 32 + 3 * -(-x.size // 8192)):
        out = torch.full((need + 4096,), 0xA5, dtype=torch.uint8, device="cuda")
        written = C.c_size_t()
        rc = _lib.lib().waltz_amd_compress(4, dev.data_ptr(), nx, ny, nz, 0.5, out.data_ptr(), size, C.byref(written),
                                           None)
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        assert (got[size:] == 0xA5).all(), size
        if size == need:
            assert rc == 0 and got[:need].tobytes() == want
        else:
            assert rc != 0 and "capacity" in _lib.lib().waltz_amd_last_error().decode(), size
