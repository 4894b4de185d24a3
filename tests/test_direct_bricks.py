"""Thread <-> sub-block map of the fused (de)quantizing coders for z bands of a
power of two: on the CPU against the recursive octant rank, and on the GPU as
archives of such fields against the oracle (one band per schedule, a last chunk
that is partial, q-outliers)."""
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

from fields import field

HERE = Path(__file__).resolve().parent


@pytest.mark.parametrize("cxx", ["g++", "/opt/rocm/llvm/bin/clang++"])
def test_map(tmp_path, cxx):
    if shutil.which(cxx) is None and not Path(cxx).exists():
        pytest.skip(cxx + " not available")
    exe = tmp_path / "direct"
    subprocess.run([cxx, "-O2", "-std=c++17", str(HERE / "test_direct_bricks_host.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout + out.stderr


# (z, y, x), z band
@pytest.mark.gpu
@pytest.mark.parametrize("shape,band", [((16, 16, 48), 8), ((512, 144, 144), 16), ((32, 32, 32), 8), ((272, 32, 16), 2),
                                        ((12, 48, 80), 2), ((1, 48, 48), 1), ((2, 64, 80), 2)],
                         ids=str)
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_archives(oracle, shape, band, dtype):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import waltz_amd
    assert oracle.geometry(*reversed(shape))[3] == band
    # (a large field of outliers exceeds the format's side channels)
    x = field(shape, "outliers" if np.prod(shape) <= 1 << 20 else "smooth", dtype)
    for bound in (1.0, 1e-2):
        want = oracle.compress(x, bound)
        a = waltz_amd.compress(torch.from_numpy(x).cuda(), abs_error=bound)
        assert a.cpu().numpy().tobytes() == want
        got = waltz_amd.decompress(a, shape=shape, dtype=torch.from_numpy(x).dtype).cpu().numpy()
        assert np.array_equal(got.view(np.uint8), oracle.decompress(want, shape, dtype).view(np.uint8))
