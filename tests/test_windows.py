"""Volumes past one 32-bit window: the rules that pick the addressing, on the
CPU against the offsets; and on the GPU a volume of 4.1 GiB, whose Z and XY
phases must equal those of its parts (slabs of rows, single planes) bit for bit."""
import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


@pytest.mark.parametrize("cxx", ["g++", "/opt/rocm/llvm/bin/clang++"])
def test_rules(tmp_path, cxx):
    if shutil.which(cxx) is None and not Path(cxx).exists():
        pytest.skip(cxx + " not available")
    exe = tmp_path / "windows"
    subprocess.run([cxx, "-O2", "-std=c++17", str(HERE / "test_windows_host.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout + out.stderr


# two Z levels of tiles that cross the window; the second case has planes of
# 275 MB, whose 16-plane tiles are past a window themselves
@pytest.mark.gpu
@pytest.mark.parametrize("shape,lz", [((99, 3300, 3370), 4), ((17, 4001, 17203), 2)], ids=str)
def test_phases_of_a_large_volume(shape, lz):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from waltz_amd import stages
    nz, ny, nx = shape
    assert 4 * nz * ny * nx > 1 << 32
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.rand(shape, device="cuda", generator=g) - 0.5
    slabs = [(0, 60), (ny // 2, 50), (ny - 40, 40)]  # rows: a Z line depends on nothing else

    def z_only(v, inverse):
        return stages.transform(v.contiguous(), 0, lz, False, inverse)

    def xy_only(v, inverse):
        return stages.transform(v.contiguous(), 5, 0, False, inverse)

    for inverse in (False, True):
        z = stages.transform(x, 0, lz, False, inverse)
        for at, rows in slabs:
            assert torch.equal(z[:, at:at + rows], z_only(x[:, at:at + rows], inverse))
        del z
        if not inverse:  # Z, then XY of every plane
            y = stages.transform(x, 5, lz, False, False)
            z = stages.transform(x, 0, lz, False, False)
            for k in (0, 1, nz // 2, nz - 2, nz - 1):
                assert torch.equal(y[k:k + 1], xy_only(z[k:k + 1], False))
        else:  # XY of every plane, then Z
            y = stages.transform(x, 5, lz, False, True)
            z = torch.cat([xy_only(x[k:k + 1], True) for k in range(nz)])
            for at, rows in slabs:
                assert torch.equal(y[:, at:at + rows], z_only(z[:, at:at + rows], True))
        del y, z
    # (in place as well)
    want = stages.transform(x, 5, lz, False, False)
    stages.transform(x, 5, lz, False, False, out=x)
    assert torch.equal(x, want)


# A plane past one window: out of place its forward levels run as strips with a
# window per row, in place as axis passes with 64-bit addresses.
@pytest.mark.gpu
@pytest.mark.parametrize("shape,dtype", [((1, 33001, 32603), "float32"), ((1, 16500, 32700), "float64")], ids=str)
def test_forward_of_a_large_plane(shape, dtype):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from waltz_amd import stages
    x = torch.rand(shape, device="cuda", dtype=getattr(torch, dtype), generator=torch.Generator("cuda").manual_seed(4))
    assert x.numel() * x.element_size() > 1 << 32
    want = stages.transform(x, 5, 0, False, False)
    stages.transform(x, 5, 0, False, False, out=x)
    assert torch.equal(x, want)
