"""The plane schedule's Z phase (one pass over rows of 64 columns): column
lengths at the tile, mirror and LDS limits, and row widths that leave partial
column blocks, bitwise against the oracle in both directions."""
import numpy as np
import pytest

from fields import field

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# (z, y, x), XY levels, Z levels: lines from 2 samples; 340/341 (float) and
# 170/171 (double) straddle the LDS limit
CASES = [
    ((2, 9, 65), 1, 1), ((5, 9, 63), 1, 2), ((8, 10, 64), 1, 3), ((9, 12, 1), 0, 1), ((16, 9, 70), 1, 2),
    ((17, 9, 129), 2, 3), ((25, 33, 40), 1, 5), ((31, 9, 66), 1, 4), ((33, 10, 20), 1, 5), ((100, 9, 68), 1, 4),
    ((169, 9, 33), 1, 5), ((170, 9, 33), 1, 5), ((171, 9, 33), 1, 5), ((172, 9, 33), 1, 5), ((340, 9, 10), 1, 5),
    ((341, 9, 10), 1, 5), ((342, 9, 10), 1, 5), ((343, 9, 10), 1, 5),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[0])) + f"_l{c[1]}{c[2]}")
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_column_pass_bitwise(oracle, case, dtype):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from waltz_amd import stages
    shape, lxy, lz = case
    x = field(shape, "noise", dtype) * 3 + field(shape, "smooth", dtype)
    c = stages.transform(torch.from_numpy(x).cuda(), lxy, lz, False, False).cpu().numpy()
    want = oracle.transform(x, lxy, lz, False, False)
    assert np.array_equal(c.view(np.uint8), want.view(np.uint8))
    back = stages.transform(torch.from_numpy(want).cuda(), lxy, lz, False, True).cpu().numpy()
    assert np.array_equal(back.view(np.uint8), oracle.transform(want, lxy, lz, False, True).view(np.uint8))


# rows whose flag words are shared with their neighbours (x not a multiple of
# 32), partial column blocks, one Z level and several, few and many repairs
@pytest.mark.parametrize("shape", [(9, 40, 33), (10, 17, 65), (12, 33, 20), (17, 70, 96), (33, 150, 130),
                                   (80, 160, 64), (100, 300, 18)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("bound", [0.5, 2e-4])
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_repairs_of_the_column_pass(oracle, shape, bound, dtype):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import waltz_amd
    nx, ny, nz = reversed(shape)
    lx, lz, dyadic, _ = oracle.geometry(nx, ny, nz)
    assert lz and not dyadic
    x = field(shape, "noise", dtype) * 30 + field(shape, "checker", dtype)
    want = oracle.compress(x, bound)
    assert int.from_bytes(want[24:28], "little") > 0  # repairs
    got = waltz_amd.compress(torch.from_numpy(x).cuda(), abs_error=bound).cpu().numpy().tobytes()
    assert got == want
