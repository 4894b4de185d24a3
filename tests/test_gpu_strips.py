"""The in-register X and Y lifting of a plane level: line lengths at the
limits of a lane group (8 to 64 lanes), of one strip and of a strip boundary,
rows at the limits of a y segment, and plane counts that leave a lane group
without a plane, bitwise against the oracle in both directions."""
import numpy as np
import pytest

from fields import field

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

WIDTHS = [2, 3, 8, 11, 12, 13, 16, 27, 28, 29, 32, 59, 60, 61, 64, 123, 124, 125, 126, 127, 128, 129, 130, 243, 244,
          245, 364, 365]
HEIGHTS = [2, 3, 7, 8, 9, 15, 16, 17, 33]


def check(oracle, shape, lxy, dtype):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from waltz_amd import stages
    x = field(shape, "noise", dtype) * 3 + field(shape, "smooth", dtype)
    c = stages.transform(torch.from_numpy(x).cuda(), lxy, 0, False, False).cpu().numpy()
    want = oracle.transform(x, lxy, 0, False, False)
    assert np.array_equal(c.view(np.uint8), want.view(np.uint8))
    back = stages.transform(torch.from_numpy(want).cuda(), lxy, 0, False, True).cpu().numpy()
    assert np.array_equal(back.view(np.uint8), oracle.transform(want, lxy, 0, False, True).view(np.uint8))


@pytest.mark.parametrize("nx", WIDTHS)
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_line_lengths(oracle, nx, dtype):
    check(oracle, (3, 40, nx), 1, dtype)


@pytest.mark.parametrize("ny", HEIGHTS)
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_line_counts(oracle, ny, dtype):
    check(oracle, (9, ny, 50), 1, dtype)


# several levels, one-sample lines on the way (the separate passes), 2-D fields
@pytest.mark.parametrize("shape,lxy", [((17, 70, 300), 5), ((1, 500, 260), 5), ((5, 3, 40), 3), ((2, 160, 26), 5),
                                       ((33, 150, 103), 5)], ids=str)
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_levels(oracle, shape, lxy, dtype):
    check(oracle, shape, lxy, dtype)


# one batch whose jobs take every schedule: columns too tall for one pass, no Z
# level, no XY level, several strips, dyadic boxes, odd extents
BATCH = [(400, 9, 20), (180, 10, 33), (1, 40, 50), (40, 5, 30), (20, 20, 300), (33, 17, 65), (40, 48, 56), (9, 9, 9)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_batch_schedules(oracle, dtype):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from waltz_amd import batch
    fields = [field(s, "smooth", dtype, seed=k + 1) for k, s in enumerate(BATCH)]
    dec = batch.BatchDecoder(BATCH, torch.float32 if dtype is np.float32 else torch.float64)
    arcs, spans = dec.compress(dec.flatten([torch.from_numpy(f).cuda() for f in fields]), 1e-2)
    tiles = dec.views(dec.decode(arcs, spans))
    for k, (f, (at, size)) in enumerate(zip(fields, spans.view(-1, 2).tolist())):
        want = oracle.compress(f, 1e-2)
        assert arcs[at:at + size].cpu().numpy().tobytes() == want, BATCH[k]
        got = tiles[k].cpu().numpy()
        assert np.array_equal(got.view(np.uint8), oracle.decompress(want, f.shape, dtype).view(np.uint8)), BATCH[k]
