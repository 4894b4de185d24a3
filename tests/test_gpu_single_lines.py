"""Transforms of boxes with lines of one sample (custom levels), at the first
level and at a later one, along every axis and in both schedules, bitwise
against the oracle. Such a line is its own neighbour on both sides."""
import numpy as np
import pytest

from fields import field

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# (z, y, x), XY levels, Z levels, dyadic
CASES = [((1, 20, 12), 1, 1, True), ((2, 20, 12), 2, 2, True), ((8, 1, 40), 1, 1, True), ((9, 33, 1), 1, 1, True),
         ((1, 1, 1), 1, 1, True), ((3, 40, 300), 3, 3, True), ((1, 9, 70), 0, 1, False), ((1, 9, 70), 1, 2, False),
         ((2, 17, 33), 1, 2, False), ((9, 12, 40), 2, 5, False), ((33, 1, 17), 2, 1, False), ((12, 2, 30), 2, 1, False)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[0])) + f"_l{c[1]}{c[2]}")
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_bitwise(oracle, case, dtype):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from waltz_amd import stages
    shape, lxy, lz, dyadic = case
    x = field(shape, "noise", dtype) * 3 + 1
    for inverse in (False, True):
        want = oracle.transform(x, lxy, lz, dyadic, inverse)
        got = stages.transform(torch.from_numpy(x).cuda(), lxy, lz, dyadic, inverse).cpu().numpy()
        assert np.array_equal(got.view(np.uint8), want.view(np.uint8)), inverse
