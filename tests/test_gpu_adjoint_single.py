"""Adjoints of lines of one sample (custom levels only): such a line is read as
every even and every odd sample of its extension, so both count in the
transpose. <T c, y> = <c, T^T y> in float64."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")]

# (shape z,y,x), levels_xy, levels_z, dyadic: one sample along x, y, z, at the
# first level and (from 2 samples) at a later one
CASES = [((8, 1, 40), 1, 1, True), ((8, 40, 1), 1, 1, True), ((1, 20, 12), 1, 1, True), ((2, 20, 12), 2, 2, True),
         ((1, 9, 70), 0, 1, False), ((33, 1, 17), 2, 1, False), ((5, 2, 30), 2, 0, False), ((1, 1, 1), 1, 1, True)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[0])) + f"_l{c[1]}{c[2]}")
@pytest.mark.parametrize("inverse", [False, True], ids=["dwt", "idwt"])
def test_transpose(case, inverse):
    from waltz_amd import stages
    shape, lxy, lz, dyadic = case
    g = torch.Generator(device="cuda").manual_seed(12)
    c, y = (torch.randn(shape, dtype=torch.float64, device="cuda", generator=g) for _ in range(2))
    tc = stages.transform(c, lxy, lz, dyadic, inverse=inverse)
    ty = stages.transform_adjoint(y, lxy, lz, dyadic, of_inverse=inverse)
    assert abs(float((tc * y).sum()) - float((c * ty).sum())) <= 1e-12 * float(tc.norm() * y.norm())
