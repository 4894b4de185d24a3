"""The adjoint levels in registers at the edges of their splits (one strip, two
strips, lines that share or fill a wave, y and z segments and the rows and
planes past them, lines of 2 and 3 samples, in place), and the passes that are
left for lines of one sample: <T c, y> = <c, T^T y> in float64, on vectors that
also weigh each end of every axis by itself."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")]

# (shape z,y,x), levels_xy, levels_z, dyadic
CASES = [((20, 17, 12), 1, 1, True), ((9, 129, 124), 1, 1, True), ((130, 33, 125), 2, 2, True),
         ((33, 16, 128), 1, 1, True), ((17, 130, 129), 3, 3, True), ((2, 3, 250), 1, 1, True),
         ((66, 20, 61), 0, 3, False), ((5, 40, 64), 2, 0, False), ((65, 35, 30), 2, 3, False),
         ((3, 2, 2), 1, 1, False), ((8, 1, 40), 1, 1, True)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[0])) + f"_l{c[1]}{c[2]}")
@pytest.mark.parametrize("inverse", [False, True], ids=["dwt", "idwt"])
def test_transpose(case, inverse):
    from waltz_amd import stages
    shape, lxy, lz, dyadic = case
    if inverse and min(shape) == 1:
        pytest.skip("adjoint_pass models an inverse line of one sample by its even half only")
    g = torch.Generator(device="cuda").manual_seed(11)

    def rand():
        return torch.randn(shape, dtype=torch.float64, device="cuda", generator=g)

    c = rand()
    tc = stages.transform(c, lxy, lz, dyadic, inverse=inverse)
    ys = [rand()]
    for axis in range(3):
        for end in (0, shape[axis] - 1):  # nothing but one end face
            y = torch.zeros(shape, dtype=torch.float64, device="cuda")
            y.select(axis, end).copy_(rand().select(axis, end))
            ys.append(y)
    for y in ys:
        ty = stages.transform_adjoint(y, lxy, lz, dyadic, of_inverse=inverse)
        lhs, rhs = float((tc * y).sum()), float((c * ty).sum())
        assert abs(lhs - rhs) <= 1e-12 * float(tc.norm() * y.norm())
    inplace = y.clone()
    stages.transform_adjoint(inplace, lxy, lz, dyadic, of_inverse=inverse, out=inplace)
    assert torch.equal(inplace, ty)
