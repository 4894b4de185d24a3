"""Gradients near the ends of the type's range. Scaling by a power of two is
exact in every lifting step, so the adjoint of a gradient whose own lifting
stays inside the type's range is the scaled adjoint of a small one, bit for bit:
nothing on the way may overflow that the lifting itself does not. How large the
lifting gets on the way is followed in 64 bits, step by step; neighbours are
added before they are multiplied, so half the range is left for that sum."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")]

A, B, G, D, K = -1.586134342059924, -0.052980118572961, 0.882911075530934, 0.443506852043971, 1.1496043988602418

# (shape z,y,x), levels_xy, levels_z, dyadic: lines of 2 to 8 samples, odd and
# even, one strip and two, both schedules, coarse planes in one launch
CASES = [((20, 17, 12), 1, 1, True), ((33, 40, 129), 2, 2, True), ((2, 3, 250), 1, 1, True), ((3, 2, 2), 1, 1, False),
         ((4, 5, 6), 2, 1, False), ((100, 130, 64), 4, 3, False), ((7, 60, 61), 3, 0, False), ((30, 9, 9), 0, 2, False)]


def _line(v, dim, inverse, seen):
    """One transposed 1-D pass of `v` (natural -> split of the inverse, else split
    -> natural), every value on the way into `seen`."""
    n = v.shape[dim]
    order = torch.cat([torch.arange(0, n, 2), torch.arange(1, n, 2)])
    even, odd = order[:n - n // 2], order[n - n // 2:]
    if not inverse:
        v = torch.empty_like(v).index_copy_(dim, order, v)
    view = [1] * v.dim()
    view[dim] = n
    scale = torch.ones(n, dtype=v.dtype)
    scale[even], scale[odd] = (1 / K, -K) if inverse else (K, -1 / K)
    if not inverse:
        v = v * scale.view(view)
    seen.append(v.abs().max())
    # a step adds c times both mirrored neighbours to the samples `to`; its
    # transpose adds c times those samples to the places they were read from
    steps = [(-A, odd), (-B, even), (-G, odd), (-D, even)] if inverse else [(D, even), (G, odd), (B, even), (A, odd)]
    for c, to in steps:
        add = c * v.index_select(dim, to)
        for side in (to - 1, to + 1):
            at = side.abs()
            at = torch.where(at >= n, 2 * (n - 1) - at, at)
            v = v.index_add(dim, at, add)
        seen.append(v.abs().max())
    if inverse:
        v = (v * scale.view(view)).index_select(dim, order)
    seen.append(v.abs().max())
    return v


def _peak(v, lxy, lz, dyadic, inverse):
    """The largest value on the way of the adjoint of `v`."""
    levels = [(0, 1, 2)] * lxy if dyadic else [(0,)] * lz + [(1, 2)] * lxy
    box, boxes = list(v.shape), []
    for i, axes in enumerate(levels):
        if i and axes != levels[i - 1]:
            box = list(v.shape)
        # finest first; passes in the order of the transposed inverse
        boxes.append((tuple(box), [1, 2, 0] if len(axes) == 3 else [0] if axes == (0,) else [1, 2]))
        box = [m - m // 2 if a in axes else m for a, m in enumerate(box)]
    seen = [v.abs().max()]
    for (nz, ny, nx), axes in boxes if inverse else reversed(boxes):
        part = v[:nz, :ny, :nx]
        for dim in axes if inverse else reversed(axes):
            part = _line(part, dim, inverse, seen)
        v = v.clone()
        v[:nz, :ny, :nx] = part
    return float(max(seen))


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[0])) + f"_l{c[1]}{c[2]}")
@pytest.mark.parametrize("inverse", [False, True], ids=["dwt", "idwt"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
def test_large_gradients(case, inverse, dtype):
    from waltz_amd import stages
    shape, lxy, lz, dyadic = case
    top, down = torch.finfo(dtype).max, 2.0 ** -32
    places = [tuple(0 for _ in shape), tuple(s - 1 for s in shape), (0, shape[1] - 1, shape[2] // 2),
              (shape[0] - 1, 0, 0), (0, shape[1] // 2, shape[2] - 1), tuple(s // 2 for s in shape)]
    for place in places:
        unit = torch.zeros(shape, dtype=torch.float64)
        unit[place] = 1.0
        value = 0.45 * top / _peak(unit, lxy, lz, dyadic, inverse)
        small = torch.zeros(shape, dtype=dtype, device="cuda")
        small[place] = value * down
        want = stages.transform_adjoint(small, lxy, lz, dyadic, of_inverse=inverse) / down
        got = stages.transform_adjoint(small / down, lxy, lz, dyadic, of_inverse=inverse)
        assert torch.isfinite(got).all(), place
        assert torch.equal(got, want), place
