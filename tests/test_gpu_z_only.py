"""Transforms of Z levels only (planes of at most 8 rows or columns, or custom
levels): the whole phase is one column pass, also in place and from an input
that is kept, with the results of the oracle. 102 (double) and 204 (float)
planes are the most that fit LDS in place; above, the pass works on a copy. Up to
256 rows of columns take workgroups of 16 waves, more of 4, in place with over
48 KiB of 8."""
import numpy as np
import pytest

from fields import field

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("shape,lz", [((100, 8, 300), 4), ((64, 70, 8), 3), ((17, 40, 50), 2), ((20, 3, 130), 1),
                                      ((102, 8, 66), 5), ((103, 8, 66), 5), ((204, 8, 66), 5), ((205, 8, 66), 5),
                                      ((20, 256, 9), 2), ((40, 257, 9), 3), ((102, 129, 65), 5), ((160, 257, 9), 5)],
                         ids=str)
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_one_pass(oracle, shape, lz, dtype):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from waltz_amd import _lib, stages
    x = field(shape, "noise", dtype)
    for inverse in (False, True):
        want = torch.from_numpy(oracle.transform(x, 0, lz, False, inverse)).cuda()
        for inplace in (False, True):
            v = torch.from_numpy(x).cuda()
            _lib.profile(True)
            try:
                _lib.profile_report()
                out = stages.transform(v, 0, lz, False, inverse, out=v if inplace else None)
                torch.cuda.synchronize()
                names = set(_lib.profile_report())
            finally:
                _lib.profile(False)
            assert torch.equal(out, want)
            assert inplace or torch.equal(v, torch.from_numpy(x).cuda())
            if shape[0] <= (340 if dtype == np.float32 else 170):  # (else axis passes)
                assert names == {"inverse_Z" if inverse else "forward_Z"}
