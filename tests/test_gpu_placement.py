"""Payload placement: streams of one chunk, of a group and a chunk more or
less, of several groups, with empty chunks and whole empty groups among full
ones, bitwise against the oracle."""
import numpy as np
import pytest

from fields import field

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")]

CHUNK = 8192


@pytest.mark.parametrize("chunks", [1, 15, 16, 17, 33, 300])
@pytest.mark.parametrize("tail", [0, 1, 4097])
@pytest.mark.parametrize("empty", ["none", "some", "groups"])
def test_streams(oracle, chunks, tail, empty):
    from waltz_amd import stages
    n = chunks * CHUNK + tail
    rng = np.random.default_rng(chunks * 7 + tail)
    mag = (rng.integers(0, 400, n) * (rng.random(n) < 0.3)).astype(np.uint16)
    c = np.arange(n) // CHUNK
    if empty == "some":
        mag[c % 3 == 1] = 0
    elif empty == "groups":
        mag[c // 16 % 2 == 0] = 0
    flags = (mag != 0) & (rng.random(n) < 0.5)
    sign = np.packbits(np.pad(flags, (0, -n % 32)), bitorder="little").view(np.uint32)
    want = oracle.wzp_encode(mag, sign)
    got = stages.wzp_encode(torch.from_numpy(mag.view(np.int16)).cuda(), torch.from_numpy(sign.view(np.int32)).cuda())
    assert got.cpu().numpy().tobytes() == want


# repair segments (rows of 64 columns) at the limits of the number of
# workgroups that share one: eight, seven, two, one, more segments than
# workgroups, and five with more repairs in a segment than a workgroup has lanes
@pytest.mark.parametrize("shape", [(10, 512, 40), (10, 513, 40), (10, 2048, 40), (10, 2049, 40), (12, 2100, 80),
                                   (160, 700, 64)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_repairs_of_many_segments(oracle, shape, dtype):
    import waltz_amd
    lx, lz, dyadic, _ = oracle.geometry(*reversed(shape))
    assert lz and not dyadic
    x = field(shape, "noise", dtype) * 30 + field(shape, "checker", dtype)
    want = oracle.compress(x, 0.5)
    assert int.from_bytes(want[24:28], "little") > 256 * 8  # repairs
    got = waltz_amd.compress(torch.from_numpy(x).cuda(), abs_error=0.5).cpu().numpy().tobytes()
    assert got == want
