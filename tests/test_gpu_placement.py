"""Payload placement: streams of one chunk, of a group and a chunk more or
less, of several groups, with empty chunks and whole empty groups among full
ones, bitwise against the oracle."""
import numpy as np
import pytest

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
