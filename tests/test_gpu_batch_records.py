"""Repair records of a batched decode: few of many jobs (most jobs of a wave's 64
records without any), one job's, and more than one round of the grid's lanes
(2^19), each tile as the single-field decoder gives it, bit for bit."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")]

# tiles, share of the tiles that are noise (the others constant: no records)
CASES = {"sparse": ([(9, 10, 11)] * 700, 0.03), "dense": ([(9, 10, 11)] * 300 + [(20, 30, 40)] * 9, 1.0),
         "one": ([(40, 50, 60)], 1.0), "rounds": ([(64, 128, 128)] * 24, 1.0)}


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
def test_records(case, dtype):
    import waltz_amd
    from waltz_amd import batch
    tiles, share = CASES[case]
    g = torch.Generator(device="cuda").manual_seed(8)
    bound, archives, want, records = 0.5, [], [], 0
    for s in tiles:
        noise = float(torch.rand((), generator=g, device="cuda")) < share
        x = torch.randn(s, dtype=dtype, device="cuda", generator=g) if noise else torch.ones(s, dtype=dtype, device="cuda")
        archives.append(waltz_amd.compress(x, abs_error=bound).clone())
        records += int.from_bytes(archives[-1][24:28].cpu().numpy().tobytes(), "little")
        want.append(waltz_amd.decompress(archives[-1], shape=s, dtype=dtype).reshape(-1))
    assert records > (1 << 19 if case == "rounds" else 0)
    packed, spans = batch.pack(archives)
    got = batch.BatchDecoder(tiles, dtype).decode(packed, spans)
    assert torch.equal(got, torch.cat(want))
