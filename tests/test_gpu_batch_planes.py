"""Plane passes of small batches (the coarse XY levels of every plane by one
workgroup): planes of one to several strips and segments, odd lines, coarse levels
under strip levels, on both sides of the 512 planes up to which they run, with
another kind of job beside them (no plane passes then), bitwise against the
oracle; and into clipped frames with holes."""
import ctypes as C

import numpy as np
import pytest

from fields import field

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")]

BATCHES = [[(1, 64, 64)] * 3, [(1, 17, 17), (1, 63, 65), (1, 100, 30)], [(2, 17, 200)], [(12, 48, 48)] * 42,
           [(12, 48, 48)] * 43, [(64, 128, 128), (20, 130, 67)], [(3, 64, 64), (32, 32, 32)],
           [(3, 33, 18), (1, 9, 9)], [(5, 300, 290), (9, 40, 50)]]


@pytest.mark.parametrize("tiles", BATCHES, ids=lambda t: "x".join(map(str, t[0])) + f"_{len(t)}")
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_batches(oracle, tiles, dtype):
    from waltz_amd import batch
    fields = [field(s, ["smooth", "noise"][j % 2], dtype, seed=j + 1) for j, s in enumerate(tiles)]
    want = [oracle.compress(f, 1e-2) for f in fields]
    plan = batch.BatchDecoder(tiles, torch.from_numpy(fields[0]).dtype)
    flat = torch.cat([torch.from_numpy(f).reshape(-1) for f in fields]).cuda()
    archives, spans = plan.compress(flat, abs_error=1e-2)
    for (o, n), w in zip(spans.view(-1, 2).tolist(), want):
        assert archives[o:o + n].cpu().numpy().tobytes() == w
    packed, spans = batch.pack([torch.from_numpy(np.frombuffer(w, np.uint8).copy()).cuda() for w in want])
    got = plan.decode(packed, spans).cpu().numpy()
    exact = np.concatenate([oracle.decompress(w, s, dtype).reshape(-1) for w, s in zip(want, tiles)])
    assert np.array_equal(got.view(np.uint8), exact.view(np.uint8))


@pytest.mark.parametrize("tile", [(8, 40, 36), (12, 40, 36)], ids=str)  # no Z levels, one
@pytest.mark.parametrize("width", [4, 8])
def test_frames(oracle, tile, width):
    from waltz_amd._lib import BatchShape, lib
    dtype = np.float32 if width == 4 else np.float64
    (tz, ty, tx), (fz, fy, fx), samples, sides = tile, (20, 59, 50), 1, 2
    gz, gy, gx = -(-fz // tz), -(-fy // ty), -(-fx // tx)
    jobs = gx * gy * gz * samples * sides
    body, table, tiles = bytearray(), [], []
    for j in range(jobs):
        if j % 5 == 2:  # a hole
            table += [0, 0]
            tiles.append(np.full(tile, -7.0, dtype))
            continue
        raw = oracle.compress(field(tile, ["smooth", "noise"][j % 2], dtype, seed=j), 1e-2)
        tiles.append(oracle.decompress(raw, tile, dtype))
        table += [len(body), len(raw)]
        body += raw + bytes((-len(raw)) % 16)
    host = np.frombuffer(bytes(body) + np.array(table, dtype="<u8").tobytes(), np.uint8).copy()
    packed = torch.from_numpy(host).cuda()
    shape = BatchShape(tx, ty, tz, fx, fy, fz, samples, sides, width)
    scratch = torch.empty(lib().waltz_gpu_batch_scratch_bytes(C.byref(shape)), dtype=torch.uint8, device="cuda")
    out = torch.empty((sides, samples, fz, fy, fx), dtype=torch.float32 if width == 4 else torch.float64, device="cuda")
    err = lib().waltz_gpu_decode_batch(C.byref(shape), host.ctypes.data, packed.data_ptr(), packed.numel(),
                                       scratch.data_ptr(), scratch.numel(), out.data_ptr(), out.numel() * width, -7.0,
                                       torch.cuda.current_stream().cuda_stream)
    assert err is None, err
    want = np.empty(out.shape, dtype)
    for j, t in enumerate(tiles):
        ox, r = (j % gx) * tx, j // gx
        oy, r = (r % gy) * ty, r // gy
        oz, r = (r % gz) * tz, r // gz
        part = t[:min(tz, fz - oz), :min(ty, fy - oy), :min(tx, fx - ox)]
        want[r % sides, r // sides, oz:oz + part.shape[0], oy:oy + part.shape[1], ox:ox + part.shape[2]] = part
    assert np.array_equal(out.cpu().numpy().view(np.uint8), want.view(np.uint8))
