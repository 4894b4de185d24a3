"""Waltz on one MI355X: compress / decompress throughput of a 512^3 float32
field at REL 1e-3 (plus ABS 1e-4), byte identity against the reference CPU
codec, per-stage roofline, and the reference CPU codec timed on this host.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--size 512] [--no-cpu]

One step = one compress + one decompress of the resident field. Prints ONE
JSON line (value = compress GB/s, decimal GB, field bytes / wall time of the
synchronous API call; inputs already in HBM).
"""
import argparse
import json
import os
import statistics
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))
METRIC = "compress/decompress GB/s at 512³ fp32 REL 1e-3 (1 GPU, % HBM peak); batched vs plain"
HBM_PEAK = 8.0e12  # MI355X HBM3E, bytes/s


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--size", type=int, default=512)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--profile-only", action="store_true", help="few calls, for rocprofv3 runs")
    ap.add_argument("--no-extra", action="store_true", help="skip the batched and autograd legs")
    ap.add_argument("--batched-only", action="store_true", help="only the batched leg, for rocprofv3 runs")
    return ap.parse_args()


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def stage_alg_bytes(name, n, w, wzp_bytes, sizes, np_repairs, writeback, folded):
    """Algorithmic HBM bytes of one pipeline stage (minimum dataflow).

    writeback: what the quantizing encoder writes back of the dequantized
    coefficients: "all", "box" (the coarser levels' box, n/8 samples, when
    the finest inverse level requantizes its high bands on load) or "none"
    (the coarse levels requantize on load as well).
    folded: the decoder's finest inverse level applies the repair list."""
    if name == "inverse_L0_repairs":
        # coefficients (7 bands + the coarser box) and the original field read,
        # flag bitmap and repair records written
        return 2 * w * n + n / 8 + np_repairs * (4 + w)
    if name == "inverse_L0" and folded:
        return 2 * w * n + np_repairs * (4 + w)  # coefficients read, field written, repair list read
    if name == "patch_keys":
        return np_repairs * (4 + w)  # the repair list read
    if name == "coarse_requant":
        return 2 * w * sizes[2]  # the level-2 box read and written compact
    if name.startswith(("forward_L", "inverse_L")):
        lvl = int(name.split("_L")[1][0])
        nb = sizes[lvl]
        return 2 * w * nb  # read + write the level's box
    table = {
        "quantize": 2 * w * n + 2 * n + n / 8,      # read coeff, write dequant, mags, signs
        "wzp_encode": 2 * n + n / 8 + wzp_bytes,    # read mags+signs, write stream
        # read coeff, write the dequantized coefficients (all, or the coarser
        # levels' box) and the chunk payloads into their staging slots
        "quantize_encode": w * n + {"all": w * n, "box": w * n / 8, "none": 0}[writeback] + wzp_bytes,
        "wzp_pack": 2 * wzp_bytes,                   # payloads from the staging slots into the archive
        "repairs": 2 * w * n,                        # read reconstruction + original
        "wzp_decode": wzp_bytes + 2 * n + n / 8,    # read stream, write mags+signs
        "dequantize": 2 * n + n / 8 + w * n,         # read mags+signs, write coefficients
        "decode_dequantize": wzp_bytes + w * n,      # read stream, write coefficients
    }
    return table.get(name)


def batched_shapes():
    import numpy as np
    rng = np.random.default_rng(20261202 + 4)
    kinds = [(32, 32, 32), (32, 64, 64), (48, 64, 96), (64, 128, 128)]  # (z, y, x)
    return [kinds[k] for k in rng.integers(0, len(kinds), 256)]


def batched_leg(torch, waltz_amd, synthetic, single_field_decompress_gbps, single_field_compress_gbps):
    """256 float32 chunks of uneven shape (seeded mix of 32^3, 64x64x32,
    96x64x48, 128x128x64; each its own k^-5/3 field), ABS 1e-3: decoded one
    archive per call through the plain API, then in one batched pass (eager
    and replayed as a captured graph) straight into one contiguous tensor."""
    from waltz_amd import batch
    shapes = batched_shapes()
    archives, fields = [], []
    for j, s in enumerate(shapes):
        f = synthetic.grf(s, slope=-5.0 / 3.0, seed=20261202 + 4 + 1000 * (j + 1))
        fields.append(f)
        archives.append(waltz_amd.compress(f, abs_error=1e-3).clone())
    packed, spans = batch.pack(archives)
    dec = batch.BatchDecoder(shapes, torch.float32)
    out_plain = torch.empty(dec.numel, dtype=torch.float32, device="cuda")
    views = dec.views(out_plain)

    def plain():
        for a, s, v in zip(archives, shapes, views):
            waltz_amd.decompress(a, shape=s, dtype=torch.float32, out=v)

    out_batch = torch.empty_like(out_plain)
    plain()
    dec.decode(packed, spans, out=out_batch)
    identical = bool(torch.equal(out_plain, out_batch))
    graph = torch.cuda.CUDAGraph()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            dec.decode(packed, spans, out=out_batch, check=False)
    torch.cuda.current_stream().wait_stream(stream)

    def timed(fn, reps):
        ts = []
        for _ in range(reps):
            torch.cuda.synchronize()
            t = time.perf_counter()
            fn()
            torch.cuda.synchronize()
            ts.append(time.perf_counter() - t)
        return statistics.median(ts)

    t_plain = timed(plain, 3)
    t_batch = timed(lambda: dec.decode(packed, spans, out=out_batch), 5)
    t_graph = timed(graph.replay, 5)
    dec.check()
    identical = identical and bool(torch.equal(out_plain, out_batch))
    nbytes = dec.numel * 4
    g_batch, g_graph, g_plain = nbytes / t_batch / 1e9, nbytes / t_graph / 1e9, nbytes / t_plain / 1e9

    # compress: one call per chunk, one batched call, the batched call replayed as a graph
    flat = dec.flatten(fields)

    def plain_c():
        for f in fields:
            waltz_amd.compress(f, abs_error=1e-3)

    barch, bspans = dec.compress(flat, abs_error=1e-3)
    same = all(bool(torch.equal(barch[int(o):int(o) + int(n)], a))
               for (o, n), a in zip(bspans.view(-1, 2).tolist(), archives))
    cgraph = torch.cuda.CUDAGraph()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        with torch.cuda.graph(cgraph, stream=stream):
            dec.compress(flat, abs_error=1e-3, archives=barch, spans=bspans, check=False)
    torch.cuda.current_stream().wait_stream(stream)
    tc_plain = timed(plain_c, 2)
    tc_batch = timed(lambda: dec.compress(flat, abs_error=1e-3, archives=barch, spans=bspans), 5)
    tc_graph = timed(cgraph.replay, 5)
    dec.compress_check()
    c_batch, c_graph, c_plain = nbytes / tc_batch / 1e9, nbytes / tc_graph / 1e9, nbytes / tc_plain / 1e9
    return {"chunks": len(shapes), "samples": dec.numel, "archive_bytes": int(packed.numel()),
            "bound": "ABS 1e-3",
            "per_chunk_calls_GBps": round(g_plain, 2), "batched_GBps": round(g_batch, 2),
            "graph_replay_GBps": round(g_graph, 2), "batched_over_per_chunk": round(g_batch / g_plain, 2),
            "graph_over_per_chunk": round(g_graph / g_plain, 2),
            "single_field_decompress_GBps_same_bound": round(single_field_decompress_gbps, 2),
            "graph_over_single_field_decompress": round(g_graph / single_field_decompress_gbps, 3),
            "bit_identical_to_per_chunk_decode": identical,
            "compress": {"per_chunk_calls_GBps": round(c_plain, 2), "batched_GBps": round(c_batch, 2),
                         "graph_replay_GBps": round(c_graph, 2),
                         "single_field_compress_GBps_same_bound": round(single_field_compress_gbps, 2),
                         "graph_over_single_field_compress": round(c_graph / single_field_compress_gbps, 3),
                         "archives_identical_to_per_chunk_compress": same}}, [f.cpu().numpy() for f in fields]


def autograd_leg(torch, waltz_amd, synthetic):
    """Batch of 8 256^3 float32 k^-5/3 fields at REL 1e-3: loss =
    MSE(IDWT(dequant(q)), field + N(0, 0.05^2)), backward to the coefficients
    through the adjoint; timed beside the plain decode of the same archives."""
    from waltz_amd import autograd, stages
    shape = (256, 256, 256)
    lxy, lz, dyadic = autograd.default_levels(shape)
    items = []
    for b in range(8):
        f = synthetic.grf(shape, slope=-5.0 / 3.0, seed=20261202 + 5 + 1000 * (b + 1))
        bound = 1e-3 * (float(f.max()) - float(f.min()))
        archive = waltz_amd.compress(f, abs_error=bound).clone()
        quantum = 1.5 * bound
        bz = int(archive[3])
        coeff = stages.quantize(stages.transform(f, lxy, lz, dyadic, inverse=False), bz, quantum)[0]
        g = torch.Generator(device="cuda").manual_seed(20261202 + 5 + b)
        target = f + 0.05 * torch.randn(shape, generator=g, device="cuda")
        items.append((archive, coeff, target))

    def step():
        total = 0.0
        for _, coeff, target in items:
            c = coeff.detach().requires_grad_()
            loss = torch.nn.functional.mse_loss(autograd.idwt(c, (lxy, lz, dyadic)), target)
            loss.backward()
            total += float(loss.detach())
        return total

    def decode():
        for archive, _, _ in items:
            waltz_amd.decompress(archive, shape=shape, dtype=torch.float32)

    step()
    decode()
    ts, td = [], []
    for _ in range(3):
        torch.cuda.synchronize()
        t = time.perf_counter()
        step()
        torch.cuda.synchronize()
        ts.append(time.perf_counter() - t)
        t = time.perf_counter()
        decode()
        torch.cuda.synchronize()
        td.append(time.perf_counter() - t)
    nbytes = 8 * 256 ** 3 * 4
    t_step, t_dec = statistics.median(ts), statistics.median(td)
    return {"batch": 8, "shape_zyx": list(shape), "forward_backward_ms": round(t_step * 1e3, 3),
            "forward_backward_GBps": round(nbytes / t_step / 1e9, 2), "plain_decode_ms": round(t_dec * 1e3, 3),
            "forward_backward_over_plain_decode": round(t_dec / t_step, 3)}


def cpu_batched_all_cores(pyoracle, fields):
    """The batched workload's 256 chunks through the reference CPU codec
    (AVX2 backend) on every host core: independent chunks over a thread pool,
    one codec workspace per thread (a workspace is not shareable)."""
    import threading
    from concurrent.futures import ThreadPoolExecutor
    threads = max(1, min(16, len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else os.cpu_count()))
    local = threading.local()

    def codec():
        if not hasattr(local, "ref"):
            local.ref = pyoracle.Reference()
        return local.ref

    def comp(f):
        r = codec()
        return r.compress(f, 1e-3, r.AVX2 if r.has_avx2 else r.SCALAR)

    def decomp(args):
        a, f = args
        r = codec()
        return r.decompress(a, f.shape, f.dtype, r.AVX2 if r.has_avx2 else r.SCALAR)

    nbytes = sum(f.nbytes for f in fields)
    with ThreadPoolExecutor(threads) as ex:
        list(ex.map(comp, fields[:threads]))  # one workspace per thread, warm
        t = time.perf_counter()
        archives = list(ex.map(comp, fields))
        tc = time.perf_counter() - t
        t = time.perf_counter()
        list(ex.map(decomp, zip(archives, fields)))
        td = time.perf_counter() - t
    return {"threads": threads, "compress_GBps": round(nbytes / tc / 1e9, 3),
            "decompress_GBps": round(nbytes / td / 1e9, 3),
            "sample": "the 256 chunks of the batched workload, ABS 1e-3, reference CPU codec, one pass"}


TRAFFIC_FILE = ROOT / "profiles" / "codec_512cube_f32_rel1e-3_traffic.md"
KERNELS_FILE = ROOT / "profiles" / "codec_512cube_f32_rel1e-3_kernels.md"
# the kernel each timed stage launches (as rocprofv3 names it)
STAGE_KERNEL = {
    "inverse_L0_repairs": "wz::inv_level_kernel<float, 2, true, true, false>",
    "inverse_L0": "wz::inv_level_kernel<float, 1, false, true, true>",
    "forward_L0": "wz::fwd_level_kernel<float>",
    "decode_dequantize": "wz::wzp_decode_direct_planned_kernel<float, true>",
    "quantize_encode": "wz::wzp_encode_kernel<wz::BrickSource<float, true> >",
}


def rocprof_duration_ms(stage):
    """Median duration (ms) of a stage's kernel in the committed rocprofv3
    kernel table (largest entry of that kernel: the finest level), or None."""
    name = STAGE_KERNEL.get(stage)
    best = None
    try:
        for line in KERNELS_FILE.read_text().splitlines():
            cells = [c.strip() for c in line.strip().strip("|").split("|")]
            if len(cells) == 4 and cells[1] == f"`{name}`":
                us = float(cells[3])
                best = us if best is None else max(best, us)
    except (OSError, ValueError):
        return None
    return None if best is None else best / 1e3


def flush_caches(torch, dev):
    """Evict L2 and the Infinity Cache: write 1 GiB that the codec never reads."""
    buf = torch.empty(256 << 20, dtype=torch.float32, device=dev)
    buf.fill_(1.0)
    torch.cuda.synchronize()
    del buf


def extra_config(torch, waltz_amd, field, rel, label, ref_cpu):
    """Compress / decompress GB/s of one more workload at a REL bound, its %
    of HBM peak on the algorithmic-bytes model and byte identity with the
    reference CPU codec (when it is built)."""
    import numpy as np
    from waltz_amd import autograd, stages as stage_api
    shape = tuple(field.shape)
    n = field.numel()
    w = field.element_size()
    lo, hi = float(field.min()), float(field.max())
    bound = rel * (hi - lo)
    stage_api.autotune(shape, field.dtype)
    archive = waltz_amd.compress(field, abs_error=bound)
    out = waltz_amd.decompress(archive, shape=shape, dtype=field.dtype)
    tc, td = [], []
    for _ in range(5):
        torch.cuda.synchronize()
        a = time.perf_counter()
        archive = waltz_amd.compress(field, abs_error=bound)
        b = time.perf_counter()
        waltz_amd.decompress(archive, shape=shape, dtype=field.dtype, out=out)
        c = time.perf_counter()
        tc.append(b - a)
        td.append(c - b)
    err = float((out.double() - field.double()).abs().max())
    A = archive.numel()
    lxy, lz, dyadic = autograd.default_levels(shape)
    if dyadic:
        coarse = sum(8.0 ** -l for l in range(1, lxy))
    else:
        coarse = 1 + sum(2.0 ** -l for l in range(1, lz)) + sum(4.0 ** -l for l in range(1, lxy))
    alg_c = (4 * w + 4.25) * n + 4 * w * n * coarse + A
    alg_d = 3 * w * n + 2 * w * n * coarse + A
    t_c, t_d = statistics.median(tc), statistics.median(td)
    res = {"workload": label, "shape_zyx": list(shape), "dtype": str(field.dtype).replace("torch.", ""),
           "levels": [lxy, lz, "dyadic" if dyadic else "plane"], "abs_bound": bound,
           "compress_GBps": round(n * w / t_c / 1e9, 2), "decompress_GBps": round(n * w / t_d / 1e9, 2),
           "compress_pct_hbm_alg": round(100 * alg_c / t_c / HBM_PEAK, 2),
           "decompress_pct_hbm_alg": round(100 * alg_d / t_d / HBM_PEAK, 2),
           "archive_bytes": A, "max_abs_error_fp64": err, "bound_held": err <= bound}
    if ref_cpu is not None:
        host = field.cpu().numpy()
        cpu = ref_cpu.compress(host, bound, ref_cpu.AVX2 if ref_cpu.has_avx2 else ref_cpu.SCALAR)
        res["byte_identical_vs_reference_cpu"] = cpu == archive.cpu().numpy().tobytes()
    return res


def measured_traffic(stage):
    """HBM bytes per launch of a stage's kernel from the committed rocprofv3
    FETCH_SIZE / WRITE_SIZE summary (calibrated against a plain copy kernel),
    or None when that summary does not list the stage."""
    try:
        for line in TRAFFIC_FILE.read_text().splitlines():
            cells = [c.strip() for c in line.strip().strip("|").split("|")]
            if len(cells) >= 5 and cells[0] == f"`{stage}`":
                return int(cells[-1])
    except (OSError, ValueError):
        pass
    return None


def main():
    args = parse()
    if args.gpus != 1:
        print(f"bench.py measures one GPU only; --gpus {args.gpus} is not supported (each MI355X "
              "compresses its own fields independently)", file=sys.stderr)
        sys.exit(2)
    import numpy as np
    import torch

    import waltz_amd
    from waltz_amd import _lib, synthetic

    assert torch.cuda.is_available(), "bench.py needs a GPU"
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    if args.batched_only:
        res, _ = batched_leg(torch, waltz_amd, synthetic, 1.0, 1.0)
        print(json.dumps({"batched": res}), flush=True)
        return
    S = args.size
    shape = (S, S, S)
    n = S ** 3
    w = 4
    seed = 20261202 + 1
    t0 = time.time()
    x = synthetic.grf(shape, slope=-5.0 / 3.0, seed=seed, offset=3.0, device=dev)
    lo, hi = float(x.min()), float(x.max())
    rel = 1e-3
    bound = rel * (float(np.float32(hi)) - float(np.float32(lo)))
    log(f"field {shape} f32 GRF k^-5/3 (+3.0) seed {seed}: range [{lo:.4f}, {hi:.4f}] abs bound {bound:.6g} "
        f"({time.time() - t0:.1f}s)")
    cap = waltz_amd.max_compressed_bytes(shape, torch.float32)
    arch = torch.empty(cap, dtype=torch.uint8, device=dev)
    out = torch.empty(shape, dtype=torch.float32, device=dev)

    def compress(b):
        return waltz_amd.compress(x, abs_error=b, out=arch)

    def decompress(a):
        return waltz_amd.decompress(a, shape=shape, dtype=torch.float32, out=out)

    # bit-neutral launch tuning of the lifting kernels for this geometry
    from waltz_amd import stages as stage_api
    t0 = time.time()
    stage_api.autotune(shape, torch.float32)
    tuning = stage_api.tuning_report()
    log(f"autotune ({time.time() - t0:.2f}s): {json.dumps(tuning)}")
    torch.cuda.synchronize()
    torch.cuda._sleep(1000)  # marks the end of tuning in kernel traces
    torch.cuda.synchronize()

    steps, warm = (2, 1) if args.profile_only else (args.steps, args.warmup)
    for _ in range(warm):
        decompress(compress(bound))
    torch.cuda.synchronize()
    tc, td = [], []
    t_begin = time.perf_counter()
    for _ in range(steps):
        a = time.perf_counter()
        archive = compress(bound)
        b = time.perf_counter()
        decompress(archive)
        c = time.perf_counter()
        tc.append(b - a)
        td.append(c - b)
    torch.cuda.synchronize()
    total = time.perf_counter() - t_begin
    A = archive.numel()
    field_bytes = n * w
    c_gbps = field_bytes / statistics.median(tc) / 1e9
    d_gbps = field_bytes / statistics.median(td) / 1e9
    log(f"compress {statistics.median(tc) * 1e3:.3f} ms ({c_gbps:.1f} GB/s), decompress "
        f"{statistics.median(td) * 1e3:.3f} ms ({d_gbps:.1f} GB/s), archive {A} B (CR {field_bytes / A:.3f})")
    if args.profile_only:
        # calibration for the HBM byte counters: one plain elementwise kernel
        # that reads 256 MiB and writes 256 MiB
        src = torch.ones(64 << 20, dtype=torch.float32, device=dev)
        dst = torch.empty_like(src)
        torch.mul(src, 2.0, out=dst)
        torch.cuda.synchronize()
        print(json.dumps({"profile_only": True, "compress_ms": statistics.median(tc) * 1e3,
                          "decompress_ms": statistics.median(td) * 1e3, "calibration_bytes": 2 * src.numel() * 4}))
        return

    # correctness: strict bound in FP64
    max_err = float((out.double() - x.double()).abs().max())
    assert max_err <= bound, (max_err, bound)

    # per-stage live timing (HIP events on the stream each stage runs on), one
    # call each; a stage launched in parts within one call (chunk ranges, index
    # ranges) counts its parts' sum, a stage of both calls their mean
    _lib.profile(True)
    _lib.profile_report()
    a_prof = compress(bound)
    per_call = [_lib.profile_report()]
    decompress(a_prof)
    per_call.append(_lib.profile_report())
    _lib.profile(False)
    stages = {}
    for rep in per_call:
        for name, (ms, cnt) in rep.items():
            tot, calls = stages.get(name, (0.0, 0))
            stages[name] = (tot + ms, calls + 1)
    sizes, side = [], S
    for lvl in range(5):
        sizes.append(side ** 3)
        side -= side // 2
    header = bytes(archive[:32].cpu().numpy())
    wzp_bytes = int.from_bytes(header[16:24], "little")
    np_repairs = int.from_bytes(header[24:28], "little")
    rows = []
    requant = "inverse_L0_repairs" in stages and "quantize_encode" in stages
    writeback = "none" if "coarse_requant" in stages else "box" if requant else "all"
    folded = "patch_keys" in stages
    for name, (ms, cnt) in stages.items():
        ab = stage_alg_bytes(name, n, w, wzp_bytes, sizes, np_repairs, writeback, folded)
        rows.append((ms / max(cnt, 1), name, ab))
    rows.sort(reverse=True)
    dom_ms, dom_name, dom_bytes = next(r for r in rows if r[2])
    achieved = dom_bytes / (dom_ms * 1e-3) / 1e9
    roofline = {"bound": "hbm", "kernel": dom_name, "achieved": round(achieved, 2), "peak": HBM_PEAK / 1e9,
                "unit": "GB/s", "frac": round(achieved * 1e9 / HBM_PEAK, 4), "traffic": measured_traffic(dom_name),
                "alg_bytes_per_launch": int(dom_bytes), "avg_launch_ms": round(dom_ms, 4)}
    rp = rocprof_duration_ms(dom_name)
    if rp:  # the committed rocprofv3 kernel table's duration of the same kernel
        roofline["rocprof_launch_ms"] = round(rp, 4)
        roofline["frac_rocprof"] = round(dom_bytes / (rp * 1e-3) / HBM_PEAK, 4)
    stage_table = {name: {"ms": round(ms, 4), "alg_GBps": round(ab / (ms * 1e-3) / 1e9, 1) if ab else None}
                   for ms, name, ab in rows}
    log("stages:", json.dumps(stage_table))

    # secondary bound: ABS 1e-4
    abs2 = 1e-4
    t2c, t2d = [], []
    for _ in range(3):
        a = time.perf_counter()
        arch2 = compress(abs2)
        b = time.perf_counter()
        decompress(arch2)
        c = time.perf_counter()
        t2c.append(b - a)
        t2d.append(c - b)
    arch2_host = arch2.cpu().numpy().tobytes()
    max_err2 = float((out.double() - x.double()).abs().max())
    assert max_err2 <= abs2

    # cold caches: L2 and the Infinity Cache evicted before every call
    tcc, tcd = [], []
    for _ in range(3):
        flush_caches(torch, dev)
        a = time.perf_counter()
        archive = compress(bound)
        b = time.perf_counter()
        tcc.append(b - a)
        flush_caches(torch, dev)
        b = time.perf_counter()
        decompress(archive)
        tcd.append(time.perf_counter() - b)

    # single-field compress / decode at the batched workload's bound (ABS 1e-3)
    t3c, t3 = [], []
    for _ in range(3):
        torch.cuda.synchronize()
        a = time.perf_counter()
        arch3 = compress(1e-3)
        b = time.perf_counter()
        decompress(arch3)
        t3.append(time.perf_counter() - b)
        t3c.append(b - a)
    d_gbps_abs1e3 = field_bytes / statistics.median(t3) / 1e9
    c_gbps_abs1e3 = field_bytes / statistics.median(t3c) / 1e9
    del arch3

    # pre-quantization coefficients in the input's precision vs an FP64 transform
    from waltz_amd import autograd
    lxy, lz, dyadic = autograd.default_levels(shape)
    c32 = stage_api.transform(x, lxy, lz, dyadic, inverse=False)
    c64 = stage_api.transform(x.double(), lxy, lz, dyadic, inverse=False)
    coeff_err = float((c32.double() - c64).abs().max())
    coeff_max = float(c64.abs().max())
    del c32, c64
    torch.cuda.empty_cache()

    # restore the REL archive for the identity check
    archive = compress(bound)
    arch_host = archive.cpu().numpy().tobytes()

    # alg bytes of the whole pipelines (compress / decompress), for % of HBM peak
    C_terms = sum(sizes[1:]) * 4 * w
    alg_c = (4 * w + 4.25) * n + C_terms + A
    alg_d = 3 * w * n + sum(sizes[1:]) * 2 * w + A
    result = {
        "metric": METRIC, "value": round(c_gbps, 2), "unit": "GB/s", "n_gpus": 1, "steps": steps, "warmup": warm,
        "ms_per_step": round(total / steps * 1e3, 3), "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"workload": f"{S}^3 float32 Gaussian random field, isotropic k^-5/3 spectrum, unit variance, "
                               f"+3.0 offset, seed {seed}; REL 1e-3 (abs {bound:.6g}); plain single-field codec",
                   "shape_zyx": list(shape), "rel_bound": rel, "abs_bound": bound},
        "compress_GBps": round(c_gbps, 2), "decompress_GBps": round(d_gbps, 2),
        "compress_ms": round(statistics.median(tc) * 1e3, 3), "decompress_ms": round(statistics.median(td) * 1e3, 3),
        "compress_pct_hbm_alg": round(100 * alg_c / statistics.median(tc) / HBM_PEAK, 2),
        "decompress_pct_hbm_alg": round(100 * alg_d / statistics.median(td) / HBM_PEAK, 2),
        "archive_bytes": A, "compression_ratio": round(field_bytes / A, 4), "max_abs_error_fp64": max_err,
        "coefficient_max_abs_error_vs_fp64_transform": coeff_err, "coefficient_max_abs": coeff_max,
        "abs_1e-4": {"compress_GBps": round(field_bytes / statistics.median(t2c) / 1e9, 2),
                     "decompress_GBps": round(field_bytes / statistics.median(t2d) / 1e9, 2),
                     "archive_bytes": len(arch2_host), "max_abs_error_fp64": max_err2},
        "cold_cache": {"compress_GBps": round(field_bytes / statistics.median(tcc) / 1e9, 2),
                       "decompress_GBps": round(field_bytes / statistics.median(tcd) / 1e9, 2),
                       "note": "1 GiB written before every call (L2 and Infinity Cache evicted); the headline "
                               "figures are warm medians"},
        "stages_ms": stage_table, "roofline": roofline, "tuning": tuning,
    }

    batch_host = None
    if not args.no_extra:
        log("batched leg ...")
        result["batched"], batch_host = batched_leg(torch, waltz_amd, synthetic, d_gbps_abs1e3, c_gbps_abs1e3)
        log("batched:", json.dumps(result["batched"]))
        log("autograd leg ...")
        result["autograd"] = autograd_leg(torch, waltz_amd, synthetic)
        log("autograd:", json.dumps(result["autograd"]))
        ref_cpu = None
        if not args.no_cpu:
            sys.path.insert(0, str(ROOT / "oracle"))
            import pyoracle
            ref_cpu = pyoracle.reference_or_none()
        log("more workloads ...")
        result["more_workloads"] = [
            extra_config(torch, waltz_amd, synthetic.fronts((96, 384, 384), seed=20261202 + 2, device=dev), 1e-6,
                         "384x384x96 float64 tanh fronts + k^-3 noise (seed 20261204), REL 1e-6", ref_cpu),
            extra_config(torch, waltz_amd, synthetic.grf((256, 256, 256), slope=-5.0 / 3.0, seed=20261202 + 5,
                                                         device=dev), 1e-3,
                         "256^3 float32 k^-5/3 Gaussian random field (seed 20261207), REL 1e-3", ref_cpu),
        ]
        log("more workloads:", json.dumps(result["more_workloads"]))
        torch.cuda.empty_cache()

    # CPU leg: byte identity with the reference CPU codec + its timing on this host
    if not args.no_cpu:
        sys.path.insert(0, str(ROOT / "oracle"))
        import pyoracle
        xh = x.cpu().numpy()
        ref = pyoracle.reference_or_none()
        all_cores = None
        if ref is not None and batch_host is not None:
            all_cores = cpu_batched_all_cores(pyoracle, batch_host)
        try:
            os.sched_setaffinity(0, {min(os.sched_getaffinity(0))})
        except (AttributeError, OSError):
            pass
        if ref is not None:
            backend = ref.AVX2 if ref.has_avx2 else ref.SCALAR
            t = time.perf_counter()
            cpu_arch = ref.compress(xh, bound, backend)
            tcpu_c = time.perf_counter() - t
            result["byte_identical_vs_reference_cpu"] = cpu_arch == arch_host
            t = time.perf_counter()
            ref.decompress(cpu_arch, shape, np.float32, backend)
            tcpu_d = time.perf_counter() - t
            cpu2 = ref.compress(xh, abs2, backend)
            result["abs_1e-4"]["byte_identical_vs_reference_cpu"] = cpu2 == arch2_host
            reps_c, reps_d = [tcpu_c], [tcpu_d]
            for _ in range(2):
                t = time.perf_counter()
                ref.compress(xh, bound, backend)
                reps_c.append(time.perf_counter() - t)
                t = time.perf_counter()
                ref.decompress(cpu_arch, shape, np.float32, backend)
                reps_d.append(time.perf_counter() - t)
            cc = field_bytes / statistics.median(reps_c) / 1e9
            # the scalar backend (the canonical arithmetic, same bytes) on a 256^3 corner
            sub = np.ascontiguousarray(xh[:256, :256, :256])
            t = time.perf_counter()
            sub_arch = ref.compress(sub, bound, ref.SCALAR)
            ts_c = time.perf_counter() - t
            t = time.perf_counter()
            ref.decompress(sub_arch, sub.shape, np.float32, ref.SCALAR)
            ts_d = time.perf_counter() - t
            result["cpu_baseline"] = {
                "value": round(cc, 4), "unit": "GB/s", "cores": 1, "kind": "reference",
                "sample": f"whole {S}^3 f32 field, REL 1e-3, reference CPU codec "
                          f"({'AVX2/FMA' if backend == ref.AVX2 else 'scalar'} backend, single-threaded, "
                          f"pinned to 1 core), median of 3 compress calls",
                "decompress_GBps": round(field_bytes / statistics.median(reps_d) / 1e9, 4),
                "gpu_over_cpu_compress": round(c_gbps / cc, 1),
                "scalar_backend": {"compress_GBps": round(sub.nbytes / ts_c / 1e9, 4),
                                   "decompress_GBps": round(sub.nbytes / ts_d / 1e9, 4), "cores": 1,
                                   "sample": "256^3 corner of the same field, same bound, one call each"}}
            if all_cores:
                result["cpu_baseline"]["batched_all_cores"] = all_cores
        else:
            o = pyoracle.Oracle()
            sub = np.ascontiguousarray(xh[:128, :128, :128])
            t = time.perf_counter()
            o.compress(sub, bound)
            tc1 = time.perf_counter() - t
            result["cpu_baseline"] = {"value": round(sub.nbytes / tc1 / 1e9, 4), "unit": "GB/s", "cores": 1,
                                      "kind": "port", "sample": "128^3 corner of the field, oracle C port, 1 call"}
    print(json.dumps(result), flush=True)


if __name__ == "__main__":
    main()
