#!/usr/bin/env python3
"""Benchmark of the batched real-FFT workload on one MI355X.

Workload (one "step"): 65536 real float32 signals of N=4096 and 65536 of N=4000 --
samples N(0,1) noise plus two unit tones at bins 100 and 1500.5 -- each through the
forward real transform (kiss_fftr_batch: N reals -> N/2+1 complex) and the inverse
(kiss_fftri_batch), inputs and outputs resident in HBM.  Throughput counts algorithmic
bytes (one read of the input, one write of the output: 4N + 8(N/2+1) per transform).

    python bench.py [--gpus 1] [--steps K] [--warmup W]

Prints one JSON line.  `roofline` is the dominant kernel (forward N=4096) timed with HIP
events on the stream it runs on; `cpu_baseline` is the reference KISS FFT built from its
own sources (oracle/_ref) timed on this host's cores on a bounded sample.
"""
from __future__ import annotations

import argparse
import json
import os
import subprocess
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBPS = 8000.0
BATCH = 65536
SIZES = (4096, 4000)


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def alg_bytes(n: int) -> int:
    return 4 * n + 8 * (n // 2 + 1)


def _cpu_model() -> str:
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def _ref_pass(exe: str, kind: str, n: int, sample: int, threads: int, mode: str) -> dict | None:
    r = subprocess.run([exe, kind, str(n), str(sample), str(threads), "5", mode], capture_output=True,
                       text=True, timeout=300)
    if r.returncode != 0:
        log("cpu baseline failed:", r.stdout, r.stderr)
        return None
    return json.loads(r.stdout)


def cpu_baseline(threads: int) -> dict | None:
    """The reference build timed on this host: kiss_fftr + kiss_fftri at N=4096 and N=4000.

    Three forms of the reference at its test flags (-O3 -ffast-math), each one warm-up pass
    and the median of 5 passes, cfgs allocated before timing:
      batch   (the reported value) OpenMP parallel for over the batch on `threads` cores, one
              cfg per thread;
      serial  the build without OpenMP, one thread;
      intra   the as-shipped OpenMP build (kiss_fft.c:250-271): one caller, each transform's
              top-level butterflies split over `threads` threads."""
    base = os.path.join(ROOT, "oracle", "_ref")
    exe, exe_serial = os.path.join(base, "cpu_baseline-float"), os.path.join(base, "cpu_baseline_serial-float")
    if not (os.path.exists(exe) and os.path.exists(exe_serial)):
        return None
    forms = (("batch", exe, threads, 16384), ("serial", exe_serial, 1, 2048), ("intra", exe, threads, 2048))
    res = {}
    for form, path, th, sample in forms:
        total_bytes = total_s = 0.0
        for n in SIZES:
            for kind in ("r2c", "c2r"):
                d = _ref_pass(path, kind, n, sample, th, "intra" if form == "intra" else "batch")
                if d is None:
                    return None
                total_s += d["median_s"]
                total_bytes += alg_bytes(n) * sample
        res[form] = {"GBps": round(total_bytes / total_s / 1e9, 3), "transforms_per_s": round(4 * sample / total_s, 1),
                     "threads": th, "signals_per_size_and_direction": sample}
    return {
        "value": res["batch"]["GBps"],
        "unit": "GB/s",
        "transforms_per_s": res["batch"]["transforms_per_s"],
        "cores": threads,
        "kind": "reference",
        "nproc": os.cpu_count(),
        "cpu_model": _cpu_model(),
        "sample": f"kiss_fftr + kiss_fftri at N=4096 and N=4000, {forms[0][3]} signals each, OpenMP parallel "
                  f"for over the batch ({threads} threads: this process's CPU share; one cfg per thread), "
                  "reference sources at -O3 -ffast-math, median of 5 passes after 1 warm-up",
        "forms": res,
    }


def _time(fn, stream, reps: int) -> float:
    """Seconds per call of `reps` back-to-back calls after two untimed calls; the wall time
    of the first call (plans, tables, first-use timing of kernel variants when the process
    has not run the workload before) is kept in _time.first_s.  The second untimed call
    runs the workload once more as it will run from then on (the first calls of a workload
    that takes a temporary map its pool memory)."""
    import torch
    t0 = time.perf_counter()
    fn()
    stream.synchronize()
    _time.first_s = time.perf_counter() - t0
    fn()
    stream.synchronize()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record(stream)
    for _ in range(reps):
        fn()
    e1.record(stream)
    e1.synchronize()
    return e0.elapsed_time(e1) / 1e3 / reps


def ceilings(stream, dev) -> dict | None:
    """Streaming rates of hand-written 16-byte-lane kernels on this device (libkfa_membench,
    kissfft_amd/csrc/bench/kfa_membench.hip): read-only, copy, and the real-forward row
    pattern of the N=4096 batch (65536 rows of 4096 floats in, 2049 complex out).  HIP events
    on `stream`, best of 3 rounds of 10 launches."""
    import ctypes

    import torch

    path = os.path.join(ROOT, "kissfft_amd", "lib", "libkfa_membench.so")
    if not os.path.exists(path):
        return None
    mb = ctypes.CDLL(path)
    vp, sz, ll, ci = ctypes.c_void_p, ctypes.c_size_t, ctypes.c_longlong, ctypes.c_int
    mb.kfa_mb_read.argtypes = [vp, sz, vp, vp, ci, ci]
    mb.kfa_mb_copy.argtypes = [vp, vp, sz, vp, ci, ci]
    mb.kfa_mb_rows.argtypes = [vp, vp, ll, ci, vp]
    mb.kfa_mb_rows8.argtypes = [vp, vp, ll, ci, vp]
    sp = stream.cuda_stream
    rows_in = BATCH * 4096 * 4
    rows_out = BATCH * 2049 * 8
    with torch.cuda.stream(stream):
        a = torch.rand(rows_in // 4, device=dev)
        b = torch.empty(rows_out // 4 + 4, device=dev)
        sink = torch.empty(1 << 20, device=dev)  # 4 MiB: 16 bytes for each of up to 256K workgroups
    stream.synchronize()

    def rate(fn, nbytes):
        best = 0.0
        if fn():
            raise RuntimeError("streaming-ceiling kernel refused its arguments")
        for _ in range(3):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record(stream)
            for _ in range(10):
                fn()
            e1.record(stream)
            e1.synchronize()
            best = max(best, nbytes * 10 / (e0.elapsed_time(e1) / 1e3) / 1e9)
        return round(best, 1)

    # the best of a few launch shapes (workgroups per CU, 16-byte loads in flight per thread)
    shapes = [(16, 4), (32, 4), (128, 4)]
    out = {
        "read_GBps": max(rate(lambda g=g, u=u: mb.kfa_mb_read(a.data_ptr(), rows_in, sink.data_ptr(), sp, g, u),
                              rows_in) for g, u in shapes),
        "copy_GBps": max(rate(lambda g=g, u=u: mb.kfa_mb_copy(a.data_ptr(), b.data_ptr(), rows_in, sp, g, u),
                              2 * rows_in) for g, u in shapes),
        "r2c_rows_16B_GBps": rate(lambda: mb.kfa_mb_rows(a.data_ptr(), b.data_ptr(), BATCH, 4096, sp),
                                  rows_in + rows_out),
        "r2c_rows_8B_GBps": rate(lambda: mb.kfa_mb_rows8(a.data_ptr(), b.data_ptr(), BATCH, 4096, sp),
                                 rows_in + rows_out),
        "unit": "GB/s",
        "kernels": "hand-written streaming kernels: read and copy in 16-byte lanes, the r2c row pattern in "
                   "16- and 8-byte lanes (kissfft_amd/csrc/bench/kfa_membench.hip)",
    }
    # the row-pattern ceiling: the faster of the two lane widths
    out["r2c_rows_GBps"] = max(out["r2c_rows_16B_GBps"], out["r2c_rows_8B_GBps"])
    del a, b, sink
    return out


def other_configs(lib, stream, dev) -> dict:
    """The reference's other workloads, each timed on its own (inputs resident in HBM)."""
    import numpy as np
    import torch

    import kissfft_amd

    out = {}

    def rec(name, secs, nbytes, transforms, **extra):
        out[name] = {"us": round(secs * 1e6, 1), "GBps": round(nbytes / secs / 1e9, 1),
                     "pct_hbm_peak": round(100 * nbytes / secs / 1e9 / HBM_PEAK_GBPS, 2),
                     "transforms_per_s": round(transforms / secs, 1), **extra}

    with torch.cuda.stream(stream):
        # complex float N=1200, 256 transforms (latency-bound: one launch of 4.9 MB)
        x = torch.rand(256, 1200, 2, device=dev) * 2 - 1
        y = torch.empty_like(x)
    cfg = lib.fft_alloc(1200)
    # back-to-back calls of the C entry point (arguments prepared once); the Python
    # binding's own per-call cost (about 3 us of argument checks) is reported beside it
    t_py = _time(lambda: lib.fft_batch(cfg, x, y, 256, 1200, 1200, stream=stream), stream, 200)
    L, xp, yp, sp = lib.L, x.data_ptr(), y.data_ptr(), stream.cuda_stream
    if L.kiss_fft_batch_async(cfg, xp, 1, 1200, yp, 1200, 256, sp) != 0:
        raise RuntimeError("kiss_fft_batch_async failed")
    t = _time(lambda: L.kiss_fft_batch_async(cfg, xp, 1, 1200, yp, 1200, 256, sp), stream, 500)
    rec("c2c_float_1200_x256", t, 256 * 16 * 1200, 256, us_via_python_binding=round(t_py * 1e6, 1),
        calls="kiss_fft_batch_async back to back on one stream")

    # the same length batched at HBM scale: complex float N=1200, 2^18 transforms (1.2 GiB
    # per side), and a power-of-two length, N=4096 x 65536 (2 GiB per side)
    for n, b in ((1200, 1 << 18), (4096, 1 << 16)):
        with torch.cuda.stream(stream):
            xb = torch.rand(b, n, 2, device=dev) * 2 - 1
            yb = torch.empty_like(xb)
        cb = lib.fft_alloc(n)
        t = _time(lambda: lib.fft_batch(cb, xb, yb, b, n, n, stream=stream), stream, 10)
        rec(f"c2c_float_{n}_x{b}", t, b * 16 * n, b, first_call_ms=round(_time.first_s * 1e3, 1))
        del xb, yb

    # Q15 complex N=512, 2^20 transforms
    lq = kissfft_amd.load("int16_t")
    B = 1 << 20
    with torch.cuda.stream(stream):
        xq = torch.randint(-16384, 16384, (B, 512, 2), dtype=torch.int16, device=dev)
        yq = torch.empty_like(xq)
    cq = lq.fft_alloc(512)
    t = _time(lambda: lq.fft_batch(cq, xq, yq, B, 512, 512, stream=stream), stream, 5)
    rec("c2c_q15_512_x1048576", t, B * 8 * 512, B, first_call_ms=round(_time.first_s * 1e3, 1))
    del xq, yq

    # Q31 complex N=512, 2^19 transforms (the same 2 GiB per side as the Q15 line)
    l31 = kissfft_amd.load("int32_t")
    B = 1 << 19
    with torch.cuda.stream(stream):
        x31 = torch.randint(-(1 << 30), 1 << 30, (B, 512, 2), dtype=torch.int32, device=dev)
        y31 = torch.empty_like(x31)
    c31 = l31.fft_alloc(512)
    t = _time(lambda: l31.fft_batch(c31, x31, y31, B, 512, 512, stream=stream), stream, 5)
    rec("c2c_q31_512_x524288", t, B * 16 * 512, B, first_call_ms=round(_time.first_s * 1e3, 1))
    del x31, y31

    # a length outside the built-in registry (3000 = 2^3 * 3 * 5^3): compiled at run time on
    # first use (plus the timing of its thread shapes); the first call is reported apart
    with torch.cuda.stream(stream):
        xr = torch.rand(65536, 3000, 2, device=dev) * 2 - 1
        yr = torch.empty_like(xr)
    stream.synchronize()
    cr = lib.fft_alloc(3000)
    t0 = time.perf_counter()
    lib.fft_batch(cr, xr, yr, 65536, 3000, 3000, stream=stream)
    stream.synchronize()
    first = time.perf_counter() - t0
    t = _time(lambda: lib.fft_batch(cr, xr, yr, 65536, 3000, 3000, stream=stream), stream, 10)
    rec("c2c_float_3000_x65536_runtime_compiled", t, 65536 * 16 * 3000, 65536, first_call_ms=round(first * 1e3, 1))
    del xr, yr

    # a length of a generic radix (2401 = 7^4, kf_bfly_generic in the reference): the odd
    # radix-7 DFT compiled at run time the same way
    with torch.cuda.stream(stream):
        xg = torch.rand(55900, 2401, 2, device=dev) * 2 - 1
        yg = torch.empty_like(xg)
    stream.synchronize()
    cg = lib.fft_alloc(2401)
    t0 = time.perf_counter()
    lib.fft_batch(cg, xg, yg, 55900, 2401, 2401, stream=stream)
    stream.synchronize()
    first = time.perf_counter() - t0
    t = _time(lambda: lib.fft_batch(cg, xg, yg, 55900, 2401, 2401, stream=stream), stream, 10)
    rec("c2c_float_2401_x55900_runtime_compiled", t, 55900 * 16 * 2401, 55900, first_call_ms=round(first * 1e3, 1))
    del xg, yg

    # 3-D complex float 64x96x120, 16 transforms
    dims = (64, 96, 120)
    with torch.cuda.stream(stream):
        x3 = torch.rand((16,) + dims + (2,), device=dev) * 2 - 1
        y3 = torch.empty_like(x3)
    c3 = lib.fftnd_alloc(dims)
    t = _time(lambda: lib.fftnd_batch(c3, x3, y3, 16, stream=stream), stream, 10)
    rec("nd_float_64x96x120_x16", t, 16 * 16 * 64 * 96 * 120, 16, first_call_ms=round(_time.first_s * 1e3, 1))
    del x3, y3

    # 2-D real float 1024x1000, 32 transforms (forward and inverse)
    d2 = (1024, 1000)
    with torch.cuda.stream(stream):
        xr = torch.randn((32,) + d2, device=dev)
        Xr = torch.empty(32, 1024, 501, 2, device=dev)
        yr = torch.empty_like(xr)
    cf, ci = lib.fftndr_alloc(d2), lib.fftndr_alloc(d2, True)
    nb = 32 * (4 * 1024 * 1000 + 8 * 1024 * 501)
    t = _time(lambda: lib.fftndr_batch(cf, xr, Xr, 32, stream=stream), stream, 10)
    rec("ndr_float_1024x1000_x32_fwd", t, nb, 32, first_call_ms=round(_time.first_s * 1e3, 1))
    t = _time(lambda: lib.fftndri_batch(ci, Xr, yr, 32, stream=stream), stream, 10)
    rec("ndr_float_1024x1000_x32_inv", t, nb, 32, first_call_ms=round(_time.first_s * 1e3, 1))
    del xr, Xr, yr

    # uneven batching: 64 batches of mixed lengths and kinds (generic prime 1009 included),
    # batch counts log-uniform in [1, 512], as one kiss_fft_multi launch replayed from a
    # hipGraph, against the same batches as one batched call each on the same stream
    rng = np.random.default_rng(11)
    menu = [(kissfft_amd.MultiBatch.C2C_FWD, 256), (kissfft_amd.MultiBatch.C2C_FWD, 1000),
            (kissfft_amd.MultiBatch.C2C_FWD, 1009), (kissfft_amd.MultiBatch.C2C_FWD, 1200),
            (kissfft_amd.MultiBatch.C2C_INV, 3072), (kissfft_amd.MultiBatch.R2C, 4096),
            (kissfft_amd.MultiBatch.C2R, 4000), (kissfft_amd.MultiBatch.C2C_FWD, 120)]
    items, calls, mbytes, mtrans = [], [], 0, 0
    for i in range(64):
        kind, n = menu[i % len(menu)]
        cnt = int(np.exp(rng.uniform(0, np.log(512))))
        nin = (n * cnt * 2) if kind in (0, 1) else (n * cnt if kind == 2 else (n // 2 + 1) * cnt * 2)
        nout = (n * cnt * 2) if kind in (0, 1) else ((n // 2 + 1) * cnt * 2 if kind == 2 else n * cnt)
        with torch.cuda.stream(stream):
            fi = torch.rand(nin, device=dev) * 2 - 1
            fo = torch.empty(nout, device=dev)
        items.append((kind, n, fi, fo, cnt))
        mbytes += 4 * (nin + nout)
        mtrans += cnt
        if kind in (0, 1):
            cf1 = lib.fft_alloc(n, kind == 1)
            calls.append(lambda c=cf1, a=fi, b=fo, k=cnt, m=n: lib.fft_batch(c, a, b, k, m, m, stream=stream))
        elif kind == 2:
            cf1 = lib.fftr_alloc(n)
            calls.append(lambda c=cf1, a=fi, b=fo, k=cnt, m=n: lib.fftr_batch(c, a, b, k, m, m // 2 + 1,
                                                                              stream=stream))
        else:
            cf1 = lib.fftr_alloc(n, True)
            calls.append(lambda c=cf1, a=fi, b=fo, k=cnt, m=n: lib.fftri_batch(c, a, b, k, m // 2 + 1, m,
                                                                               stream=stream))
    torch.cuda.synchronize()
    mb = kissfft_amd.MultiBatch(lib, items)
    mb.capture(stream)
    t_multi = _time(lambda: mb.replay(stream), stream, 20)

    # the same multi-batch with one launch per group instead of the fused launch
    prev = os.environ.get("KISSFFT_AMD_MULTI_FUSED")
    os.environ["KISSFFT_AMD_MULTI_FUSED"] = "0"
    try:
        mb_sep = kissfft_amd.MultiBatch(lib, items)
    finally:
        if prev is None:
            del os.environ["KISSFFT_AMD_MULTI_FUSED"]
        else:
            os.environ["KISSFFT_AMD_MULTI_FUSED"] = prev
    mb_sep.capture(stream)
    t_sep = _time(lambda: mb_sep.replay(stream), stream, 20)
    mb_sep.close()

    def per_batch():
        for c in calls:
            c()
    t_calls = _time(per_batch, stream, 20)
    rec("multi_uneven_64_batches", t_multi, mbytes, mtrans,
        separate_launches_us=round(t_sep * 1e6, 1),
        per_batch_calls_us=round(t_calls * 1e6, 1), speedup_vs_per_batch_calls=round(t_calls / t_multi, 2),
        kinds_lengths="c2c 256/1000/1009/1200/120, c2c inverse 3072, r2c 4096, c2r 4000",
        launch=mb.info())
    mb.close()
    del items, calls

    # fast FIR (overlap-scrap, kiss_fastfir): 2^28 real samples (1 GiB) through a 1000-tap
    # filter, one call on device buffers, with the reference's default block (the next power
    # of two >= 2 (taps - 1): 2048) and with 4096 and 8192: the block sets how many samples a
    # call completes, the transform length is the library's own choice
    nsamp, ntap = 1 << 28, 1000
    h = np.random.default_rng(13).standard_normal(ntap).astype(np.float32)
    with torch.cuda.stream(stream):
        fin = torch.rand(nsamp, device=dev) * 2 - 1
        fout = torch.empty(nsamp, device=dev)
    torch.cuda.synchronize()
    for nfft in (0, 4096, 8192):
        ff = lib.fastfir_alloc(h, real=True, nfft=nfft)
        written = [0]

        def fir():
            ff.offset = 0
            written[0] = ff.filter(fin, fout, nsamp)
        # the kiss_fastfir call is synchronous (results valid on return): wall time per call
        fir()
        t0 = time.perf_counter()
        for _ in range(5):
            fir()
        t = (time.perf_counter() - t0) / 5
        rec(f"fastfir_real_2p28_samples_1000_taps_nfft{ff.nfft}", t, 4 * nsamp + 4 * written[0],
            written[0] // ff.ngood, samples_per_s=round(nsamp / t, 1), good_per_block=ff.ngood)
    del fin, fout
    return out


def serving(lib, dev, count: int, rate: float, streams: int = 0) -> dict:
    """The serving stream: `count` seeded requests (c2c / r2c / inverse, n in {256, 1000,
    1009, 3072, 65536, 1048576}, batch log-uniform in [1, 4096]) through one request server.

    open loop:  Poisson arrivals at `rate` per second (and the same arrivals at half that
                rate), submitted at their arrival times; p50 / p99 latency (submit to
                completion) under that offered load.
    saturated:  the same requests all submitted at once; throughput = algorithmic bytes /
                (first submit to last completion).
    per-call:   the same requests as a loop of single-transform kiss_fft / kiss_fftr /
                kiss_fftri calls (one call per transform, device pointers, synchronous), the
                drop-in API used one transform at a time.
    Inputs (uniform [-1, 1)) and outputs are resident in HBM before timing starts; every
    request of one (kind, n) reads the same input buffer (read-only), each request writes
    its own output buffer."""
    import torch

    from kissfft_amd import workloads as W

    reqs = W.serving_stream(count, rate)
    kinds = {"c2c": 0, "c2c_inv": 1, "r2c": 2, "c2r": 3}
    inputs = {}
    for r in reqs:
        key = (r["kind"], r["n"])
        inputs[key] = max(inputs.get(key, 0), W.request_bytes(r["kind"], r["n"], r["batch"])[0])
    ibufs = {k: (torch.rand(v // 4, device=dev) * 2 - 1) for k, v in inputs.items()}
    obufs = [torch.empty(W.request_bytes(r["kind"], r["n"], r["batch"])[1] // 4, device=dev) for r in reqs]
    torch.cuda.synchronize()
    total_bytes = sum(sum(W.request_bytes(r["kind"], r["n"], r["batch"])) for r in reqs)
    transforms = sum(r["batch"] for r in reqs)

    srv = lib.server(streams=streams)
    # warm-up: plans, twiddles and variant choice of every (kind, n), one transform each;
    # each first request is timed (submit to completion): the cold-start latency a new
    # server pays once per (kind, n)
    cold = {}
    for key in inputs:
        warm_out = torch.empty(W.request_bytes(key[0], key[1], 1)[1] // 4, device=dev)
        tw = time.perf_counter()
        srv.wait(srv.submit(kinds[key[0]], key[1], ibufs[key], warm_out, 1))
        cold[f"{key[0]}_{key[1]}"] = round((time.perf_counter() - tw) * 1e3, 1)
    srv.reset_stats()

    def run(open_loop: bool, stretch: float = 1.0):
        # stretch > 1: the same arrivals spread over stretch times as long (rate / stretch)
        t0 = time.perf_counter()
        tickets = []
        for r, ob in zip(reqs, obufs):
            if open_loop:
                while time.perf_counter() - t0 < r["t"] * stretch:
                    pass
            tickets.append(srv.submit(kinds[r["kind"]], r["n"], ibufs[(r["kind"], r["n"])], ob, r["batch"]))
        for t in tickets:
            srv.wait(t)
        st = srv.stats()
        srv.reset_stats()
        return st

    ol = run(True)
    ol_half = run(True, 2.0)
    sat = run(False)
    sample = [0, len(reqs) // 2, len(reqs) - 1]
    served = {i: obufs[i][: W.request_bytes(reqs[i]["kind"], reqs[i]["n"], 1)[1] // 4].cpu() for i in sample}

    cfgs = {}
    for key in inputs:
        kind, n = key
        cfgs[key] = (lib.fft_alloc(n, kind == "c2c_inv") if kind.startswith("c2c")
                     else lib.fftr_alloc(n, kind == "c2r"))
    L = lib.L
    calls = {"c2c": L.kiss_fft, "c2c_inv": L.kiss_fft, "r2c": L.kiss_fftr, "c2r": L.kiss_fftri}
    # every single call is timed (each returns with its result valid), and each request's
    # run of calls; the per-call latency under the same open-loop arrivals is the FIFO
    # queue of those request durations on one caller thread
    call_s, req_s = [], []
    pc = time.perf_counter
    t0 = pc()
    for r, ob in zip(reqs, obufs):
        key = (r["kind"], r["n"])
        ib, ob1 = W.request_bytes(r["kind"], r["n"], 1)
        fn, cfg = calls[r["kind"]], cfgs[key]
        ip, op = ibufs[key].data_ptr(), ob.data_ptr()
        tr = pc()
        for b in range(r["batch"]):
            tc = pc()
            fn(cfg, ip + b * ib, op + b * ob1)
            call_s.append(pc() - tc)
        req_s.append(pc() - tr)
    torch.cuda.synchronize()
    per_call_s = pc() - t0
    done, fifo = 0.0, []
    for r, d in zip(reqs, req_s):
        done = max(done, r["t"]) + d
        fifo.append(done - r["t"])
    same = all(torch.equal(served[i], obufs[i][: served[i].numel()].cpu()) for i in sample)
    srv.close()
    del ibufs, obufs
    torch.cuda.empty_cache()

    def ms(v):
        return round(v * 1e3, 3)

    def q(v, f):
        v = sorted(v)
        return v[min(len(v) - 1, int(f * (len(v) - 1) + 0.5))] if v else 0.0

    sat_gbps = total_bytes / sat["span_s"] / 1e9
    pc_gbps = total_bytes / per_call_s / 1e9
    return {
        "requests": len(reqs), "transforms": transforms, "alg_bytes": total_bytes,
        "sizes": list(W.SERVE_SIZES), "kinds": "c2c, r2c, inverse (c2r; at odd n 1009: r2c->c2c, inverse->c2c inverse)",
        "open_loop": {"rate_per_s": rate, "offered_GBps": round(total_bytes / reqs[-1]["t"] / 1e9, 1),
                      "p50_ms": ms(ol["p50_s"]), "p99_ms": ms(ol["p99_s"]), "max_ms": ms(ol["max_s"]),
                      "GBps": round(total_bytes / ol["span_s"] / 1e9, 1), "launches": ol["launches"]},
        "open_loop_half_rate": {"rate_per_s": rate / 2, "offered_GBps": round(total_bytes / reqs[-1]["t"] / 2e9, 1),
                                "p50_ms": ms(ol_half["p50_s"]), "p99_ms": ms(ol_half["p99_s"]),
                                "max_ms": ms(ol_half["max_s"]), "GBps": round(total_bytes / ol_half["span_s"] / 1e9, 1),
                                "launches": ol_half["launches"]},
        "saturated": {"GBps": round(sat_gbps, 1), "transforms_per_s": round(transforms / sat["span_s"], 1),
                      "span_ms": ms(sat["span_s"]), "p50_ms": ms(sat["p50_s"]), "p99_ms": ms(sat["p99_s"]),
                      "launches": sat["launches"]},
        "per_call": {"GBps": round(pc_gbps, 2), "transforms_per_s": round(transforms / per_call_s, 1),
                     "seconds": round(per_call_s, 3),
                     "call_p50_us": round(1e6 * q(call_s, 0.50), 1), "call_p99_us": round(1e6 * q(call_s, 0.99), 1),
                     "request_p50_ms": ms(q(req_s, 0.50)), "request_p99_ms": ms(q(req_s, 0.99)),
                     "open_loop_p50_ms": ms(q(fifo, 0.50)), "open_loop_p99_ms": ms(q(fifo, 0.99)),
                     "open_loop_rate_per_s": rate},
        "speedup_vs_per_call": round(sat_gbps / pc_gbps, 2),
        "cold_first_request_ms": {"per_kind_n": cold, "max": max(cold.values()), "sum": round(sum(cold.values()), 1)},
        "served_equals_per_call": bool(same),
    }


def _profile_setup(name, lib, stream, dev):
    """(call, algorithmic bytes per call) of one named workload, inputs resident in HBM."""
    import torch

    import kissfft_amd
    with torch.cuda.stream(stream):
        if name in ("c2c_1m", "c2c_64k"):
            n, b = (1 << 20, 256) if name == "c2c_1m" else (65536, 4096)
            x = torch.rand(b, n, 2, device=dev) * 2 - 1
            y = torch.empty_like(x)
            cfg = lib.fft_alloc(n)
            return (lambda: lib.fft_batch(cfg, x, y, b, n, n, stream=stream)), 16 * n * b
        if name in ("r2c_1m", "c2r_1m"):
            n, b = 1 << 20, 256
            x = torch.rand(b, n, device=dev)
            X = torch.rand(b, n // 2 + 1, 2, device=dev)
            nb = (4 * n + 8 * (n // 2 + 1)) * b
            if name == "r2c_1m":
                cfg = lib.fftr_alloc(n)
                return (lambda: lib.fftr_batch(cfg, x, X, b, n, n // 2 + 1, stream=stream)), nb
            cfg = lib.fftr_alloc(n, True)
            return (lambda: lib.fftri_batch(cfg, X, x, b, n // 2 + 1, n, stream=stream)), nb
        if name == "nd_64x96x120":
            dims = (64, 96, 120)
            x = torch.rand((16,) + dims + (2,), device=dev) * 2 - 1
            y = torch.empty_like(x)
            cfg = lib.fftnd_alloc(dims)
            return (lambda: lib.fftnd_batch(cfg, x, y, 16, stream=stream)), 16 * 16 * 64 * 96 * 120
        if name in ("ndr_1024x1000", "ndri_1024x1000"):
            d2 = (1024, 1000)
            xr = torch.randn((32,) + d2, device=dev)
            Xr = torch.randn(32, 1024, 501, 2, device=dev)
            nb = 32 * (4 * 1024 * 1000 + 8 * 1024 * 501)
            if name == "ndr_1024x1000":
                cfg = lib.fftndr_alloc(d2)
                return (lambda: lib.fftndr_batch(cfg, xr, Xr, 32, stream=stream)), nb
            cfg = lib.fftndr_alloc(d2, True)
            return (lambda: lib.fftndri_batch(cfg, Xr, xr, 32, stream=stream)), nb
        if name == "c2c_1200":
            x = torch.rand(256, 1200, 2, device=dev) * 2 - 1
            y = torch.empty_like(x)
            cfg = lib.fft_alloc(1200)
            return (lambda: lib.fft_batch(cfg, x, y, 256, 1200, 1200, stream=stream)), 256 * 16 * 1200
        if name == "q15_512":
            lq = kissfft_amd.load("int16_t")
            b = 1 << 20
            x = torch.randint(-16384, 16384, (b, 512, 2), dtype=torch.int16, device=dev)
            y = torch.empty_like(x)
            cfg = lq.fft_alloc(512)
            return (lambda: lq.fft_batch(cfg, x, y, b, 512, 512, stream=stream)), b * 8 * 512
        if name == "multi_64":
            import numpy as np
            rng = np.random.default_rng(11)
            M = kissfft_amd.MultiBatch
            menu = [(M.C2C_FWD, 256), (M.C2C_FWD, 1000), (M.C2C_FWD, 1009), (M.C2C_FWD, 1200), (M.C2C_INV, 3072),
                    (M.R2C, 4096), (M.C2R, 4000), (M.C2C_FWD, 120)]
            items, nbytes = [], 0
            for i in range(64):
                kind, n = menu[i % len(menu)]
                cnt = int(np.exp(rng.uniform(0, np.log(512))))
                nin = (n * cnt * 2) if kind in (0, 1) else (n * cnt if kind == 2 else (n // 2 + 1) * cnt * 2)
                nout = (n * cnt * 2) if kind in (0, 1) else ((n // 2 + 1) * cnt * 2 if kind == 2 else n * cnt)
                items.append((kind, n, torch.rand(nin, device=dev) * 2 - 1, torch.empty(nout, device=dev), cnt))
                nbytes += 4 * (nin + nout)
            stream.synchronize()
            mb = M(lib, items)
            mb.capture(stream)
            return (lambda: mb.replay(stream)), nbytes
    raise ValueError(name)


PROFILE_WORKLOADS = ("c2c_1m", "c2c_64k", "r2c_1m", "c2r_1m", "nd_64x96x120", "ndr_1024x1000", "ndri_1024x1000",
                     "c2c_1200", "q15_512", "multi_64")


def profile_workload(name, lib, stream, dev) -> int:
    import torch
    call, nbytes = _profile_setup(name, lib, stream, dev)
    call()  # plans, kernel choices, tuning
    stream.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record(stream)
    for _ in range(3):
        call()
    e1.record(stream)
    e1.synchronize()
    s = e0.elapsed_time(e1) / 1e3 / 3
    print(json.dumps({"profile": name, "us_per_call": round(s * 1e6, 1), "alg_bytes": nbytes,
                      "GBps": round(nbytes / s / 1e9, 1)}), flush=True)
    return 0


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-other-configs", action="store_true",
                    help="skip the secondary workloads reported under other_configs")
    ap.add_argument("--no-serving", action="store_true", help="skip the serving-stream measurement")
    ap.add_argument("--serve-requests", type=int, default=192)
    ap.add_argument("--serve-rate", type=float, default=2000.0, help="open-loop arrivals per second")
    ap.add_argument("--serve-streams", type=int, default=0,
                    help="streams of the request server (0: the library default)")
    ap.add_argument("--pmc-run", action="store_true",
                    help="for rocprofv3 --pmc: one plain copy of a known size (the counter scale), "
                         "then one forward and one inverse N=4096 launch, and exit")
    ap.add_argument("--pmc-long-real", action="store_true",
                    help="for rocprofv3: 256 real signals of 2^20 points, forward and inverse three "
                         "times each (the fused four-step real passes), and exit")
    ap.add_argument("--pmc-q15", action="store_true",
                    help="for rocprofv3: Q15 c2c N=512 over 2^20 transforms, three launches after "
                         "the plan's first call, and exit")
    ap.add_argument("--profile", choices=sorted(PROFILE_WORKLOADS),
                    help="for rocprofv3: one workload -- its first call (plans, tuning), then three "
                         "timed calls on one stream -- and exit")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU only: --gpus {args.gpus} is not supported (batches shard "
              "trivially across GPUs; no multi-GPU path is built)", file=sys.stderr)
        return 2

    import torch

    import kissfft_amd

    if not torch.cuda.is_available():
        log("no GPU visible")
        return 1
    dev = torch.device("cuda:0")
    lib = kissfft_amd.load("float")
    stream = torch.cuda.Stream(device=dev)

    if args.profile:
        return profile_workload(args.profile, lib, stream, dev)

    if args.pmc_long_real:
        n, b = 1 << 20, 256
        with torch.cuda.stream(stream):
            x = torch.rand(b, n, device=dev)
            X = torch.empty(b, n // 2 + 1, 2, device=dev)
            y = torch.empty_like(x)
        fcfg, icfg = lib.fftr_alloc(n, False), lib.fftr_alloc(n, True)
        for _ in range(3):
            lib.fftr_batch(fcfg, x, X, b, n, n // 2 + 1, stream=stream)
            lib.fftri_batch(icfg, X, y, b, n // 2 + 1, n, stream=stream)
        stream.synchronize()
        print(json.dumps({"pmc_long_real": True, "n": n, "signals": b}), flush=True)
        return 0

    if args.pmc_q15:
        lq = kissfft_amd.load("int16_t")
        b = 1 << 20
        with torch.cuda.stream(stream):
            xq = torch.randint(-16384, 16384, (b, 512, 2), dtype=torch.int16, device=dev)
            yq = torch.empty_like(xq)
        cq = lq.fft_alloc(512)
        lq.fft_batch(cq, xq, yq, b, 512, 512, stream=stream)  # plan + variant choice
        for _ in range(3):
            lq.fft_batch(cq, xq, yq, b, 512, 512, stream=stream)
        stream.synchronize()
        print(json.dumps({"pmc_q15": True, "n": 512, "transforms": b, "alg_bytes": b * 8 * 512}), flush=True)
        return 0

    bufs = {}
    with torch.cuda.stream(stream):
        g = torch.Generator(device=dev).manual_seed(2)
        for n in SIZES:
            t = torch.arange(n, device=dev, dtype=torch.float64)
            tones = (torch.cos(2 * torch.pi * 100.0 * t / n) + torch.cos(2 * torch.pi * 1500.5 * t / n)).float()
            x = torch.randn(BATCH, n, generator=g, device=dev) + tones
            X = torch.empty(BATCH, n // 2 + 1, 2, device=dev)
            y = torch.empty(BATCH, n, device=dev)
            bufs[n] = (x, X, y, lib.fftr_alloc(n, False), lib.fftr_alloc(n, True))
    stream.synchronize()

    if args.pmc_run:
        x, X, y, fcfg, icfg = bufs[4096]
        with torch.cuda.stream(stream):
            src = torch.empty(256 << 20, dtype=torch.float32, device=dev)  # 1 GiB
            dst = torch.empty_like(src)
            dst.copy_(src)
        lib.fftr_batch(fcfg, x, X, BATCH, 4096, 2049, stream=stream)  # plan + tuning
        lib.fftri_batch(icfg, X, y, BATCH, 2049, 4096, stream=stream)
        stream.synchronize()
        lib.fftr_batch(fcfg, x, X, BATCH, 4096, 2049, stream=stream)
        lib.fftri_batch(icfg, X, y, BATCH, 2049, 4096, stream=stream)
        stream.synchronize()
        print(json.dumps({"pmc_run": True, "copy_bytes": 2 * src.numel() * 4,
                          "r2c_alg_bytes": alg_bytes(4096) * BATCH}), flush=True)
        return 0

    def step():
        for n in SIZES:
            x, X, y, fcfg, icfg = bufs[n]
            lib.fftr_batch(fcfg, x, X, BATCH, n, n // 2 + 1, stream=stream)
            lib.fftri_batch(icfg, X, y, BATCH, n // 2 + 1, n, stream=stream)

    # the first step also builds the plans and times the kernel variants of the four
    # (direction, length) keys: reported as the first-use cost
    t_first = time.perf_counter()
    step()
    torch.cuda.synchronize()
    first_step_s = time.perf_counter() - t_first
    for _ in range(max(0, args.warmup - 1)):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    step_bytes = sum(2 * alg_bytes(n) * BATCH for n in SIZES)
    value = step_bytes * args.steps / dt / 1e9
    transforms_per_s = 4 * BATCH * args.steps / dt

    # dominant kernel: forward N=4096, HIP events on its stream
    x, X, y, fcfg, icfg = bufs[4096]
    reps = max(10, args.steps)
    ev0 = torch.cuda.Event(enable_timing=True)
    ev1 = torch.cuda.Event(enable_timing=True)
    ev0.record(stream)
    for _ in range(reps):
        lib.fftr_batch(fcfg, x, X, BATCH, 4096, 2049, stream=stream)
    ev1.record(stream)
    ev1.synchronize()
    kern_s = ev0.elapsed_time(ev1) / 1e3 / reps
    kbytes = alg_bytes(4096) * BATCH
    achieved = kbytes / kern_s / 1e9
    per_kernel = {}
    for n in SIZES:
        x, X, y, fcfg, icfg = bufs[n]
        for name, fn in (("r2c", lambda: lib.fftr_batch(fcfg, x, X, BATCH, n, n // 2 + 1, stream=stream)),
                         ("c2r", lambda: lib.fftri_batch(icfg, X, y, BATCH, n // 2 + 1, n, stream=stream))):
            ev0.record(stream)
            for _ in range(5):
                fn()
            ev1.record(stream)
            ev1.synchronize()
            s = ev0.elapsed_time(ev1) / 1e3 / 5
            per_kernel[f"{name}_{n}"] = {"us": round(s * 1e6, 1), "GBps": round(alg_bytes(n) * BATCH / s / 1e9, 1)}

    ceil = ceilings(stream, dev)
    others = {} if args.no_other_configs else other_configs(lib, stream, dev)
    serve = None
    if not args.no_serving:
        del bufs, x, X, y
        torch.cuda.empty_cache()
        serve = serving(lib, dev, args.serve_requests, args.serve_rate, args.serve_streams)

    traffic = None
    tfile = os.path.join(ROOT, "profiles", "traffic_r2c_4096.json")
    if os.path.exists(tfile):
        with open(tfile) as f:
            traffic = json.load(f).get("hbm_bytes_per_launch")

    cpu = None
    if not args.no_cpu_baseline:
        threads = int(os.environ.get("OMP_NUM_THREADS", "0") or 0) or (os.cpu_count() or 1)
        try:
            cpu = cpu_baseline(threads)
        except Exception as e:  # the baseline is reported, never required
            log("cpu baseline skipped:", e)

    out = {
        "metric": "HBM GB/s (% peak) + transforms/s; served p50/p99 vs per-call @ rel-L2<=1e-6",
        "value": round(value, 2),
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(dt / args.steps * 1e3, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {
            "workload": "kiss_fftr/kiss_fftri batched real float32, N=4096 and N=4000, 65536 signals each, "
                        "forward+inverse, N(0,1)+two tones, resident in HBM",
            "batch": BATCH,
            "nfft": list(SIZES),
        },
        "pct_hbm_peak": round(100 * value / HBM_PEAK_GBPS, 2),
        "other_configs": others,
        "serving": serve,
        "transforms_per_s": round(transforms_per_s, 1),
        "first_step_ms": round(first_step_s * 1e3, 1),
        "per_kernel": per_kernel,
        "roofline": {
            "bound": "hbm",
            "kernel": "forward real N=4096 (k_fast<F32, FK_R2C>: LDS-resident Stockham + real split)",
            "achieved": round(achieved, 1),
            "peak": HBM_PEAK_GBPS,
            "unit": "GB/s",
            "frac": round(achieved / HBM_PEAK_GBPS, 4),
            "traffic": traffic,
            "alg_bytes_per_launch": kbytes,
            "avg_launch_us": round(kern_s * 1e6, 2),
            "ceiling": ceil,
            "frac_of_rows_ceiling": round(achieved / ceil["r2c_rows_GBps"], 4) if ceil else None,
        },
        "cpu_baseline": cpu,
    }
    print(json.dumps(out), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
