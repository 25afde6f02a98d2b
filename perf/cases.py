"""Performance cases: what programs run this library for, through its public entry points.

The library replaces KISS FFT's C API on one GPU, so the cases are its callers' work:
batches of complex and real 1-D transforms resident in HBM (the batched, asynchronous
calls), N-D transforms, lines longer than one workgroup holds, the two fixed-point builds,
prime lengths, a list of uneven batches run as one multi-batch, a long signal through the
fast FIR filter, and the reference's own call on host memory.

A case is a dict of plain values:
    op      c2c | r2c | c2r       batched 1-D transforms
            nd                    complex N-D transforms
            ndr                   a real N-D transform and its inverse, one after the other
            multi                 a list of uneven batches in one launch sequence
            fir                   overlap-scrap FIR filter of one long real or complex signal
            host                  kiss_fft / kiss_fftr on one line of host memory
    dtype   float | int16_t (Q15) | int32_t (Q31)
    n, batch, inverse, stride, dims ("64x96x120"), taps, items, seed, graph, real

Inputs: float lines are Gaussian noise, Q15 and Q31 lines are uniform over half the
scalar's range (what the fixed-point transforms, which divide by the radix at every stage,
are fed), real spectra are Hermitian-consistent at DC and Nyquist.
"""
import math
import random

import numpy as np
import torch

import kissfft_amd

_TORCH = {"float": torch.float32, "int16_t": torch.int16, "int32_t": torch.int32}
_BYTES = {"float": 4, "int16_t": 2, "int32_t": 4}


def _dims(case):
    return tuple(int(d) for d in case["dims"].split("x"))


def listed():
    return [
        # A small batch of one length, called again and again: the latency of a launch and
        # of one line through a workgroup.
        dict(name="c2c_1200_b256", op="c2c", dtype="float", n=1200, batch=256, inverse=False, stride=1),
        # The reference's own call, unchanged: one line of host memory, result valid on return.
        dict(name="host_c2c_1024", op="host", dtype="float", n=1024, real=False),
        # Real signals to spectra and back, as many as fill the card: the throughput cases.
        dict(name="r2c_4096_b65536", op="r2c", dtype="float", n=4096, batch=65536),
        dict(name="c2r_4000_b65536", op="c2r", dtype="float", n=4000, batch=65536),
        # Q15 lines, the fixed-point build's usual length.
        dict(name="q15_c2c_512_b1m", op="c2c", dtype="int16_t", n=512, batch=1 << 20, inverse=False, stride=1),
        # A prime length: no radix of the schedule divides it.
        dict(name="c2c_1009_b4096", op="c2c", dtype="float", n=1009, batch=4096, inverse=False, stride=1),
        # A batch of 3-D arrays, complex.
        dict(name="nd_64x96x120_b16", op="nd", dtype="float", dims="64x96x120", batch=16, inverse=False),
        # Real images to spectra and back, as a 2-D filter does.
        dict(name="ndr_1024x1000_b32", op="ndr", dtype="float", dims="1024x1000", batch=32),
        # Lines too long for one workgroup.
        dict(name="c2c_1m_b64", op="c2c", dtype="float", n=1 << 20, batch=64, inverse=False, stride=1),
        # 3-D arrays in the Q15 build.
        dict(name="q15_nd_64x96x120_b16", op="nd", dtype="int16_t", dims="64x96x120", batch=16, inverse=False),
        # 64 uneven batches of eight kinds and lengths, replayed from a graph.
        dict(name="multi_64", op="multi", dtype="float", items=64, seed=11, graph=True),
        # A recorded signal of 2^26 real samples through a 1000-tap filter.
        dict(name="fir_1000_2p26", op="fir", dtype="float", n=1 << 26, taps=1000, real=True),
    ]


# ---- drawn cases -------------------------------------------------------------------------


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth(n, odd=False):
    """The next length not below n whose factors are 2, 3 and 5 (odd: 3 and 5)."""
    while True:
        m = n
        for p in (3, 5) if odd else (2, 3, 5):
            while m % p == 0:
                m //= p
        if m == 1:
            return n
        n += 1


def _length(rng, lo, hi):
    """Mostly lengths as kiss_fft_next_fast_size gives them, a third powers of two."""
    n = _log(rng, lo, hi)
    if rng.random() < 0.33:
        return 1 << max(1, round(math.log2(n)))
    return min(_smooth(n, odd=rng.random() < 0.15), 1 << 21)


_MAX_POINTS = 1 << 27  # complex float values of one side: 1 GiB


def _batch(rng, points, top=_MAX_POINTS):
    most = max(1, top // points)
    return max(1, min(most, _log(rng, 1, most + 1)))


def _fixed(rng):
    return rng.choice(["int16_t", "int32_t"])


def draw(rng):
    op = rng.choice(["c2c", "c2c", "real", "real", "fixed", "odd", "long", "long", "nd", "nd", "ndr", "ndr",
                     "multi", "fir", "host"])
    if op == "c2c":
        n = _length(rng, 16, 8192)
        return dict(op="c2c", dtype="float", n=n, batch=_batch(rng, n), inverse=rng.random() < 0.5,
                    stride=rng.choice([1, 1, 1, 1, 1, 2]))
    if op == "real":
        n = 2 * _length(rng, 16, 8192)
        dtype = rng.choice(["float", "float", "float", "int16_t", "int32_t"])
        return dict(op=rng.choice(["r2c", "c2r"]), dtype=dtype, n=n, batch=_batch(rng, n // 2))
    if op == "fixed":
        n = _length(rng, 16, 8192)
        return dict(op="c2c", dtype=_fixed(rng), n=n, batch=_batch(rng, n), inverse=rng.random() < 0.5, stride=1)
    if op == "odd":  # any length at all, primes among them
        n = _log(rng, 17, 4096)
        return dict(op="c2c", dtype="float", n=n, batch=_batch(rng, n, 1 << 23), inverse=rng.random() < 0.5, stride=1)
    if op == "long":
        n = _length(rng, 1 << 14, 1 << 21)
        kind = rng.choice(["c2c", "c2c", "r2c", "c2r"])
        dtype = rng.choice(["float", "float", "float", "int16_t", "int32_t"])
        if kind == "c2c":
            return dict(op="c2c", dtype=dtype, n=n, batch=_batch(rng, n, 1 << 26), inverse=rng.random() < 0.5,
                        stride=1)
        return dict(op=kind, dtype=dtype, n=2 * n, batch=_batch(rng, n, 1 << 26))
    if op in ("nd", "ndr"):
        k = rng.choice([2, 2, 3])
        dims = [_length(rng, 12, 1200 if k == 2 else 160) for _ in range(k)]
        if op == "ndr":
            dims[-1] += dims[-1] % 2
        dtype = rng.choice(["float", "float", "float", "int16_t", "int32_t"])
        case = dict(op=op, dtype=dtype, dims="x".join(map(str, dims)), batch=_batch(rng, math.prod(dims), 1 << 25))
        return dict(case, inverse=rng.random() < 0.5) if op == "nd" else case
    if op == "multi":
        return dict(op="multi", dtype="float", items=rng.randint(4, 48), seed=rng.randrange(1, 1 << 20),
                    graph=rng.random() < 0.7)
    if op == "fir":
        return dict(op="fir", dtype="float", n=_log(rng, 1 << 16, 1 << 25), taps=_log(rng, 16, 2000),
                    real=rng.random() < 0.7)
    return dict(op="host", dtype="float", n=2 * _length(rng, 8, 16384), real=rng.random() < 0.5)


# ---- inputs --------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _signal(dtype, shape, seed):
    """Gaussian noise (float) or uniform integers, `shape` scalars on the GPU."""
    g = _gen(seed)
    if dtype == "float":
        return torch.randn(shape, generator=g, device="cuda")
    half = 1 << (14 if dtype == "int16_t" else 30)
    return torch.randint(-half, half, shape, generator=g, device="cuda", dtype=_TORCH[dtype])


def _spectrum(dtype, shape, seed):
    """(..., bins, 2): spectra of real lines, DC and Nyquist real."""
    x = _signal(dtype, shape, seed)
    x[..., 0, 1] = 0
    x[..., -1, 1] = 0
    return x


# The lengths of a multi-batch: the eight kinds of the uneven workload.
_MENU = (("c2c", 256), ("c2c", 1000), ("c2c", 1009), ("c2c", 1200), ("c2c_inv", 3072), ("r2c", 4096), ("c2r", 4000),
         ("c2c", 120))


def _multi_items(case):
    """(kind, n, count) of every batch; counts log-uniform in [1, 512]."""
    r = random.Random(case["seed"])
    out = []
    for i in range(case["items"]):
        kind, n = _MENU[i % len(_MENU)]
        out.append((kind, n, int(math.exp(r.uniform(0, math.log(512))))))
    return out


def _multi_buffers(case, seed):
    """Input tensors of every batch."""
    ins = []
    for i, (kind, n, count) in enumerate(_multi_items(case)):
        s = seed * 64 + i
        if kind == "r2c":
            ins.append(_signal("float", (count, n), s))
        elif kind == "c2r":
            ins.append(_spectrum("float", (count, n // 2 + 1, 2), s))
        else:
            ins.append(_signal("float", (count, n, 2), s))
    return ins


def _input(case, seed):
    """The input array of every op but multi and host, on the GPU."""
    op, dtype = case["op"], case["dtype"]
    if op == "c2c":
        return _signal(dtype, (case["batch"], case["n"] * case["stride"], 2), seed)
    if op == "r2c":
        return _signal(dtype, (case["batch"], case["n"]), seed)
    if op == "c2r":
        return _spectrum(dtype, (case["batch"], case["n"] // 2 + 1, 2), seed)
    if op == "nd":
        return _signal(dtype, (case["batch"],) + _dims(case) + (2,), seed)
    if op == "ndr":
        return _signal(dtype, (case["batch"],) + _dims(case), seed)
    return _signal(dtype, (case["n"],) if case["real"] else (case["n"], 2), seed)  # fir


def _taps(case, seed):
    """A decaying random impulse response on the host."""
    r = np.random.default_rng(seed)
    nh = case["taps"]
    h = r.standard_normal((nh,) if case["real"] else (nh, 2))
    return (h.T * np.exp(-2.0 * np.arange(nh) / nh)).T.astype(np.float32)


def _host_line(case, seed):
    r = np.random.default_rng(seed)
    return r.standard_normal((case["n"],) if case["real"] else (case["n"], 2)).astype(np.float32)


def prepare(case, seed):
    lib = kissfft_amd.load(case["dtype"])
    op, dtype = case["op"], case["dtype"]
    s = dict(case=case, lib=lib)
    if op == "host":
        n = case["n"]
        s["x"] = _host_line(case, seed)
        s["y"] = np.empty((n // 2 + 1 if case["real"] else n, 2), np.float32)
        s["cfg"] = lib.fftr_alloc(n) if case["real"] else lib.fft_alloc(n)
        return s
    s["stream"] = torch.cuda.Stream()
    if op == "multi":
        M = kissfft_amd.MultiBatch
        kinds = {"c2c": M.C2C_FWD, "c2c_inv": M.C2C_INV, "r2c": M.R2C, "c2r": M.C2R}
        s["y"], items = [], []
        for (kind, n, count), x in zip(_multi_items(case), _multi_buffers(case, seed)):
            shape = {"r2c": (count, n // 2 + 1, 2), "c2r": (count, n)}.get(kind, (count, n, 2))
            y = torch.empty(shape, device="cuda")
            s["y"].append(y)
            items.append((kinds[kind], n, x, y, count))
        torch.cuda.synchronize()
        s["multi"] = lib.multi(items)
        if case["graph"]:
            s["multi"].capture(s["stream"])
        return s
    x = s["x"] = _input(case, seed)
    new = lambda shape: torch.empty(shape, dtype=_TORCH[dtype], device="cuda")  # noqa: E731
    if op == "c2c":
        s["cfg"] = lib.fft_alloc(case["n"], case["inverse"])
        s["y"] = new((case["batch"], case["n"], 2))
    elif op == "r2c":
        s["cfg"] = lib.fftr_alloc(case["n"])
        s["y"] = new((case["batch"], case["n"] // 2 + 1, 2))
    elif op == "c2r":
        s["cfg"] = lib.fftr_alloc(case["n"], True)
        s["y"] = new((case["batch"], case["n"]))
    elif op == "nd":
        s["cfg"] = lib.fftnd_alloc(_dims(case), case["inverse"])
        s["y"] = torch.empty_like(x)
    elif op == "ndr":
        d = _dims(case)
        s["cfg"], s["inv"] = lib.fftndr_alloc(d), lib.fftndr_alloc(d, True)
        s["y"] = new((case["batch"],) + d[:-1] + (d[-1] // 2 + 1, 2))
        s["z"] = torch.empty_like(x)
    else:  # fir
        s["fir"] = lib.fastfir_alloc(_taps(case, seed), real=case["real"])
        s["y"] = torch.empty_like(x)
    torch.cuda.synchronize()  # the inputs are there before another stream reads them
    return s


def run(s):
    case, lib = s["case"], s["lib"]
    op = case["op"]
    if op == "c2c":
        n = case["n"]
        lib.fft_batch(s["cfg"], s["x"], s["y"], case["batch"], n * case["stride"], n, in_stride=case["stride"],
                      stream=s["stream"])
    elif op == "r2c":
        n = case["n"]
        lib.fftr_batch(s["cfg"], s["x"], s["y"], case["batch"], n, n // 2 + 1, stream=s["stream"])
    elif op == "c2r":
        n = case["n"]
        lib.fftri_batch(s["cfg"], s["x"], s["y"], case["batch"], n // 2 + 1, n, stream=s["stream"])
    elif op == "nd":
        lib.fftnd_batch(s["cfg"], s["x"], s["y"], case["batch"], stream=s["stream"])
    elif op == "ndr":
        lib.fftndr_batch(s["cfg"], s["x"], s["y"], case["batch"], stream=s["stream"])
        lib.fftndri_batch(s["inv"], s["y"], s["z"], case["batch"], stream=s["stream"])
        return s["y"], s["z"]
    elif op == "multi":
        if case["graph"]:
            s["multi"].replay(s["stream"])
        else:
            s["multi"].exec(s["stream"])
        return s["y"]
    elif op == "fir":
        # one whole recording per pass; the call returns with its result in place and moves
        # the samples it did not use to the front of the input, as the reference's does
        s["fir"].offset = 0
        return s["y"][: s["fir"].filter(s["x"], s["y"], case["n"])]
    elif case["real"]:
        lib.kiss_fftr(s["cfg"], s["x"], s["y"])
    else:
        lib.kiss_fft(s["cfg"], s["x"], s["y"])
    return s["y"]


# ---- what a pass cannot do without ---------------------------------------------------------


def _line_work(kind, n, count, scalar=4):
    """(bytes, flops) of `count` transforms of length n: input once, output once."""
    cpx, half = 2 * scalar * n, 2 * scalar * (n // 2 + 1)
    if kind in ("r2c", "c2r"):
        return count * (scalar * n + half), count * 2.5 * n * math.log2(max(2, n))
    return count * 2 * cpx, count * 5.0 * n * math.log2(max(2, n))


def work(case):
    op, scalar = case["op"], _BYTES[case["dtype"]]
    if op in ("c2c", "r2c", "c2r"):
        b, f = _line_work(op, case["n"], case["batch"], scalar)
    elif op == "nd":
        tot = math.prod(_dims(case)) * case["batch"]
        b, f = 4 * scalar * tot, 5.0 * tot * math.log2(math.prod(_dims(case)))
    elif op == "ndr":
        d = _dims(case)
        tot = math.prod(d) * case["batch"]
        bins = tot // d[-1] * (d[-1] // 2 + 1)
        b, f = 2 * scalar * (tot + 2 * bins), 5.0 * tot * math.log2(math.prod(d))
    elif op == "multi":
        b = f = 0
        for kind, n, count in _multi_items(case):
            w = _line_work(kind, n, count)
            b, f = b + w[0], f + w[1]
    elif op == "fir":
        c = 1 if case["real"] else 2
        b = 2 * scalar * c * case["n"] + 4 * c * case["taps"]
        f = case["n"] * c * 5.0 * math.log2(4 * case["taps"])
    else:
        b, f = _line_work("r2c" if case["real"] else "c2c", case["n"], 1, scalar)
    return {"bytes": b, "flops": f}


# ---- the same in 64 bits, from torch on the CPU ----------------------------------------------


def _cpx64(x):
    return torch.view_as_complex(x.double().cpu().contiguous())


def _pairs(z):
    return torch.view_as_real(z.resolve_conj().contiguous())


def _line_exact(kind, x, n):
    if kind == "r2c":
        return _pairs(torch.fft.rfft(x.double().cpu(), dim=-1))
    if kind == "c2r":
        return torch.fft.irfft(_cpx64(x), n, dim=-1, norm="forward")
    f = torch.fft.ifft if kind == "c2c_inv" else torch.fft.fft
    return _pairs(f(_cpx64(x), dim=-1, norm="forward" if kind == "c2c_inv" else "backward"))


def _fir_exact(x, h, written):
    """The first `written` samples of the linear convolution's valid part, by blocks."""
    N, nh = 1 << 17, h.shape[-1]
    good = N - nh + 1
    H = torch.fft.fft(h, N)
    out = torch.empty(written, dtype=x.dtype)
    for b in range(0, written, good):
        seg = x[b:b + N]
        y = torch.fft.ifft(torch.fft.fft(seg, N) * H)[nh - 1:nh - 1 + min(good, written - b)]
        out[b:b + y.shape[0]] = y if x.is_complex() else y.real
    return out


def exact(case, seed):
    op = case["op"]
    if case["dtype"] != "float":
        return None  # whole numbers
    if op == "host":
        x = torch.from_numpy(_host_line(case, seed))
        return _line_exact("r2c" if case["real"] else "c2c", x, case["n"])
    if op == "multi":
        return [_line_exact(kind, x, n)
                for (kind, n, _), x in zip(_multi_items(case), _multi_buffers(case, seed))]
    x = _input(case, seed)
    if op == "c2c":
        x = x[:, ::case["stride"]]
        return _line_exact("c2c_inv" if case["inverse"] else "c2c", x, case["n"])
    if op in ("r2c", "c2r"):
        return _line_exact(op, x, case["n"])
    if op == "nd":
        axes = tuple(range(1, 1 + len(_dims(case))))
        z = _cpx64(x)
        return _pairs(torch.fft.ifftn(z, dim=axes, norm="forward") if case["inverse"] else torch.fft.fftn(z, dim=axes))
    if op == "ndr":
        axes = tuple(range(1, 1 + len(_dims(case))))
        d = x.double().cpu()
        return _pairs(torch.fft.rfftn(d, dim=axes)), d * float(math.prod(_dims(case)))
    nh = case["taps"]
    h = torch.from_numpy(_taps(case, seed))
    nfft = _fir_block(nh, case["real"])
    good = nfft - nh + 1
    written = ((case["n"] - nfft) // good + 1) * good
    if case["real"]:
        return _fir_exact(x.double().cpu(), h.double(), written)
    return _pairs(_fir_exact(_cpx64(x), torch.view_as_complex(h.double().contiguous()), written))


def _fir_block(nh, real):
    """The filter's default block: a power of two, at least twice the response, from 2048
    (real) or 1024 (complex)."""
    nfft, k = 2, nh - 1
    while True:
        nfft *= 2
        k >>= 1
        if not k:
            break
    return max(nfft, 2048 if real else 1024)
