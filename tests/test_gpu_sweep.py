"""GPU parity over a sweep of lengths, fixed point and float, complex and real.

Every length from 1 to 72 (complex) and every even length from 2 to 144 (real) plus lengths
with mixed and generic radices, each through one batched call of 3 transforms in both
directions: Q15 and Q31 bit-exact against the oracle (itself pinned bit-exact to the
reference build), float within the float bar of FP64.  The sweep reaches every kernel
family a length can fall to: the general line kernel (any radix, kf_bfly_generic for 7,
11, 13, ...), the compiled registry, and runtime-compiled kernels from 128 points up (144,
160, 400, 1331, 2310; KISSFFT_AMD_RTC_MIN=128 keeps the shorter lines on the general
kernel here).  test_short_lengths_compiled runs short lengths through the runtime-compiled
kernels they take by default (from 16 points).
"""
import sys

import numpy as np
import pytest

import kissfft_amd
from helpers import ABS_FLOAT_BOUND, cplx, rel_l2
from oracle import Oracle

pytestmark = pytest.mark.gpu

C2C_SIZES = list(range(1, 73)) + [77, 91, 96, 100, 121, 125, 143, 144, 160, 169, 243, 400, 1331, 2310]
REAL_SIZES = list(range(2, 145, 2)) + [154, 182, 200, 250, 338, 400, 486, 2310]
B = 3


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def rnd(rng, dtype, shape):
    if dtype == "float":
        return rng.uniform(-1, 1, shape).astype(np.float32)
    if dtype == "int16_t":
        return rng.integers(-32768, 32768, shape).astype(np.int16)
    return rng.integers(-(1 << 31), 1 << 31, shape, dtype=np.int64).astype(np.int32)


@pytest.fixture
def general_short(monkeypatch):
    monkeypatch.setenv("KISSFFT_AMD_RTC_MIN", "128")


@pytest.mark.parametrize("dtype", ["int16_t", "int32_t", "float"])
def test_c2c_length_sweep(dtype, general_short):
    lib = kissfft_amd.load(dtype)
    O = Oracle(dtype) if dtype != "float" else None
    rng = np.random.default_rng(71)
    worst = 0.0
    for n in C2C_SIZES:
        x = rnd(rng, dtype, (B, n, 2))
        for inv in (False, True):
            say("case sweep c2c", dtype, n, "inverse", inv)
            y = np.zeros_like(x)
            lib.fft_batch(lib.fft_alloc(n, inv), x, y, B, n, n)
            if O is not None:
                want = O.fft(x, inv)
                assert np.array_equal(y, want), f"{dtype} n={n} inverse={inv}: differs from the oracle"
            else:
                want = np.fft.ifft(cplx(x), axis=-1) * n if inv else np.fft.fft(cplx(x), axis=-1)
                err = rel_l2(cplx(y), want)
                worst = max(worst, err)
                assert err <= ABS_FLOAT_BOUND, (n, inv, err)
    say("worst float rel-L2", worst)


@pytest.mark.parametrize("dtype", ["int16_t", "int32_t", "float"])
def test_real_length_sweep(dtype, general_short):
    lib = kissfft_amd.load(dtype)
    O = Oracle(dtype) if dtype != "float" else None
    rng = np.random.default_rng(72)
    worst = 0.0
    for n in REAL_SIZES:
        say("case sweep real", dtype, n)
        x = rnd(rng, dtype, (B, n))
        X = np.zeros((B, n // 2 + 1, 2), lib.scalar)
        lib.fftr_batch(lib.fftr_alloc(n, False), x, X, B, n, n // 2 + 1)
        Z = rnd(rng, dtype, (B, n // 2 + 1, 2))
        z = np.zeros((B, n), lib.scalar)
        lib.fftri_batch(lib.fftr_alloc(n, True), Z, z, B, n // 2 + 1, n)
        if O is not None:
            assert np.array_equal(X, O.fftr(x)), f"{dtype} n={n}: forward differs from the oracle"
            assert np.array_equal(z, O.fftri(Z, n)), f"{dtype} n={n}: inverse differs from the oracle"
        else:
            err = rel_l2(cplx(X), np.fft.rfft(x.astype(np.float64), axis=-1))
            # kiss_fftri ignores the imaginary parts of the DC and Nyquist bins (kiss_fftr.c:131-134)
            zc = cplx(Z)
            zc[..., 0] = zc[..., 0].real
            zc[..., -1] = zc[..., -1].real
            erri = rel_l2(z.astype(np.float64), np.fft.irfft(zc, n, axis=-1) * n)
            worst = max(worst, err, erri)
            assert err <= ABS_FLOAT_BOUND and erri <= ABS_FLOAT_BOUND, (n, err, erri)
    say("worst float rel-L2", worst)


SHORT_C2C = [16, 20, 36, 49, 60, 77, 100, 121, 126]
SHORT_REAL = [32, 40, 98, 120, 154]


@pytest.mark.parametrize("dtype", ["int16_t", "int32_t", "float"])
def test_short_lengths_compiled(dtype, monkeypatch, capfd):
    """Short lines (16 to 127 points) on the kernels compiled at run time by default:
    bit-exact against the oracle in fixed point, within the float bar of FP64."""
    monkeypatch.setenv("KISSFFT_AMD_VERBOSE", "1")
    lib = kissfft_amd.load(dtype)
    lib.L.kiss_fft_cleanup()  # kernel choices made afresh (and reported) for these lengths
    O = Oracle(dtype) if dtype != "float" else None
    rng = np.random.default_rng(73)
    for n in SHORT_C2C:
        x = rnd(rng, dtype, (17, n, 2))
        for inv in (False, True):
            say("case short c2c", dtype, n, "inverse", inv)
            y = np.zeros_like(x)
            lib.fft_batch(lib.fft_alloc(n, inv), x, y, 17, n, n)
            if O is not None:
                assert np.array_equal(y, O.fft(x, inv)), f"{dtype} n={n} inverse={inv}"
            else:
                want = np.fft.ifft(cplx(x), axis=-1) * n if inv else np.fft.fft(cplx(x), axis=-1)
                assert rel_l2(cplx(y), want) <= ABS_FLOAT_BOUND, (n, inv)
    for n in SHORT_REAL:
        say("case short real", dtype, n)
        x = rnd(rng, dtype, (17, n))
        X = np.zeros((17, n // 2 + 1, 2), lib.scalar)
        lib.fftr_batch(lib.fftr_alloc(n, False), x, X, 17, n, n // 2 + 1)
        if O is not None:
            assert np.array_equal(X, O.fftr(x)), f"{dtype} n={n}"
        else:
            assert rel_l2(cplx(X), np.fft.rfft(x.astype(np.float64), axis=-1)) <= ABS_FLOAT_BOUND, n
    err = capfd.readouterr().err
    assert "fast variant rtc_c2c60" in err and "fast variant rtc_r2c49" in err, err[-2000:]


@pytest.mark.parametrize("n", [2049, 2176, 2201, 3077, 3162, 3751, 4096 + 1, 4099, 4301, 5002, 6800, 8167, 8191])
def test_float_lengths_above_2048_with_large_primes(n):
    """Lengths with prime factors above 13 past 2048 points: factors of 17 .. 31 on rows
    compiled at run time, above 50 on Bluestein's kernel (8192 and 16384 points)."""
    lib = kissfft_amd.load("float")
    x = np.random.default_rng(n).uniform(-1, 1, (3, n, 2)).astype(np.float32)
    for inv in (False, True):
        y = np.zeros_like(x)
        lib.fft_batch(lib.fft_alloc(n, inv), x, y, 3, n, n)
        z = x[..., 0] + 1j * x[..., 1].astype(np.float64)
        want = np.fft.ifft(z, axis=-1) * n if inv else np.fft.fft(z, axis=-1)
        got = y[..., 0] + 1j * y[..., 1].astype(np.float64)
        assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want), (n, inv)


@pytest.mark.parametrize("n", [2 * 53, 2 * 68, 2 * 563, 2 * 899, 2 * 1009, 2 * 2047, 2 * 3162, 2 * 4099, 2 * 8191])
def test_float_real_rows_with_large_primes(n):
    """Real rows whose half length has prime factors above 13: to 31 on compiled rows, above
    50 on Bluestein's kernel with the split / merge as a pass of its own; in place too."""
    import torch
    lib = kissfft_amd.load("float")
    x = np.random.default_rng(n).standard_normal((5, n)).astype(np.float32)
    X = np.zeros((5, n // 2 + 1, 2), np.float32)
    lib.fftr_batch(lib.fftr_alloc(n), x, X, 5, n, n // 2 + 1)
    want = np.fft.rfft(x.astype(np.float64), axis=-1)
    assert rel_l2(cplx(X), want) <= ABS_FLOAT_BOUND
    z = np.zeros_like(x)
    lib.fftri_batch(lib.fftr_alloc(n, True), X, z, 5, n // 2 + 1, n)
    assert rel_l2(z, n * x.astype(np.float64)) <= 2 * ABS_FLOAT_BOUND
    one = torch.zeros(n + 2, device="cuda")
    one[:n] = torch.from_numpy(x[0]).cuda()
    torch.cuda.synchronize()
    lib.kiss_fftr(lib.fftr_alloc(n), one, one)
    np.testing.assert_array_equal(one.cpu().numpy().reshape(-1, 2), X[0])


@pytest.mark.parametrize("n", [1007, 2014, 4028, 4081, 7950, 8109, 8162])
def test_factor_53_is_as_exact_as_direct_sums(n):
    """Lengths with a factor of 53 in a nearly full convolution keep direct sums, summed in FP64:
    a stage rounds its inputs' twiddle products and its result, so 3 or 4 stages stay within
    sqrt(2 * 4) * 2^-24 * 0.6 = 1.0e-7; 1.5e-7 leaves half as much again.  Float sums are at
    1.7e-7 and Bluestein's convolution at 1.9e-7.  Real rows of this half length, and complex
    lines of it above 2048 points."""
    lib = kissfft_amd.load("float")
    rng = np.random.default_rng(n)
    x = rng.standard_normal((16, 2 * n)).astype(np.float32)
    X = np.zeros((16, n + 1, 2), np.float32)
    lib.fftr_batch(lib.fftr_alloc(2 * n), x, X, 16, 2 * n, n + 1)
    assert rel_l2(cplx(X), np.fft.rfft(x.astype(np.float64), axis=-1)) <= 1.5e-7
    if n <= 2048:
        return
    z = x.reshape(16, n, 2)
    for inv in (False, True):
        y = np.zeros_like(z)
        lib.fft_batch(lib.fft_alloc(n, inv), z, y, 16, n, n)
        want = np.fft.ifft(cplx(z), axis=-1) * n if inv else np.fft.fft(cplx(z), axis=-1)
        assert rel_l2(cplx(y), want) <= 1.5e-7, inv


def test_tables_made_under_capture():
    """A call captured on a blocking stream whose length needs tables that no call has made yet
    (4093: Bluestein's): they are uploaded without ending the capture, and every replay
    gives the transform of the input of that moment."""
    import torch
    n, b = 4093, 4
    lib = kissfft_amd.load("float")
    lib.L.kiss_fft_cleanup()
    x = torch.from_numpy(np.random.default_rng(n).uniform(-1, 1, (b, n, 2)).astype(np.float32)).cuda()
    y = torch.empty_like(x)
    cfg, st, g = lib.fft_alloc(n), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    lib.fft_batch(cfg, x, y, 0, n, n)  # (the device plan alone)
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=st, capture_error_mode="thread_local"):
        lib.fft_batch(cfg, x, y, b, n, n, stream=st)
    for rep in range(3):
        x.mul_(1.25).add_(0.25)
        y.fill_(9.0)
        torch.cuda.synchronize()
        with torch.cuda.stream(st):
            g.replay()
        torch.cuda.synchronize()
        assert rel_l2(cplx(y.cpu().numpy()), np.fft.fft(cplx(x.cpu().numpy()), axis=-1)) <= ABS_FLOAT_BOUND, rep


@pytest.mark.parametrize("n,path", [(2176, "fast variant rtc_c2c2176"), (3162, "fast variant rtc_c2c3162"), (2809, "Bluestein blue8192"),
                                    (4093, "Bluestein blue8192"), (5002, "Bluestein blue16384"), (8191, "Bluestein blue16384")])
def test_large_prime_lengths_take_their_path(n, path, monkeypatch, capfd):
    """Above 2048 points: rows compiled for factors of 17 .. 31, Bluestein's kernel for larger
    ones where it is exact enough (2809 = 53^2 in a convolution 0.69 full)."""
    lib = kissfft_amd.load("float")
    monkeypatch.setenv("KISSFFT_AMD_VERBOSE", "1")
    lib.L.kiss_fft_cleanup()
    x = np.random.default_rng(n).uniform(-1, 1, (2, n, 2)).astype(np.float32)
    y = np.zeros_like(x)
    lib.fft_batch(lib.fft_alloc(n), x, y, 2, n, n)
    assert rel_l2(cplx(y), np.fft.fft(cplx(x), axis=-1)) <= ABS_FLOAT_BOUND
    assert path in capfd.readouterr().err
