"""GPU tests of multi-pass lines whose two passes run on tile kernels compiled at run time.

Float lengths without a built-in four-step split (kfa_engine.hip bailey_plan), and the
fixed-point builds' reference-order split, whose second pass reads its own rows of the
full-length twiddle tables (TM_REF in kfa_tile.hpp).  Fixed point is bit-exact against the
oracle, float within the float bar of FP64; contiguous and strided input, both directions.
"""
import os
import re
import subprocess
import sys

import numpy as np
import pytest

import kissfft_amd
from conftest import ROOT
from helpers import ABS_FLOAT_BOUND, cplx, rel_l2
from oracle import Oracle

pytestmark = pytest.mark.gpu

# halves of equal and of very different radices, odd lengths, a generic radix, a half with
# component-wise hand-overs
LENGTHS = [18750, 19683, 16807 * 2, 65536, 98304, 118098, 218700, 2 ** 18 * 3]


def rnd(rng, dtype, shape):
    if dtype == "float":
        return rng.uniform(-1, 1, shape).astype(np.float32)
    if dtype == "int16_t":
        return rng.integers(-32768, 32768, shape).astype(np.int16)
    return rng.integers(-(1 << 31), 1 << 31, shape, dtype=np.int64).astype(np.int32)


@pytest.mark.parametrize("dtype", ["float", "int16_t", "int32_t"])
@pytest.mark.parametrize("n", LENGTHS)
def test_two_pass_lines(n, dtype, monkeypatch, capfd):
    lib = kissfft_amd.load(dtype)
    monkeypatch.setenv("KISSFFT_AMD_VERBOSE", "1")
    lib.L.kiss_fft_cleanup()
    b = 3
    x = rnd(np.random.default_rng(n), dtype, (b, n, 2))
    for inv in (False, True):
        print("case", dtype, n, inv, flush=True)
        y = np.zeros_like(x)
        lib.fft_batch(lib.fft_alloc(n, inv), x, y, b, n, n)
        if dtype == "float":
            want = np.fft.ifft(cplx(x), axis=-1) * n if inv else np.fft.fft(cplx(x), axis=-1)
            assert rel_l2(cplx(y), want) <= ABS_FLOAT_BOUND
        else:
            np.testing.assert_array_equal(y, Oracle(dtype).fft(x, inv))
    xs = rnd(np.random.default_rng(n + 1), dtype, (1, 2 * n, 2))  # every other element
    ys = np.zeros((1, n, 2), lib.scalar)
    lib.fft_batch(lib.fft_alloc(n), xs, ys, 1, 2 * n, n, in_stride=2)
    xd = np.ascontiguousarray(xs[:, ::2])
    if dtype == "float":
        assert rel_l2(cplx(ys), np.fft.fft(cplx(xd), axis=-1)) <= ABS_FLOAT_BOUND
    else:
        np.testing.assert_array_equal(ys, Oracle(dtype).fft(xd))
    assert "tile" in capfd.readouterr().err


def float_error(y, x):
    return rel_l2(cplx(y), np.fft.fft(cplx(x), axis=-1))


# 96 x 512 and 96 x 1024: built-in halves, less balanced than a split that can be compiled
@pytest.mark.parametrize("n", [49152, 98304])
def test_builtin_split_without_the_compiler(n, monkeypatch, capfd):
    """With the runtime compiler off a length whose preferred split would be compiled runs its
    built-in one, not the general kernel."""
    lib = kissfft_amd.load("float")
    x = rnd(np.random.default_rng(n), "float", (2, n, 2))
    y = np.zeros_like(x)
    monkeypatch.setenv("KISSFFT_AMD_VERBOSE", "1")
    monkeypatch.setenv("KISSFFT_AMD_RTC", "0")
    lib.L.kiss_fft_cleanup()
    try:
        lib.fft_batch(lib.fft_alloc(n), x, y, 2, n, n)
    finally:
        lib.L.kiss_fft_cleanup()
    assert float_error(y, x) <= ABS_FLOAT_BOUND
    split = re.findall(rf"four-step n={n} inverse=0: columns h?tile(\d+)_\S+, rows h?tile(\d+)_", capfd.readouterr().err)
    assert len(split) == 1 and int(split[0][0]) * int(split[0][1]) == n, split


def test_captured_first_call_runs_the_builtin_split(monkeypatch, capfd):
    """A first call under capture compiles nothing: it takes the built-in split, and a later
    eager call still gets the compiled one.  Every replay, also after that call, gives the
    transform of the input of that moment."""
    import torch
    n, b = 98304, 2
    lib = kissfft_amd.load("float")
    monkeypatch.setenv("KISSFFT_AMD_VERBOSE", "1")
    lib.L.kiss_fft_cleanup()
    x = torch.from_numpy(rnd(np.random.default_rng(5), "float", (b, n, 2))).cuda()
    y, z = torch.empty_like(x), torch.empty_like(x)
    cfg, st, g = lib.fft_alloc(n), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    lib.fft_batch(lib.fft_alloc(65536), x, y, 1, 65536, 65536)  # (the pool of captured temporaries)
    lib.fft_batch(cfg, x, y, 0, n, n)  # (the device plan alone)
    capfd.readouterr()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=st, capture_error_mode="thread_local"):
        lib.fft_batch(cfg, x, y, b, n, n, stream=st)
    err = capfd.readouterr().err
    assert re.search(rf"four-step n={n} inverse=0: columns h?tile\d+_\S+, rows h?tile\d+_", err), err
    for rep in range(3):
        x.mul_(1.25).add_(0.25)
        y.fill_(9.0)
        torch.cuda.synchronize()
        with torch.cuda.stream(st):
            g.replay()
        torch.cuda.synchronize()
        assert float_error(y.cpu().numpy(), x.cpu().numpy()) <= ABS_FLOAT_BOUND, rep
        lib.fft_batch(cfg, x, z, b, n, n)
        assert float_error(z.cpu().numpy(), x.cpu().numpy()) <= ABS_FLOAT_BOUND, rep
    assert re.search(rf"four-step n={n} inverse=0: columns .*rtc_tile", capfd.readouterr().err)


CAPTURED = """
import numpy as np, torch, kissfft_amd
n, b = 65536, 3
lib = kissfft_amd.load("int16_t")
x = torch.from_numpy(np.random.default_rng(1).integers(-9999, 9999, (b, n, 2)).astype(np.int16)).cuda()
y, want = torch.empty_like(x), torch.empty_like(x)
cfg, st, g = lib.fft_alloc(n), torch.cuda.Stream(), torch.cuda.CUDAGraph()
lib.fft_batch(cfg, x, want, b, n, n)
torch.cuda.synchronize()
with torch.cuda.graph(g, stream=st, capture_error_mode="thread_local"):
    lib.fft_batch(cfg, x, y, b, n, n, stream=st)
for rep in range(3):
    x.add_(7)
    lib.fft_batch(cfg, x, want, b, n, n)
    y.zero_()
    torch.cuda.synchronize()
    with torch.cuda.stream(st):
        g.replay()
    torch.cuda.synchronize()
    assert torch.equal(y, want), rep
print("same")
"""


def test_capture_after_one_eager_call():
    """In a fresh process one eager call is all the preparation that a captured call of the same
    kind needs: its temporary comes from the graph's pool, which no call has used before."""
    r = subprocess.run([sys.executable, "-c", CAPTURED], capture_output=True, text=True, timeout=110, cwd=ROOT,
                       env=dict(os.environ, PYTHONPATH=ROOT))
    assert r.returncode == 0 and "same" in r.stdout, r.stderr[-2000:]


@pytest.mark.parametrize("dtype", ["float", "int16_t", "int32_t"])
@pytest.mark.parametrize("n", [18750, 19683, 65536, 98304, 2 ** 18 * 3])
def test_both_passes_run_on_tiles(n, dtype, monkeypatch, capfd):
    """The engine reports a pair of tiles only when both are there, and then runs both: two
    lines of its report per fixed-point plan, one naming both tiles per float plan."""
    lib = kissfft_amd.load(dtype)
    monkeypatch.setenv("KISSFFT_AMD_VERBOSE", "1")
    lib.L.kiss_fft_cleanup()
    x = rnd(np.random.default_rng(n), dtype, (1, n, 2))
    for inv in (False, True):
        capfd.readouterr()
        lib.fft_batch(lib.fft_alloc(n, inv), x, np.zeros_like(x), 1, n, n)
        err = capfd.readouterr().err
        if dtype == "float":
            assert len(re.findall(rf"four-step n={n} inverse={int(inv)}: columns \S*tile\S+, rows \S*tile", err)) == 1, err
        else:
            halves = [int(h) for h in re.findall(rf"tile n=(\d+) of {n} inverse={int(inv)} ", err)]
            assert len(halves) == 2 and halves[0] * halves[1] == n, err
