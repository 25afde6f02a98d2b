"""GPU tests of N-D axes on tile kernels compiled at run time (kfa_rtc.hip, kfa_tile.hpp).

Axes of lengths without a built-in tile, all three scalar kinds: one-stage lengths, odd
radices, butterflies that do not divide among the threads, lengths whose tiles hand one
component over at a time or take fewer lines, and column counts that leave the last tile
part empty or spread a tile over several slices.  Fixed point is bit-exact against the
oracle (kiss_fftnd.c:150-188 per axis), float within the float bar of FP64; the engine's
own report shows that a compiled tile ran.
"""
import sys

import numpy as np
import pytest

import kissfft_amd
from helpers import ABS_FLOAT_BOUND, cplx, rel_l2
from oracle import Oracle

pytestmark = pytest.mark.gpu

DIMS = [(5, 13000), (13, 33, 160), (25, 37), (45, 3, 50), (60, 36, 20), (77, 40), (120, 7), (243, 19), (375, 33),
        (540, 21), (625, 20), (720, 17), (1000, 9), (1250, 11), (2000, 5), (4096, 3), (7500, 3)]


def rnd(rng, dtype, shape):
    if dtype == "float":
        return rng.uniform(-1, 1, shape).astype(np.float32)
    if dtype == "int16_t":
        return rng.integers(-32768, 32768, shape).astype(np.int16)
    return rng.integers(-(1 << 31), 1 << 31, shape, dtype=np.int64).astype(np.int32)


@pytest.mark.parametrize("dtype", ["float", "int16_t", "int32_t"])
@pytest.mark.parametrize("dims", DIMS, ids=["x".join(map(str, d)) for d in DIMS])
def test_compiled_axes(dims, dtype, monkeypatch, capfd):
    lib = kissfft_amd.load(dtype)
    monkeypatch.setenv("KISSFFT_AMD_VERBOSE", "1")
    monkeypatch.setenv("KISSFFT_AMD_PLANE", "0")  # an axis each, also where a plane would do
    lib.L.kiss_fft_cleanup()
    x = rnd(np.random.default_rng(sum(dims)), dtype, (2,) + dims + (2,))
    for inv in (False, True):
        print("case", dtype, dims, inv, flush=True)
        sys.stdout.flush()
        y = np.zeros_like(x)
        lib.fftnd_batch(lib.fftnd_alloc(dims, inv), x, y, 2)
        if dtype == "float":
            axes = tuple(range(1, len(dims) + 1))
            want = np.fft.ifftn(cplx(x), axes=axes) * np.prod(dims) if inv else np.fft.fftn(cplx(x), axes=axes)
            assert rel_l2(cplx(y), want) <= ABS_FLOAT_BOUND
        else:
            np.testing.assert_array_equal(y, Oracle(dtype).fftnd(x, dims, inv))
    assert f"tile n={dims[0]} " in capfd.readouterr().err
