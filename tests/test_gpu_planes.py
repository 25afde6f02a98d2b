"""GPU tests of plane kernels compiled at run time (kfa_plane.hpp, kfa_rtc.hip): the last two
axes of an N-D transform in one pass, all three scalar kinds.

Planes whose lines do not divide among the threads, odd and even row lengths, one-stage
axes, under 0 to 2 leading axes, in place too.  Fixed point transforms the columns first, as
kiss_fftnd's axis order requires (kiss_fftnd.c:150-188): bit-exact against the oracle.
Float is within the float bar of FP64.  The engine's report shows that the plane ran.
"""
import numpy as np
import pytest

import kissfft_amd
from helpers import ABS_FLOAT_BOUND, cplx, rel_l2
from oracle import Oracle

pytestmark = pytest.mark.gpu

SHAPES = [((2, 5), 130), ((12, 16), 3), ((25, 27), 129), ((30, 60), 2), ((40, 120), 128), ((80, 60), 130),
          ((3, 96, 50), 44), ((2, 2, 15, 100), 33), ((60, 5), 1), ((5, 375), 140)]


@pytest.mark.parametrize("dtype", ["float", "int16_t", "int32_t"])
@pytest.mark.parametrize("dims,b", SHAPES, ids=["x".join(map(str, s[0])) for s in SHAPES])
def test_compiled_planes(dims, b, dtype, monkeypatch, capfd):
    import torch
    lib = kissfft_amd.load(dtype)
    monkeypatch.setenv("KISSFFT_AMD_VERBOSE", "1")
    lib.L.kiss_fft_cleanup()
    rng = np.random.default_rng(b)
    shape = (b,) + dims + (2,)
    if dtype == "float":
        x = rng.uniform(-1, 1, shape).astype(np.float32)
    else:
        m = 1 << (15 if dtype == "int16_t" else 31)
        x = rng.integers(-m, m, shape, dtype=np.int64).astype(lib.scalar)
    for inv in (False, True):
        print("case", dtype, dims, b, inv, flush=True)
        y = np.zeros_like(x)
        cfg = lib.fftnd_alloc(dims, inv)
        lib.fftnd_batch(cfg, x, y, b)
        if dtype == "float":
            axes = tuple(range(1, len(dims) + 1))
            want = np.fft.ifftn(cplx(x), axes=axes) * np.prod(dims) if inv else np.fft.fftn(cplx(x), axes=axes)
            assert rel_l2(cplx(y), want) <= ABS_FLOAT_BOUND
        else:
            np.testing.assert_array_equal(y, Oracle(dtype).fftnd(x, dims, inv))
        d = torch.from_numpy(x).cuda()
        torch.cuda.synchronize()
        lib.fftnd_batch(cfg, d, d, b)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(d.cpu().numpy(), y)
    assert f"plane {dims[-2]}x{dims[-1]} " in capfd.readouterr().err


def test_few_planes_after_many():
    """A call of few planes takes the axis passes whatever ran before it: its launches and its
    bits are those of the same call in a fresh process, also after a batch of the same
    planes that is worth a compiled kernel."""
    lib = kissfft_amd.load("float")
    dims, many, few = (80, 60), 130, 4
    x = np.random.default_rng(3).uniform(-1, 1, (many,) + dims + (2,)).astype(np.float32)
    cfg = lib.fftnd_alloc(dims)

    def run(b):
        y = np.zeros_like(x[:b])
        n0 = lib.stats()["launches"]
        lib.fftnd_batch(cfg, x[:b], y, b)
        return y, lib.stats()["launches"] - n0

    lib.L.kiss_fft_cleanup()
    fresh, n_fresh = run(few)
    _, n_many = run(many)
    after, n_after = run(few)
    assert (n_fresh, n_many, n_after) == (2, 1, 2)
    np.testing.assert_array_equal(after, fresh)
