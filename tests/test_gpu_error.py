"""Errors of the mixed-radix lines and tiles, uniform and ragged, held to what
the lengths had when every twiddle was a table entry of its own.

The bounds are rel-L2 errors of Gaussian samples measured with that engine
(the two-buffer lines, four-steps and Bluestein passes these lines replaced),
plus 2 %: three standard deviations of an error estimated from 2^15 points."""
import ctypes

import numpy as np
import pytest

from gpu_util import run_plan

pytestmark = pytest.mark.gpu


def _samples(n, batch, prec):
    rng = np.random.default_rng(7 * 1000003 + n)
    return rng.standard_normal(2 * n * batch).astype(np.float32 if prec == "f32" else np.float64)


def _exact(x, n, prec):
    """FP64 spectrum of FP32 samples, the long-double one of FP64 samples."""
    real = np.float64 if prec == "f32" else np.longdouble
    z = x[0::2].astype(real) + 1j * x[1::2].astype(real)
    return np.fft.fft(z.reshape(-1, n), axis=1).reshape(-1)


def _error(y, want):
    d = y[0::2].astype(np.float64) + 1j * y[1::2].astype(np.float64) - want
    return float(np.sqrt((np.abs(d) ** 2).sum() / (np.abs(want) ** 2).sum()))


# lengths that were further off with FP32 products of table entries: as large
# batches run them, and as small ones do (shorter radices, tiles)
@pytest.mark.parametrize("few,bounds", [
    (False, {196: 9.79e-8, 288: 1.039e-7, 10125: 1.413e-7, 10240: 1.259e-7, 14000: 1.354e-7, 20000: 1.420e-7,
             20160: 1.399e-7, 196608: 1.543e-7}),
    (True, {216: 1.059e-7, 252: 1.073e-7, 14000: 1.354e-7, 15000: 1.436e-7, 16000: 1.330e-7, 80000: 1.517e-7,
            100000: 1.629e-7})])
def test_f32_lines_and_tiles(pkg, dev, few, bounds, monkeypatch):
    monkeypatch.setenv("NFFT_FEW", "1" if few else "0")
    over = {}
    for n, bound in bounds.items():
        batch = max(3, 32768 // n)
        x = _samples(n, batch, "f32")
        err = _error(run_plan(pkg, dev, "dft", [n], x, batch, "f32"), _exact(x, n, "f32"))
        if not err < 1.02 * bound:
            over[n] = (err, bound)
    assert not over, over


def _ragged_over(pkg, dev, prec, bounds):
    """{n: (error, bound)} of the lengths beyond their bound, all in one batch."""
    import torch
    lib = pkg.core()
    reps = {n: max(3, 32768 // n) for n in bounds}
    sizes = [n for n in bounds for _ in range(reps[n])]
    h = ctypes.c_void_p()
    pkg.check(lib.nfft_ragged_create(ctypes.byref(h), 0 if prec == "f32" else 1, len(sizes),
                                     (ctypes.c_int * len(sizes))(*sizes), 0), "ragged_create")
    x = {n: _samples(n, reps[n], prec) for n in bounds}
    xd = torch.from_numpy(np.concatenate([x[n] for n in bounds])).to(dev)
    yd = torch.empty_like(xd)
    pkg.check(lib.nfft_ragged_execute(h, 0, xd.data_ptr(), yd.data_ptr(), None), "ragged_execute")
    pkg.check(lib.nfft_ragged_check(h, None), "ragged_check")
    y = yd.cpu().numpy()
    lib.nfft_ragged_destroy(h)
    over, off = {}, 0
    for n, bound in bounds.items():
        err = _error(y[off:off + x[n].size], _exact(x[n], n, prec))
        off += x[n].size
        if not err < 1.02 * bound:
            over[n] = (err, bound)
    return over


def test_f32_ragged_lines(pkg, dev):
    bounds = {84: 8.96e-8, 300: 1.036e-7, 1000: 1.184e-7, 1134: 1.280e-7, 1620: 1.261e-7, 3136: 1.204e-7,
              3584: 1.217e-7, 13720: 1.355e-7, 14000: 1.341e-7, 15360: 1.314e-7, 20160: 1.403e-7}
    over = _ragged_over(pkg, dev, "f32", bounds)
    assert not over, over


@pytest.mark.parametrize("prec,bounds", [
    ("f32", {41: 1.358e-7, 67: 1.406e-7, 139: 1.653e-7, 577: 1.812e-7, 1051: 1.780e-7, 1103: 1.808e-7}),
    ("f64", {41: 3.52e-16, 67: 3.64e-16, 139: 3.86e-16, 577: 4.29e-16, 1051: 4.28e-16, 1103: 4.37e-16})])
def test_ragged_bluestein(pkg, dev, prec, bounds):
    """Lengths just above a power of two: M is about 4 n as a power of two."""
    over = _ragged_over(pkg, dev, prec, bounds)
    assert not over, over
