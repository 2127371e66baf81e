"""Errors of the mixed-radix lines and tiles, uniform and ragged, held to what
the lengths had when every twiddle was a table entry of its own.

The bounds are rel-L2 errors of Gaussian samples measured with that engine
(the two-buffer lines, four-steps and Bluestein passes these lines replaced),
plus 2 %: three standard deviations of an error estimated from 2^15 points."""
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
