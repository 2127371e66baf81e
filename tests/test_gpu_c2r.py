"""Long invrealdft with the pack in its first column pass (k_col_pack) against
pocketfft, and its half-weighted form (the adjoint of realdft): the shortest
lengths that take it, both row passes behind it, and odd batches (the spectra
of a batch are N/2 + 1 points apart, so all but the first are unaligned to
segments).

Tolerance: as a random walk over log2 N levels of a handful of roundings
each, with the pack as one more: 4 eps sqrt(log2 N)."""
import math

import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import pocket, rounded, run_plan

pytestmark = pytest.mark.gpu

EPS = {"f32": 2.0 ** -24, "f64": 2.0 ** -53}


@pytest.mark.parametrize("prec,lg", [("f32", lg) for lg in (17, 18, 19, 20, 21, 22)] +
                         [("f64", lg) for lg in (16, 17, 18, 20, 21)])
def test_packed_inverse(pkg, dev, prec, lg):
    n, h = 1 << lg, (1 << lg) // 2
    tol = 4 * EPS[prec] * math.sqrt(lg)
    for batch in (1, 3):
        x = rounded(ol.uniform(71, (n + 2) * batch), prec)  # bins 0 and N/2 with imaginary parts, to be ignored
        want = pocket("invrealdft", [n], x, batch)
        err = ol.rel_l2(run_plan(pkg, dev, "invrealdft", [n], x, batch, prec), want)
        assert err < tol, (prec, n, batch, err)
        w = np.full((batch, h + 1, 2), 0.5)
        w[:, [0, h]] = 1.0
        want = pocket("invrealdft", [n], x * w.reshape(-1), batch)
        err = ol.rel_l2(run_plan(pkg, dev, "realdft", [n], x, batch, prec, vjp=True), want)
        assert err < tol, (prec, n, batch, "vjp", err)
