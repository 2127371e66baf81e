"""DCT / DST along strided axes (nfft_kernels_tcol.h) against the oracle:
every tile shape at its edges (one column up to several tiles over several
arrays), the longest axis with a column kernel and the first one without,
in place and with the adjoint's weight of the DC term.

Tolerance: as a random walk over log2(points) levels of a handful of
roundings each, for every axis: 8 eps sqrt(log2 P)."""
import math

import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import rounded, run_plan

pytestmark = pytest.mark.gpu

EPS = {"f32": 2.0 ** -24, "f64": 2.0 ** -53}
# dims, batch
CASES = [([2, 2], 1), ([2, 2], 300), ([4, 32], 3), ([8, 8], 33), ([16, 2], 130), ([16, 64], 5), ([32, 4], 9),
         ([64, 16], 3), ([128, 8, 4], 2), ([512, 2], 3), ([1024, 64], 1), ([2048, 16], 1), ([4096, 2], 2),
         ([4096, 32], 1), ([8192, 4], 1), ([2, 4, 8, 16], 2), ([1, 64, 2], 2)]


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("dims,batch", CASES)
def test_strided_trig(pkg, dev, prec, dims, batch):
    p = int(np.prod(dims))
    x = rounded(ol.uniform(61, p * batch), prec)
    tol = 8 * EPS[prec] * math.sqrt(math.log2(p))
    for op in ("dct2", "dst2", "dct3", "dst3", "dct4", "dst4"):
        want = ol.run_oracle(op, dims, x, batch)
        for inplace in (False, True):
            err = ol.rel_l2(run_plan(pkg, dev, op, dims, x, batch, prec, inplace=inplace), want)
            assert err < tol, (prec, op, dims, batch, inplace, err)


@pytest.mark.parametrize("dims", [[64, 8], [2, 16, 4]])
@pytest.mark.parametrize("op", ["dct2", "dst2", "dct3", "dst3", "dct4"])
def test_strided_trig_adjoint(pkg, dev, dims, op):
    """<vjp(g), x> = <g, f(x)> in FP64."""
    p = int(np.prod(dims))
    x, g = ol.uniform(62, p), ol.uniform(63, p)
    fx = run_plan(pkg, dev, op, dims, x, 1, "f64")
    v = run_plan(pkg, dev, op, dims, g, 1, "f64", vjp=True)
    scale = np.linalg.norm(g) * np.linalg.norm(fx)
    assert abs(np.dot(v, x) - np.dot(g, fx)) < 64 * EPS["f64"] * scale


@pytest.mark.parametrize("prec,kind,dims,batch,few", [
    ("f32", "t4", [4096, 64], 3, True), ("f32", "t4", [4096, 256], 1, False), ("f64", "t4", [4096, 64], 1, True),
    ("f64", "t4", [4096, 128], 1, False), ("f32", "t4", [2048, 2], 32, True), ("f64", "t4", [2048, 2], 33, False),
    ("f32", "t2t3", [4096, 2], 32, True), ("f32", "t2t3", [4096, 2], 33, False), ("f32", "t2t3", [4096, 4], 8, True),
    ("f32", "t2t3", [4096, 4], 9, False), ("f64", "t2t3", [4096, 2], 3, False)])
def test_few_long_columns(pkg, dev, prec, kind, dims, batch, few):
    """A few long columns are transposed (through the plan's workspace), one
    more is not."""
    plan = pkg.Plan(kind, prec, dims, batch)
    transposed = plan.workspace_bytes > 0
    plan.close()
    assert transposed == few
    p = int(np.prod(dims))
    x = rounded(ol.uniform(64, p * batch), prec)
    for op in ("dct4", "dst4") if kind == "t4" else ("dct2", "dst3"):
        err = ol.rel_l2(run_plan(pkg, dev, op, dims, x, batch, prec), ol.run_oracle(op, dims, x, batch))
        assert err < 8 * EPS[prec] * math.sqrt(math.log2(p)), (op, err)
