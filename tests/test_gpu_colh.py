"""Column tiles by rule.  Strided axes, FP64 four-step columns and the weighted power through half a
tile of LDS (k_col_h, k_col_wpow_h): each length and width at the smallest number of tiles that takes
it, with whole and with partial tiles, forward and inverse, against pocketfft,
and the far strides against torch.fft in FP64.  Narrow tiles: partial ones, the
most tiles that take them and one more, and a four-step's.

Tolerance: the suite's, 1e-6 (FP32) / 1e-14 (FP64) log2 of the points."""
import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import pocket, rounded, run_plan, tol_for
from test_gpu_c5 import gauss_mask, np_ref, run_wpow

pytestmark = pytest.mark.gpu

# prec, op, dims, batch
CASES = [
    # the default width, two workgroups a CU
    ("f32", "dft", [1024, 16], 512), ("f32", "invdft", [1024, 64], 128), ("f32", "realdft", [1024, 32], 256),
    ("f32", "realdft", [2048, 16], 256), ("f32", "dft", [2048, 8], 513), ("f32", "realdft", [4096, 16], 171),
    ("f64", "dft", [1024, 16], 256), ("f64", "invdft", [2048, 8], 256), ("f64", "realdft", [2048, 16], 171),
    # twice the width
    ("f32", "invdft", [2048, 512], 16), ("f32", "dft", [4096, 512], 4), ("f32", "realdft", [4096, 2], 4096),
    ("f64", "dft", [2048, 4], 4096), ("f64", "invdft", [4096, 4], 512), ("f64", "realdft", [4096, 4], 512),
    # FP64 four-steps
    ("f64", "dft", [1 << 20], 4), ("f64", "invdft", [1 << 20], 5), ("f64", "dft", [1 << 21], 16),
]


@pytest.mark.parametrize("prec,op,dims,batch", CASES)
def test_half_tile_columns(pkg, dev, prec, op, dims, batch):
    p = int(np.prod(dims))
    x = rounded(ol.uniform(71, p * batch * (1 if op == "realdft" else 2)), prec)
    err = ol.rel_l2(run_plan(pkg, dev, op, dims, x, batch, prec), pocket(op, dims, x, batch))
    assert err < tol_for(prec, p), err


@pytest.mark.parametrize("prec,dims", [("f32", [512, 1 << 18]), ("f32", [1024, 512, 512]), ("f64", [512, 512, 256])])
def test_half_tile_columns_far_apart(pkg, dev, prec, dims):
    import torch
    p = int(np.prod(dims))
    dt = torch.float32 if prec == "f32" else torch.float64
    x = torch.empty(2 * p, dtype=dt, device=dev)
    pkg.fill_uniform(x.data_ptr(), x.numel(), 72, 0, prec)
    y = torch.empty_like(x)
    plan = pkg.Plan("dft", prec, dims, 1)
    plan.execute("dft", x.data_ptr(), y.data_ptr())
    torch.cuda.synchronize()
    plan.check()
    plan.close()
    want = torch.fft.fftn(torch.view_as_complex(x.double().view(dims + [2])))
    got = torch.view_as_complex(y.double().view(dims + [2]))
    assert float((got - want).norm() / want.norm()) < tol_for(prec, p)


@pytest.mark.parametrize("prec,dims,batch", [("f32", [1024, 18], 256), ("f32", [4096, 6], 256), ("f64", [2048, 9], 171),
                                             ("f32", [2048, 512], 16), ("f64", [2048, 4], 4096), ("f64", [4096, 5], 342)])
def test_half_tile_weighted_power(pkg, dev, prec, dims, batch, monkeypatch):
    p = int(np.prod(dims))
    x = rounded(ol.uniform(73, 2 * p * batch), prec)
    w = rounded(gauss_mask(dims), prec)
    lref, gref = np_ref(x, w, dims, batch)
    loss, grad = run_wpow(pkg, dev, prec, dims, batch, x, w, monkeypatch)
    assert np.max(np.abs(loss - lref) / lref) < tol_for(prec, p)
    assert ol.rel_l2(grad, gref) < tol_for(prec, p)


@pytest.mark.parametrize("prec,op,dims,batch", [
    ("f32", "dft", [256, 2], 1), ("f64", "realdft", [512, 16], 1), ("f32", "invdft", [1024, 2048], 1),
    ("f32", "dft", [1024, 2064], 1), ("f64", "dft", [2048, 512], 1), ("f32", "realdft", [2048, 64], 2),
    ("f32", "dft", [1 << 20], 1), ("f64", "invdft", [1 << 18], 1), ("f32", "dct2", [512, 8], 1),
    ("f32", "dct3", [1024, 32, 2], 1), ("f64", "dst2", [512, 2048], 1), ("f64", "dct4", [1024, 16], 1),
    ("f32", "dst3", [512, 32], 128), ("f32", "dct2", [512, 32], 129)])
def test_narrow_columns(pkg, dev, prec, op, dims, batch):
    p = int(np.prod(dims))
    x = rounded(ol.uniform(74, p * batch * (2 if op in ("dft", "invdft") else 1)), prec)
    want = ol.run_oracle(op, dims, x, batch) if op[:2] in ("dc", "ds") else pocket(op, dims, x, batch)
    err = ol.rel_l2(run_plan(pkg, dev, op, dims, x, batch, prec), want)
    assert err < tol_for(prec, p), err


@pytest.mark.parametrize("prec,dims,batch", [("f32", [64, 64], 3), ("f32", [64, 64], 1025), ("f32", [2048, 64], 5),
                                             ("f32", [256, 33], 3), ("f64", [64, 64], 7), ("f64", [32, 512], 4),
                                             ("f64", [128, 24], 9)])
def test_weighted_power_tile_orders(pkg, dev, prec, dims, batch, monkeypatch):
    """Tiles in each order: arrays that the L2s hold, of tiles that are whole
    lines and that are not, and larger ones."""
    p = int(np.prod(dims))
    x = rounded(ol.uniform(75, 2 * p * batch), prec)
    w = rounded(gauss_mask(dims), prec)
    lref, gref = np_ref(x, w, dims, batch)
    loss, grad = run_wpow(pkg, dev, prec, dims, batch, x, w, monkeypatch)
    assert np.max(np.abs(loss - lref) / lref) < tol_for(prec, p)
    assert ol.rel_l2(grad, gref) < tol_for(prec, p)


@pytest.mark.parametrize("n,batch", [(1 << 16, 63), (1 << 16, 64), (1 << 17, 33), (1 << 18, 7)])
def test_four_step_tile_orders(pkg, dev, n, batch):
    """FP32 batches that the L2s hold, and the smallest larger one."""
    x = rounded(ol.uniform(76, 2 * n * batch), "f32")
    err = ol.rel_l2(run_plan(pkg, dev, "dft", [n], x, batch, "f32"), pocket("dft", [n], x, batch))
    assert err < tol_for("f32", n), err
