"""One-pass mixed-radix lines (nfft_kernels_mix.h) against pocketfft: one to
six stages, groups of lines with a ragged last group, the longest lines of
each precision, Bluestein over a 7-smooth M in one workgroup, and both in
phases of tiles (last tiles of a few columns, rows padded to whole segments).

Tolerance: each point passes about log2(N) levels of butterflies, with a
handful of roundings (sums, one twiddle product of two rounded factors) per
level; as a random walk that is below 4 eps sqrt(log2 N), doubled for the
two transforms and three products of Bluestein."""
import math

import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import pocket, rounded, run_plan

pytestmark = pytest.mark.gpu

EPS = {"f32": 2.0 ** -24, "f64": 2.0 ** -53}
# single stage, two and three, odd ones, all radices of 7, up to the limit
LINES = [3, 6, 7, 30, 35, 54, 100, 189, 640, 1029, 2401, 4374, 5000, 9216, 10206]
LINES32 = LINES + [10290, 15625, 16807, 19683, 20000, 20412, 20480]
LINES64 = LINES + [10240]


@pytest.fixture(autouse=True)
def _large(monkeypatch, request):
    """These lengths as large batches run them, whatever the batch here."""
    if "small" not in request.node.name:
        monkeypatch.setenv("NFFT_FEW", "0")


# lines and batches of one and of several to a workgroup; tiles instead of a
# full line; Bluestein on either side of the batch where it changes
@pytest.mark.parametrize("prec,n,batch", [
    ("f32", 3, 1), ("f32", 30, 30000), ("f64", 30, 2049), ("f64", 210, 7), ("f32", 480, 257), ("f64", 720, 40),
    ("f64", 1000, 300), ("f32", 1200, 436), ("f32", 1200, 437), ("f32", 10206, 3), ("f64", 10240, 2),
    ("f32", 12005, 1), ("f32", 20480, 2), ("f64", 15000, 18), ("f64", 50000, 1), ("f32", 30000, 10), ("f32", 30000, 11),
    ("f32", 10007, 44), ("f32", 10007, 45), ("f64", 4099, 60), ("f64", 4099, 61), ("f32", 40009, 64), ("f32", 40009, 65)])
def test_small_batches(pkg, dev, prec, n, batch):
    blue = any(n % p == 0 for p in (4099, 10007, 40009))
    tol = (2 if blue else 1) * 4 * EPS[prec] * math.sqrt(math.log2(n))
    x = rounded(ol.uniform(45, 2 * n * batch), prec)
    for op, inplace in (("dft", False), ("invdft", True)):
        err = ol.rel_l2(run_plan(pkg, dev, op, [n], x, batch, prec, inplace=inplace), pocket(op, [n], x, batch))
        assert err < tol, (op, err)


@pytest.mark.parametrize("prec,n", [("f32", n) for n in LINES32] + [("f64", n) for n in LINES64])
def test_lines(pkg, dev, prec, n):
    plan = pkg.Plan("dft", prec, [n], 1)
    desc = plan.describe()
    plan.close()
    assert desc.startswith("mixed-radix") and "lines on" in desc, desc
    tol = 4 * EPS[prec] * math.sqrt(math.log2(n))
    lines = int(desc.split(", ")[1].split()[0])  # per workgroup
    for batch in (1, 2 * lines + 1):
        x = rounded(ol.uniform(41, 2 * n * batch), prec)
        for op, inplace in (("dft", False), ("dft", True), ("invdft", False)):
            got = run_plan(pkg, dev, op, [n], x, batch, prec, inplace=inplace)
            err = ol.rel_l2(got, pocket(op, [n], x, batch))
            assert err < tol, (prec, n, batch, op, inplace, err, desc)


@pytest.mark.parametrize("prec,n", [("f32", n) for n in (8209, 9973, 10007, 10169)] +
                         [("f64", n) for n in (4099, 5003, 5101)])
def test_bluestein_one_pass(pkg, dev, prec, n):
    plan = pkg.Plan("dft", prec, [n], 1)
    desc = plan.describe()
    plan.close()
    assert desc.startswith("bluestein") and "one pass" in desc, desc
    tol = 2 * 4 * EPS[prec] * math.sqrt(math.log2(n))
    for batch in (1, 3):
        x = rounded(ol.uniform(42, 2 * n * batch), prec)
        for op, inplace in (("dft", False), ("invdft", True)):
            got = run_plan(pkg, dev, op, [n], x, batch, prec, inplace=inplace)
            err = ol.rel_l2(got, pocket(op, [n], x, batch))
            assert err < tol, (prec, n, batch, op, inplace, err, desc)


@pytest.mark.parametrize("prec,n", [("f32", n) for n in (20736, 22050, 65610, 196608, 1000000)] +
                         [("f64", n) for n in (10290, 15625, 65610, 196608, 1000000)] +
                         [("f32", n) for n in (10247, 10301, 16381, 33333, 65537, 100003)] +
                         [("f64", n) for n in (17011, 33331, 65537, 70001)])
def test_tiles(pkg, dev, prec, n):
    plan = pkg.Plan("dft", prec, [n], 1)
    desc = plan.describe()
    plan.close()
    blue = not desc.startswith("mixed-radix four-step")
    assert not blue or "in tiles" in desc, desc
    tol = (2 if blue else 1) * 4 * EPS[prec] * math.sqrt(math.log2(n))
    for batch in (1, 3):
        x = rounded(ol.uniform(44, 2 * n * batch), prec)
        for op, inplace in (("dft", False), ("invdft", True)):
            got = run_plan(pkg, dev, op, [n], x, batch, prec, inplace=inplace)
            err = ol.rel_l2(got, pocket(op, [n], x, batch))
            assert err < tol, (prec, n, batch, op, inplace, err, desc)


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("dims", [[100, 48, 30], [5, 5000], [1000, 81]])
def test_axes(pkg, dev, prec, dims):
    """Contiguous and strided axes of an N-D transform through the same lines."""
    p = int(np.prod(dims))
    x = rounded(ol.uniform(43, 2 * p * 2), prec)
    tol = 4 * EPS[prec] * math.sqrt(math.log2(p))
    for op in ("dft", "invdft"):
        got = run_plan(pkg, dev, op, dims, x, 2, prec)
        err = ol.rel_l2(got, pocket(op, dims, x, 2))
        assert err < tol, (prec, dims, op, err)


@pytest.mark.parametrize("prec,dims,batch", [("f32", [10007, 4], 1), ("f32", [10007, 4], 40), ("f64", [5003, 16], 2),
                                             ("f32", [1200, 8], 3), ("f64", [15000, 8], 1)])
def test_small_realdft_leading_axes(pkg, dev, prec, dims, batch):
    """The leading axes of a realdft are planned for the lines they have."""
    n, h = dims[0], dims[1] // 2 + 1
    plan, axis = pkg.Plan("realdft", prec, dims, batch), pkg.Plan("dft", prec, [n], batch * h)
    desc, want = plan.describe(), axis.describe()
    plan.close()
    axis.close()
    assert desc.endswith("| " + want), (desc, want)
    tol = 2 * 4 * EPS[prec] * math.sqrt(math.log2(n * dims[1]))
    x = rounded(ol.uniform(46, n * dims[1] * batch), prec)
    y = pocket("realdft", dims, x, batch)
    assert ol.rel_l2(run_plan(pkg, dev, "realdft", dims, x, batch, prec), y) < tol
    y = rounded(y, prec)
    assert ol.rel_l2(run_plan(pkg, dev, "invrealdft", dims, y, batch, prec), pocket("invrealdft", dims, y, batch)) < tol


@pytest.mark.parametrize("n,batch,tiles", [(16381, 896, False), (16381, 897, True), (12007, 576, False),
                                           (12007, 577, True), (24001, 448, False), (24001, 449, True),
                                           (17011, 128, False), (17011, 129, True), (40009, 65, True)])
def test_small_bluestein_tiles_begin(pkg, dev, n, batch, tiles):
    """FP32 batches on either side of the size where tiles replace the power
    of two's three passes."""
    plan = pkg.Plan("dft", "f32", [n], batch)
    desc = plan.describe()
    plan.close()
    assert ("in tiles" in desc) == tiles, desc
    x = rounded(ol.uniform(47, 2 * n * batch), "f32")
    err = ol.rel_l2(run_plan(pkg, dev, "dft", [n], x, batch, "f32"), pocket("dft", [n], x, batch))
    assert err < 2 * 4 * EPS["f32"] * math.sqrt(math.log2(n)), (desc, err)


@pytest.mark.parametrize("prec,n,batch,tiles", [
    ("f64", 10240, 51, True), ("f64", 10240, 52, False), ("f64", 10000, 3, False), ("f64", 24000, 13, True),
    ("f64", 24000, 22, True), ("f64", 100000, 5, True), ("f32", 20480, 38, True), ("f32", 20480, 39, False),
    ("f32", 15000, 34, True), ("f32", 15000, 35, False), ("f32", 30000, 26, True), ("f32", 30000, 27, True)])
def test_small_batches_of_tiles(pkg, dev, prec, n, batch, tiles):
    """Tiles of a quarter, a half and all of the points, and lines, on either
    side of the batches where they change."""
    plan = pkg.Plan("dft", prec, [n], batch)
    desc = plan.describe()
    plan.close()
    assert desc.startswith("mixed-radix four-step") == tiles, desc
    x = rounded(ol.uniform(48, 2 * n * batch), prec)
    for op in ("dft", "invdft"):
        err = ol.rel_l2(run_plan(pkg, dev, op, [n], x, batch, prec), pocket(op, [n], x, batch))
        assert err < 4 * EPS[prec] * math.sqrt(math.log2(n)), (op, err, desc)


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("n", [3, 5, 7, 9, 12, 15, 21, 28, 30])
def test_small_lines_of_one_butterfly(pkg, dev, prec, n):
    """Copied through LDS: one line, a partial last group, and the batch from
    which the groups are larger; in place and both directions."""
    for batch in (1, 300, (1 << 21) // n + 1):
        x = rounded(ol.uniform(49, 2 * n * batch), prec)
        for op, inplace in (("dft", True), ("invdft", False)):
            err = ol.rel_l2(run_plan(pkg, dev, op, [n], x, batch, prec, inplace=inplace), pocket(op, [n], x, batch))
            assert err < 4 * EPS[prec] * math.sqrt(math.log2(n)), (batch, op, err)


@pytest.mark.parametrize("prec,n,batch", [("f64", 720, 819), ("f64", 720, 820), ("f64", 480, 5461), ("f64", 480, 5462),
                                          ("f64", 100, 26215), ("f64", 100, 94371), ("f64", 100, 94372),
                                          ("f32", 480, 2185)])
def test_small_middling_batches(pkg, dev, prec, n, batch):
    """On either side of the sizes where the schedules of small batches end."""
    x = rounded(ol.uniform(50, 2 * n * batch), prec)
    for op in ("dft", "invdft"):
        err = ol.rel_l2(run_plan(pkg, dev, op, [n], x, batch, prec), pocket(op, [n], x, batch))
        assert err < 4 * EPS[prec] * math.sqrt(math.log2(n)), (op, err)
