"""The team four-step (nfft_kernels_team.h: FP64, 2^15 and 2^17 points)
against the length's other path and the oracle: the smallest batch that takes
it and one transform fewer, batches no multiple of the XCDs, several times the
intermediate slots, in place, the scaled inverse, the launch cap, and replays
of a captured graph.

Tolerance: the FP64 suite's, 1e-14 log2 N, for either path against the exact
spectrum, so twice that between the two."""
import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import tol_for

pytestmark = pytest.mark.gpu


def _plan(pkg, n, batch, team, monkeypatch, norm="reference"):
    monkeypatch.setenv("NFFT_TEAM", "1" if team else "0")
    plan = pkg.Plan("dft", "f64", [n], batch, norm)
    assert ("in teams of" in plan.describe()) == team, plan.describe()
    return plan


def _worst(a, b, n):
    """Largest rel-L2 difference over the transforms."""
    a, b = a.view(-1, 2 * n), b.view(-1, 2 * n)
    return float(((a - b).norm(dim=1) / b.norm(dim=1)).max())


@pytest.mark.parametrize("n,batch", [(1 << 15, 127), (1 << 15, 128), (1 << 15, 203), (1 << 15, 4099), (1 << 17, 31),
                                     (1 << 17, 32), (1 << 17, 101)])
@pytest.mark.parametrize("op,norm", [("dft", "reference"), ("invdft", "inverse")])
def test_team_matches_other_path_and_oracle(pkg, dev, n, batch, op, norm, monkeypatch):
    import torch
    xd = torch.empty(2 * n * batch, dtype=torch.float64, device=dev)
    pkg.fill_uniform(xd.data_ptr(), xd.numel(), 11, 0, "f64")
    got, want = torch.empty_like(xd), torch.empty_like(xd)
    for out, team in ((want, False), (got, True)):
        plan = _plan(pkg, n, batch, team, monkeypatch, norm)
        for _ in range(2):
            plan.execute(op, xd.data_ptr(), out.data_ptr())
        torch.cuda.synchronize()
        plan.check()
        plan.close()
    assert _worst(got, want, n) < 2 * tol_for("f64", n)
    for t in (0, batch // 2, batch - 1):
        sl = slice(2 * n * t, 2 * n * (t + 1))
        ref = ol.run_oracle(op, [n], xd[sl].cpu().numpy())
        if norm == "inverse":
            ref = ref / n
        assert ol.rel_l2(got[sl].cpu().numpy(), ref) < tol_for("f64", n), t


@pytest.mark.parametrize("n,batch", [(1 << 15, 150), (1 << 17, 40)])
def test_team_in_place_and_captured(pkg, dev, n, batch, monkeypatch):
    import torch
    plan = _plan(pkg, n, batch, True, monkeypatch)
    ref = _plan(pkg, n, batch, False, monkeypatch)
    buf = torch.empty(2 * n * batch, dtype=torch.float64, device=dev)
    want = torch.empty_like(buf)
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        plan.execute("dft", buf.data_ptr(), buf.data_ptr(), torch.cuda.current_stream().cuda_stream)
    for seed in range(4):  # eager first, then replays, other inputs each time
        pkg.fill_uniform(buf.data_ptr(), buf.numel(), 20 + seed, 0, "f64")
        torch.cuda.synchronize()
        ref.execute("dft", buf.data_ptr(), want.data_ptr())
        torch.cuda.synchronize()
        if seed == 0:
            plan.execute("dft", buf.data_ptr(), buf.data_ptr())
        else:
            graph.replay()
        torch.cuda.synchronize()
        assert _worst(buf, want, n) < 2 * tol_for("f64", n), seed
    plan.check()
    plan.close()
    ref.close()


def test_team_small_scratch(pkg, dev, monkeypatch):
    """Less scratch than the slots: the other path."""
    import torch
    n, batch = 1 << 15, 130
    monkeypatch.setenv("NFFT_PERSIST_MB", "4")
    x = torch.empty(2 * n * batch, dtype=torch.float64, device=dev)
    pkg.fill_uniform(x.data_ptr(), x.numel(), 12, 0, "f64")
    out = [torch.empty_like(x) for _ in range(2)]
    for y, team in zip(out, (True, False)):
        plan = _plan(pkg, n, batch, team, monkeypatch)
        plan.execute("dft", x.data_ptr(), y.data_ptr())
        torch.cuda.synchronize()
        plan.check()
        plan.close()
    assert torch.equal(out[0], out[1])


def _families(pkg, plan, x, y):
    """Kernels of one execute, by the library's timer."""
    import torch
    pkg.prof_enable(True)
    plan.execute("dft", x.data_ptr(), y.data_ptr())
    torch.cuda.synchronize()
    names = " ".join(pkg.prof_read())
    pkg.prof_enable(False)
    return names


@pytest.mark.parametrize("n,batch,mb,team", [(1 << 15, 128, 0, True), (1 << 15, 127, 0, False), (1 << 15, 130, 4, False),
                                             (1 << 17, 32, 0, True), (1 << 17, 31, 0, False), (1 << 17, 40, 8, False)])
def test_team_path_taken(pkg, dev, n, batch, mb, team, monkeypatch):
    """The team kernel runs from its smallest batch on and with scratch for its
    slots (budgets of `mb` MiB), and not otherwise."""
    import torch
    if mb:
        monkeypatch.setenv("NFFT_PERSIST_MB" if n == 1 << 15 else "NFFT_CHUNK_MB", str(mb))
    plan = _plan(pkg, n, batch, True, monkeypatch)
    x = torch.empty(2 * n * batch, dtype=torch.float64, device=dev)
    pkg.fill_uniform(x.data_ptr(), x.numel(), 13, 0, "f64")
    y = torch.empty_like(x)
    names = _families(pkg, plan, x, y)
    plan.check()
    plan.close()
    assert ("k_four_team" in names) == team, names
    ref = ol.run_oracle("dft", [n], x[-2 * n:].cpu().numpy())
    assert ol.rel_l2(y[-2 * n:].cpu().numpy(), ref) < tol_for("f64", n)


def test_team_scratch(pkg, dev, monkeypatch):
    """A large batch has scratch for the teams' slots (two transforms an XCD),
    not for the whole batch."""
    n, batch = 1 << 17, 300
    plan = _plan(pkg, n, batch, True, monkeypatch)
    assert plan.workspace_bytes <= 2 * 16 * 16 * n, plan.workspace_bytes
    plan.close()
