"""The sum of a K split over panels.

The sum of the partial tiles adds them in split order in
16-byte and in 4-byte rows: both give the same bits, at row lengths around a
block's width and at split counts around the four that are loaded together.
"""
import numpy as np
import pytest


@pytest.fixture(scope="module")
def pr():
    import importlib
    return importlib.import_module("sparse-register-tiling_amd").precision


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
@pytest.mark.parametrize("ks", [2, 3, 4, 5, 6, 9])
@pytest.mark.parametrize("n", [4, 60, 256, 1028])
def test_split_sum_wide_and_narrow_rows(pr, dtype, ks, n):
    import torch
    print("panel split sum", dtype, ks, n, flush=True)
    g = torch.Generator().manual_seed(n + ks)
    A = torch.randn(100, 320, generator=g) * (torch.rand(100, 320, generator=g) < 0.3)
    B = torch.randn(320, n, generator=g).cuda()
    plan = pr.PanelPlan.from_dense(A, dtype)
    Bq, t = plan.prepare_b(B)
    wide = torch.full((100, n), float("nan"), device="cuda")
    pad = torch.full((100, n + 3), float("nan"), device="cuda")
    off = torch.full((100 * n + 1,), float("nan"), device="cuda")
    plan(wide, Bq, t, shape=4, ksplit=ks)
    plan(pad[:, 1:n + 1], Bq, t, shape=4, ksplit=ks)
    plan(off[1:].view(100, n), Bq, t, shape=4, ksplit=ks)
    torch.cuda.synchronize()
    w = wide.cpu().numpy()
    assert np.isfinite(w).all()
    assert np.array_equal(pad[:, 1:n + 1].cpu().numpy(), w)
    assert np.array_equal(off[1:].view(100, n).cpu().numpy(), w)
    assert torch.isnan(pad[:, 0]).all() and torch.isnan(pad[:, n + 1:]).all() and torch.isnan(off[0])
    # ks partial sums of 320 / ks products each: within fp32 rounding of the
    # one-chain result, |A| |B| * (320 + ks) * 2^-24 per element
    one = torch.empty_like(wide)
    plan(one, Bq, t, shape=4, ksplit=1)
    bound = (A.abs().cuda() @ B.abs()).double() * (320 + ks) * 2.0 ** -24 * 2
    assert bool(((one.double() - wide.double()).abs() <= bound + 1e-30).all())
