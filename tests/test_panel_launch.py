"""The panel launch rule and the K split's sum.

The rule never splits further than its workspace limit and names a launch
shape that exists.  The sum of the partial tiles adds them in split order in
16-byte and in 4-byte rows: both give the same bits, at row lengths around a
block's width and at split counts around the four that are loaded together.
"""
import numpy as np
import pytest


@pytest.fixture(scope="module")
def pr():
    import importlib
    return importlib.import_module("sparse-register-tiling_amd").precision


def test_rule_stays_within_its_workspace(pr):
    for panels in (0, 1, 3, 16, 63, 64, 255, 4096):
        for blocks in (0, 1, 4, 5, 31, 128, 1024):
            for n in (1, 31, 32, 33, 100, 512, 4096, 100000):
                shape, ks = pr.default_launch(panels, blocks, n)
                assert shape in pr.SHAPES
                assert 1 <= ks <= pr._split_limit(panels, blocks, n)
                assert ks == 1 or ks * 4 <= blocks


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
