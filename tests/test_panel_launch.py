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


@pytest.mark.parametrize("m,k,n", [(228, 4203, 4622), (240, 6214, 4258), (1024, 4096, 1024)])
def test_wide_products_stay_in_one_round(pr, m, k, n):
    """64-column tiles that nearly fill the chip are not cut into 32-column ones
    of which a few run after all others."""
    panels, blocks = -(-m // 16), -(-k // 32)
    shape, ks = pr.default_launch(panels, blocks, n)
    nt, wp, pw = pr.SHAPES[shape]
    assert -(-panels // (wp * pw)) * -(-n // nt) * ks <= 256


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


def test_one_reservation_covers_every_default_width(pr, monkeypatch):
    """Calls of falling and rising width through one plan reserve once, as much
    as any of them splits into; an own K split reserves what it needs."""
    for panels, blocks, m in [(64, 128, 1024), (1, 400, 16), (256, 32, 4096), (3, 64, 40), (300, 9, 4800), (7, 3, 100)]:
        n0, ks0 = pr.split_reservation(panels, blocks)
        assert n0 * ks0 * panels * 16 <= 2 << 20
        for n in list(range(1, 200)) + [256, 500, 512, 1024, 2048, 4096, 65536]:
            _, ks = pr.default_launch(panels, blocks, n)
            assert ks == 1 or ks * m * n <= ks0 * m * n0
    import torch

    class Lib:
        def srt_mfma_plan_execute(self, h, C, ldc, B, ldb, cs, n, shape, ks, s):
            assert ks == 1 or ks * plan.m * n <= plan._reserved
            return 0

    class Tensor:
        dtype, is_cuda = torch.bfloat16, True

        def __init__(self, *shape):
            self.shape = shape

        def stride(self, i):
            return 1 if i else self.shape[1]

        def data_ptr(self):
            return 16

    plan = pr.PanelPlan.__new__(pr.PanelPlan)
    plan.m, plan.k, plan.dtype, plan._reserved, plan._lib = 1024, 4096, "bf16", 0, Lib()
    plan._panels, plan._k_blocks, plan._h = 64, 128, None
    calls = []
    monkeypatch.setattr(pr._lib, "call", lambda name, *a: calls.append(a))
    monkeypatch.setattr(pr, "current_raw_stream", lambda i: 0)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    assert len({pr.default_launch(64, 128, n)[1] for n in (2048, 512, 128, 64)}) > 1
    for n in (2048, 512, 128, 64, 1, 300, 512, 1024):
        C = Tensor(1024, n)
        C.dtype = torch.float32
        plan(C, Tensor(n, 4096))
    assert len(calls) == 1
    C = Tensor(1024, 4096)
    C.dtype = torch.float32
    plan(C, Tensor(4096, 4096), shape=4, ksplit=8)
    assert len(calls) == 2 and calls[-1][1:] == (4096, 8)


@pytest.mark.gpu
def test_outgrown_workspace_stays_for_its_graph(pr):
    """A captured K-split launch replays the same bits after narrower, wider and
    further split calls have been made, and memory allocated in between written."""
    import torch
    print("panel workspace under a graph", flush=True)
    g = torch.Generator().manual_seed(3)
    A = torch.randn(1024, 2048, generator=g) * (torch.rand(1024, 2048, generator=g) < 0.3)
    B = torch.randn(2048, 512, generator=g).cuda()
    plan = pr.PanelPlan.from_dense(A, "bf16")
    Bq, _ = plan.prepare_b(B)
    C = torch.empty((1024, 96), device="cuda")
    plan(C, Bq, n=96, ksplit=2)
    torch.cuda.synchronize()
    eager = C.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plan(C, Bq, n=96, ksplit=2)
    wide = torch.empty((1024, 512), device="cuda")
    junk = []
    for n, ks in ((96, None), (512, None), (64, None), (32, 16), (512, 16)):
        plan(wide, Bq, n=n, ksplit=ks)
        junk.append(torch.full((1 << 22,), float("nan"), device="cuda"))
        C.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, eager)

