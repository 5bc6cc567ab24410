"""Dense panels of a hybrid plan: output tiles and K splits.

Every launch the rule can take covers all rows, columns and K ranges: sizes
around the tiles' edges (32, 64, 128 rows; 64, 128 columns; 64 deep), widths
that are no multiple of 4 (the narrow B loads), and products from one tile to
several rounds of the chip.  K chains of fp32 products and their sums: within
(K + 40) * 2^-24 * |A| |B| of the float64 product, and equal bits on a repeat.
"""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def srt():
    import importlib
    return importlib.import_module("sparse-register-tiling_amd")


@pytest.mark.parametrize("mkn", [(16, 64, 16), (33, 65, 64), (31, 700, 65), (96, 130, 127), (64, 64, 128), (129, 513, 129),
                                 (512, 512, 128), (512, 2048, 256), (300, 1500, 333), (256, 4096, 512), (1024, 1024, 512),
                                 (4096, 256, 512), (2048, 512, 100), (4096, 4096, 64), (2064, 192, 1030),
                                 (1024, 4096, 512)])
def test_tiles_and_splits(srt, mkn):
    import torch
    M, K, N = mkn
    print("dense tiles", mkn, flush=True)
    g = torch.Generator().manual_seed(M + K + N)
    A = torch.randn(M, K, generator=g) * (torch.rand(M, K, generator=g) < 0.5)
    B = torch.randn(K, N, generator=g).cuda()
    plan = srt.MatMulSpecialized.from_csr(A.to_sparse_csr().cuda(), N, mapping_id=srt.named_mapping(4, "orig"),
                                          dense_threshold=0.2)
    out = torch.full((M, N), float("nan"), device="cuda")
    plan(out, B)
    again = torch.full((M, N), float("nan"), device="cuda")
    plan(again, B)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    Ad = A.cuda().double()
    err = (out.double() - Ad @ B.double()).abs()
    bound = (Ad.abs() @ B.double().abs()) * (K + 40) * 2.0 ** -24
    assert bool((err <= bound + 1e-30).all())
    # a narrower product through the same plan: another grid, the same workspace
    n = max(1, N // 3)
    part = torch.full((M, n), float("nan"), device="cuda")
    plan(part, B[:, :n].contiguous())
    assert bool(((part.double() - Ad @ B[:, :n].double()).abs() <= bound[:, :n] + 1e-30).all())


@pytest.mark.parametrize("M,K,widths", [(1024, 4096, (1600, 900, 512, 300, 100, 1)), (512, 2000, (4096, 700, 256)),
                                        (100, 300, (5000, 129))])
def test_narrower_products_split_as_in_a_plan_of_their_own(srt, M, K, widths):
    """Fewer columns than a plan was made for: the bits of a plan made for them."""
    import torch
    g = torch.Generator().manual_seed(M + K)
    A = (torch.randn(M, K, generator=g) * (torch.rand(M, K, generator=g) < 0.5)).to_sparse_csr().cuda()

    def make(n):
        return srt.MatMulSpecialized.from_csr(A, n, mapping_id=srt.named_mapping(4, "orig"), dense_threshold=0.2)

    wide = make(widths[0])
    for n in widths:
        print("narrow", M, K, widths[0], n, flush=True)
        B = torch.randn((K, n), generator=g).cuda()
        out, own = (torch.full((M, n), float("nan"), device="cuda") for _ in range(2))
        plan = make(n)
        wide(out, B)
        plan(own, B)
        torch.cuda.synchronize()
        assert torch.equal(out, own)


@pytest.mark.parametrize("mkn", [(64, 2048, 128), (129, 513, 129), (512, 2048, 256), (256, 4096, 512), (1024, 4096, 512),
                                 (2064, 192, 1030), (33, 4000, 63)])
def test_tile_and_split_change_no_bit(srt, mkn):
    """A plan made for no columns has no workspace: every range of a tile in one
    workgroup, and the tile that is fastest so.  The bits of the split launch."""
    import torch
    M, K, N = mkn
    g = torch.Generator().manual_seed(M + K + N)
    A = (torch.randn(M, K, generator=g) * (torch.rand(M, K, generator=g) < 0.5)).to_sparse_csr().cuda()
    B = torch.randn(K, N, generator=g).cuda()
    out = []
    for n in (N, 0):
        print("dense bits", mkn, n, flush=True)
        plan = srt.MatMulSpecialized.from_csr(A, n, mapping_id=srt.named_mapping(4, "orig"), dense_threshold=0.2)
        out.append(torch.full((M, N), float("nan"), device="cuda"))
        plan(out[-1], B)
    assert not bool(torch.isnan(out[0]).any())
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("mkn", [(33, 8192, 63), (1500, 2692, 127), (1500, 1472, 128), (16, 6100, 300)])
def test_long_ranges_are_their_own_groups(srt, mkn):
    """More than eight groups of three stages and more; the third has shorter ones, in eight groups."""
    import torch
    M, K, N = mkn
    g = torch.Generator().manual_seed(M + K + N)
    A = torch.randn(M, K, generator=g) * (torch.rand(M, K, generator=g) < 0.5)
    B = torch.randn(K, N, generator=g).cuda()
    ref, mag = A.double() @ B.cpu().double(), A.abs().double() @ B.cpu().abs().double()
    out = []
    for n in (N, 0):
        print("dense groups", mkn, n, flush=True)
        plan = srt.MatMulSpecialized.from_csr(A.to_sparse_csr().cuda(), n, mapping_id=srt.named_mapping(4, "orig"),
                                              dense_threshold=0.2)
        out.append(torch.full((M, N), float("nan"), device="cuda"))
        plan(out[-1], B)
    assert bool(((out[0].cpu().double() - ref).abs() <= K * 2.0 ** -24 * mag + 1e-30).all())
    assert torch.equal(out[0], out[1])
