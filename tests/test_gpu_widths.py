"""The gather executor at every width and alignment: the last lane moves back
where the lane width does not divide N.  Bits of the oracle's chain, nothing
written outside C's columns, B and C rows at any 4-byte address."""
import numpy as np
import pytest

from test_gpu_parity import _oracle_table, _plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M_r,name", [(4, "identity"), (8, "orig")])
@pytest.mark.parametrize("V", [2, 4])
@pytest.mark.parametrize("N", [1, 2, 3, 5, 127, 129, 255, 257, 259, 333])
def test_any_width_bitexact(srt, oracle, M_r, name, V, N):
    import torch
    so, cb = oracle
    A = srt.workloads.magnitude_pruned(70, 150, 0.8, seed=N)
    B = srt.workloads.dense_b(150, N, seed=N + 1)
    print("case", M_r, name, V, N, flush=True)
    plan = _plan(srt, torch, A, N, M_r, name, vec_width=V, waves_per_block=8, nsplit=4, chunk_cols=16)
    wide = torch.full((150, N + 6), float("nan"), device="cuda")
    wide[:, 1:1 + N] = torch.from_numpy(B).cuda()
    C = torch.full((70, N + 3), 7.0, device="cuda")
    plan(C[:, 1:], wide[:, 1:1 + N], n=N)
    torch.cuda.synchronize()
    got = C.cpu().numpy()
    ref = cb.exec_packed(cb.pack_dense(A, M_r, _oracle_table(so, M_r, name)), B, nsplit=plan.split_counts())
    assert np.array_equal(np.ascontiguousarray(got[:, 1:1 + N]).view(np.uint32), ref.view(np.uint32))
    assert (got[:, 0] == 7.0).all() and (got[:, 1 + N:] == 7.0).all()


def test_group_of_widths(srt, oracle):
    """One launch over problems of 1, 2 and 4 floats per lane, odd widths among them."""
    import torch
    so, cb = oracle
    mapping = srt.resolve_mapping(srt.named_mapping(4, "orig"))
    cfg = srt.TileConfig(vec_width=4, unroll=4, waves_per_block=8, nsplit=8)
    shapes = [(64, 100, 49), (40, 60, 1), (96, 80, 100), (33, 128, 131), (64, 64, 512), (20, 40, 257)]
    plans, Bs, Cs, refs = [], [], [], []
    for i, (M, K, N) in enumerate(shapes):
        A = srt.workloads.magnitude_pruned(M, K, 0.8, seed=i)
        rp, ci, v = srt.workloads.to_csr(A)
        p = srt.MatMulSpecialized(M, K, N, torch.from_numpy(v), torch.from_numpy(rp), torch.from_numpy(ci),
                                  tile_config=cfg, mapping_id=mapping)
        B = srt.workloads.dense_b(K, N, seed=i + 50)
        plans.append(p)
        Bs.append(torch.from_numpy(B).cuda())
        Cs.append(torch.full((M, N), float("nan"), device="cuda"))
        refs.append(cb.exec_packed(cb.pack_dense(A, 4, _oracle_table(so, 4, "orig")), B, nsplit=p.split_counts()))
    g = srt.cnn.GroupedPlans(plans, Bs, Cs)
    g()
    torch.cuda.synchronize()
    assert g.info()["vec_width"] == 1
    for C, ref in zip(Cs, refs):
        assert np.array_equal(C.cpu().numpy().view(np.uint32), ref.view(np.uint32))
    g.close()


@pytest.mark.parametrize("index_dtype", [np.int32, np.int64])
@pytest.mark.parametrize("N", [1, 3, 63, 65, 127, 130, 255, 257, 513])
def test_csr_rows_at_batch_edges(srt, oracle, index_dtype, N):
    """CSR rows of every length around the kernel's batches of 16 and 64, columns in no order."""
    import torch
    _, cb = oracle
    rng = np.random.default_rng(N)
    lengths = [0, 1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 79, 80, 81, 127, 128, 129, 192, 193, 200]
    K = 200
    cols = [rng.permutation(K)[:l] for l in lengths]
    rp = np.concatenate([[0], np.cumsum(lengths)]).astype(index_dtype)
    ci = np.concatenate(cols).astype(index_dtype)
    v = rng.standard_normal(len(ci)).astype(np.float32)
    B = rng.uniform(-1, 1, (K, N)).astype(np.float32)
    A = torch.sparse_csr_tensor(torch.from_numpy(rp), torch.from_numpy(ci), torch.from_numpy(v),
                                size=(len(lengths), K)).cuda()
    wide = torch.full((K, N + 5), float("nan"), device="cuda")
    wide[:, 3:3 + N] = torch.from_numpy(B).cuda()
    C = torch.full((len(lengths), N + 3), 7.0, device="cuda")
    srt.csr.spmm(A, wide[:, 3:3 + N], C[:, 1:1 + N])
    torch.cuda.synchronize()
    got = C.cpu().numpy()
    ref = cb.csr_exec(rp.astype(np.int64), ci.astype(np.int64), v, len(lengths), B)
    assert np.array_equal(np.ascontiguousarray(got[:, 1:1 + N]).view(np.uint32), ref.view(np.uint32))
    assert (got[:, 0] == 7.0).all() and (got[:, 1 + N:] == 7.0).all()


@pytest.mark.parametrize("K", [1, 31, 64, 65, 127, 129, 300, 2100])
@pytest.mark.parametrize("N", [1, 3, 16, 31, 33, 66])
def test_operand_preparation(srt, K, N):
    """prepare_b at the edges of its tiles, from rows at any 4-byte address:
    transposed BF16 and e4m3 operands and column scales, bit for bit."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(K * 100 + N)
    wide = torch.full((K, N + 5), float("nan"), device="cuda")
    B = wide[:, 3:3 + N]
    B.copy_(torch.randn((K, N), generator=g, device="cuda") * torch.exp(4 * torch.randn((1, N), generator=g, device="cuda")))
    B[:, N // 2] = 0
    ldk = -(-K // 32) * 32
    A = torch.zeros((16, K))
    A[0, 0] = 1
    plans = {d: srt.precision.PanelPlan.from_dense(A, d) for d in ("bf16", "fp8")}
    Bt, _ = plans["bf16"].prepare_b(B)
    ref = torch.zeros((N, ldk), dtype=torch.bfloat16, device="cuda")
    ref[:, :K] = B.t().to(torch.bfloat16)
    assert torch.equal(Bt.view(torch.int16), ref.view(torch.int16))
    Bq, t = plans["fp8"].prepare_b(B)
    top = B.abs().amax(dim=0).double()
    scale = torch.where(top > 0, (top / 448.0).float(), torch.ones_like(t))
    assert torch.equal(t, scale)
    q = torch.zeros((N, ldk), dtype=torch.uint8, device="cuda")
    q[:, :K] = (B.double() / scale.double()).float().t().contiguous().to(torch.float8_e4m3fn).view(torch.uint8)
    assert torch.equal(Bq, q)


@pytest.mark.parametrize("N", [3, 70, 130])
def test_csr_rows_at_the_end_of_the_index_range(srt, oracle, N):
    """int32 indices and 2^31 - 1 stored entries: the last rows end where a sum
    past the end does not fit the index type.  Only those rows are in the
    product, and only their entries of the arrays are written."""
    import torch
    _, cb = oracle
    nnz, K, lengths = 2 ** 31 - 1, 200, [1, 64, 65, 130, 40, 0, 20]
    if torch.cuda.mem_get_info()[0] < 24 << 30:
        pytest.skip("needs 24 GiB of device memory")
    print("csr at 2^31 - 1 entries", N, flush=True)
    rng = np.random.default_rng(N)
    used = sum(lengths)
    ci = np.concatenate([rng.permutation(K)[:l] for l in lengths]).astype(np.int32)
    v = rng.standard_normal(used).astype(np.float32)
    B = rng.uniform(-1, 1, (K, N)).astype(np.float32)
    rp = (nnz - used + np.concatenate([[0], np.cumsum(lengths)])).astype(np.int32)
    cols, vals = torch.empty(nnz, dtype=torch.int32, device="cuda"), torch.empty(nnz, device="cuda")
    cols[-used:], vals[-used:] = torch.from_numpy(ci).cuda(), torch.from_numpy(v).cuda()
    shape = torch.sparse_csr_tensor(torch.zeros(len(lengths) + 1, dtype=torch.int32), torch.zeros(0, dtype=torch.int32),
                                    torch.zeros(0), size=(len(lengths), K))
    C = srt.csr.spmm(shape, torch.from_numpy(B).cuda(), _parts_cache=(torch.from_numpy(rp).cuda(), cols, vals))
    torch.cuda.synchronize()
    ref = cb.csr_exec((rp - rp[0]).astype(np.int64), ci.astype(np.int64), v, len(lengths), B)
    assert np.array_equal(C.cpu().numpy().view(np.uint32), ref.view(np.uint32))


def test_lane_width_of_many_waves_stays_within_its_lds(srt):
    """16 waves of 8-row panels reduce in 64 KiB: two floats per lane, whatever
    the width asked for, and a problem table entry of four is refused."""
    import ctypes as ct

    import torch
    A = srt.workloads.magnitude_pruned(256, 300, 0.8, seed=1)
    rp, ci, v = srt.workloads.to_csr(A)
    plan = srt.MatMulSpecialized(256, 300, 512, torch.from_numpy(v), torch.from_numpy(rp), torch.from_numpy(ci),
                                 tile_config=srt.TileConfig(vec_width=4, waves_per_block=16, nsplit=16, unroll=4),
                                 mapping_id=srt.named_mapping(8, "orig"))
    assert plan.get_config().vec_width == 2
    assert max(plan.split_counts()) > 1  # the plan reduces
    B, C = torch.zeros((300, 512), device="cuda"), torch.zeros((256, 512), device="cuda")
    out = (ct.c_uint8 * 128)()
    fill = srt._lib.lib().srt_exec_problem_fill
    args = lambda V: (plan._h, B.data_ptr(), 512, C.data_ptr(), 512, 512, V, 0, ct.byref(out))
    assert fill(*args(2)) == 0
    assert fill(*args(4)) == srt._lib.SRT_ERR_UNSUPPORTED


@pytest.mark.parametrize("M,K,s,N,V", [(1211, 9904, 0.887, 199, 1), (2699, 6439, 0.985, 104, 1), (4163, 2281, 0.92, 384, 4),
                                       (2424, 524, 0.708, 320, 4), (63, 199, 0.583, 3168, 4), (512, 512, 0.95, 128, 1),
                                       (16384, 256, 0.9, 128, 2)])
def test_default_lane_width(srt, M, K, s, N, V):
    """Sizes on either side of the lines of the default rule."""
    import torch
    csr = (torch.rand(M, K, device="cuda") >= s).float().to_sparse_csr()
    plan = srt.MatMulSpecialized.from_csr(csr, N, mapping_id=srt.named_mapping(4, "orig"))
    assert plan.get_config().vec_width == V


@pytest.mark.parametrize("M,K,s,N,halved", [(64, 6325, 0.928, 2605, False), (260, 2497, 0.975, 3110, True), (148, 2003, 0.54, 1564, True),
                                            (3492, 7320, 0.991, 309, True), (1024, 4096, 0.9, 128, False)])
def test_default_chunk_is_halved_where_a_panel_has_few(srt, M, K, s, N, halved):
    """More than four N tiles and fewer than four chunks a panel: half the columns a chunk."""
    import torch
    csr = (torch.rand(M, K, device="cuda") >= s).float().to_sparse_csr()
    plan = srt.MatMulSpecialized.from_csr(csr, N, mapping_id=srt.named_mapping(4, "orig"),
                                          tile_config=srt.TileConfig(vec_width=1))
    whole = -(-plan.stats()["packed_cols"] * -(-N // 64) // 4096)
    assert whole > 60
    assert plan.get_config().chunk_cols == (max(60, whole // 2) if halved else whole)


@pytest.mark.parametrize("M,K,s,N,V", [(5334, 4719, 0.9951, 88, 1), (6034, 3033, 0.9944, 80, 1), (3002, 3357, 0.9869, 201, 1),
                                       (5200, 1892, 0.924, 128, 2), (42, 70, 0.8787, 2373, 1), (192, 238, 0.9896, 3020, 4),
                                       (3122, 165, 0.9911, 152, 4), (166, 529, 0.9957, 4028, 4), (331, 10472, 0.9293, 983, 1)])
def test_default_lane_width_with_few_gathers(srt, M, K, s, N, V):
    """Rows of B that few panels gather are read by narrow lanes, unless the whole work is small."""
    import torch
    csr = (torch.rand(M, K, device="cuda") >= s).float().to_sparse_csr()
    plan = srt.MatMulSpecialized.from_csr(csr, N, mapping_id=srt.named_mapping(4, "orig"))
    assert plan.get_config().vec_width == V


def test_open_plans_of_a_group_take_the_group_s_lane_width(srt, oracle):
    """Plans that leave the lane width open: a lone launch of these has too few
    workgroups for wide lanes, the group has not.  One problem of few columns
    does not narrow the others, a plan given a width keeps it; same bits."""
    import torch
    so, cb = oracle
    mapping = srt.resolve_mapping(srt.named_mapping(4, "orig"))

    def plan(A, N, **cfg):
        rp, ci, v = srt.workloads.to_csr(A)
        return srt.MatMulSpecialized(A.shape[0], A.shape[1], N, torch.from_numpy(v), torch.from_numpy(rp),
                                     torch.from_numpy(ci), tile_config=srt.TileConfig(**cfg), mapping_id=mapping)

    A = srt.workloads.magnitude_pruned(160, 300, 0.8, seed=1)
    B = srt.workloads.dense_b(300, 400, seed=2)
    assert plan(A, 400).get_config().vec_width == 1
    for cfgs, narrow, want in (([{}] * 12, None, 4), ([{}] * 11 + [dict(vec_width=2)], None, 2), ([{}] * 12, 40, 1),
                               ([{}] * 2, None, 1)):
        plans = [plan(A, 400, **c) for c in cfgs]
        n = [400] * len(plans)
        if narrow:
            n[3] = narrow
        Bs = [torch.from_numpy(np.ascontiguousarray(B[:, :k])).cuda() for k in n]
        Cs = [torch.full((160, k), float("nan"), device="cuda") for k in n]
        g = srt.cnn.GroupedPlans(plans, Bs, Cs)
        g()
        torch.cuda.synchronize()
        assert g.info()["vec_width"] == want
        if narrow:  # 12 x 40 panels x 7 slices, 11 of them at four floats per lane: two workgroups a panel
            assert g.info()["workgroups"] < 12 * 40 * 7
        for p, C, k in zip(plans, Cs, n):
            ref = cb.exec_packed(cb.pack_dense(A, 4, _oracle_table(so, 4, "orig")), np.ascontiguousarray(B[:, :k]),
                                 nsplit=p.split_counts())
            assert np.array_equal(C.cpu().numpy().view(np.uint32), ref.view(np.uint32))
        g.close()


def test_operand_preparation_of_values_that_are_not_ordinary(srt):
    """FP8 columns with NaN, infinities, signed zeros, and values so small that
    their scale is subnormal or underflows to zero: the bytes of B / scale
    rounded once to FP32, then NaN to 0x7f, saturated at +-448, nearest even."""
    import torch
    K, N = 200, 64
    g = np.random.default_rng(8)
    B = g.standard_normal((K, N)).astype(np.float32)
    B[3, 0], B[5, 1], B[6, 2], B[7, 2], B[9, 3] = np.nan, np.inf, -np.inf, np.nan, -0.0
    B[:, 4], B[:, 5] = -0.0, np.nan
    B[:, 6] *= np.float32(1e-38)
    B[:, 7] = (B[:, 7] * np.float32(1e-44)).astype(np.float32)
    B[:, 8] *= np.float32(3e37)
    B[1:, 9] *= np.float32(1e-7)  # one value at 448, the others far below the least subnormal
    B[:, 10] = np.float32(448.0) * np.sign(B[:, 10])
    mag = np.abs(B)
    top = np.where(np.isnan(mag), 0, mag).max(axis=0)
    with np.errstate(all="ignore"):
        scale = np.where(top > 0, (top.astype(np.float64) / 448.0).astype(np.float32), np.float32(1))
        q = (B.astype(np.float64) / scale.astype(np.float64)).astype(np.float32)
    assert scale[7] == 0 and 0 < scale[6] < 2.0 ** -126 and np.isinf(scale[1])
    ref = torch.from_numpy(np.clip(q, -448, 448)).to(torch.float8_e4m3fn).view(torch.uint8).numpy().copy()
    ref[np.isnan(q)] = 0x7f
    A = torch.zeros((16, K))
    A[0, 0] = 1
    Bq, t = srt.precision.PanelPlan.from_dense(A, "fp8").prepare_b(torch.from_numpy(B).cuda())
    assert np.array_equal(t.cpu().numpy().view(np.uint32), scale.view(np.uint32))
    assert np.array_equal(Bq.cpu().numpy()[:, :K].T, ref)


@pytest.mark.parametrize("n_tile", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("N", [40, 100, 200])
def test_csr_lane_width_is_the_columns_not_the_tile(srt, oracle, n_tile, N):
    """One, two and four floats per lane (by N); n_tile changes no bit."""
    import torch
    _, cb = oracle
    A = srt.workloads.magnitude_pruned(90, 300, 0.8, seed=N)
    B = srt.workloads.dense_b(300, N, seed=N + 1)
    rp, ci, v = srt.workloads.to_csr(A)
    csr = torch.sparse_csr_tensor(torch.from_numpy(rp), torch.from_numpy(ci), torch.from_numpy(v), size=A.shape).cuda()
    C = srt.csr.spmm(csr, torch.from_numpy(B).cuda(), n_tile=n_tile)
    ref = cb.csr_exec(rp, ci, v, 90, B)
    assert np.array_equal(C.cpu().numpy().view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("index_dtype", [np.int32, np.int64])
@pytest.mark.parametrize("N", [65, 127, 128, 129, 255, 258, 515])
def test_csr_many_short_rows(srt, oracle, index_dtype, N):
    """Enough rows of few entries for the short-row kernel, rows of every length
    around its batches, its long rows and their batches among them, the last
    workgroup short of rows; columns in no order and outside the matrix."""
    import torch
    _, cb = oracle
    rng = np.random.default_rng(N)
    M, K = 4099, 300
    lengths = rng.integers(0, 6, M)
    edges = [0, 1, 3, 4, 5, 7, 8, 9, 31, 32, 33, 34, 47, 48, 49, 63, 64, 65, 80, 81, 96, 97, 127, 128, 129, 200, 300]
    lengths[rng.permutation(M)[:len(edges)]] = edges
    lengths[-3:] = [33, 2, 70]
    lengths[8:12] = [64, 65, 40, 300]  # a workgroup of long rows
    rp = np.concatenate([[0], np.cumsum(lengths)]).astype(index_dtype)
    assert rp[-1] <= 8 * M
    ci = np.concatenate([rng.permutation(K)[:l] for l in lengths]).astype(index_dtype)
    v = rng.standard_normal(len(ci)).astype(np.float32)
    B = rng.uniform(-1, 1, (K, N)).astype(np.float32)
    ref = cb.csr_exec(rp.astype(np.int64), ci.astype(np.int64), v, M, B)
    wide = torch.full((K, N + 5), float("nan"), device="cuda")
    wide[:, 3:3 + N] = torch.from_numpy(B).cuda()
    parts = tuple(torch.from_numpy(x).cuda() for x in (rp, ci, v))
    A = torch.sparse_csr_tensor(torch.zeros(M + 1, dtype=torch.int64), torch.zeros(0, dtype=torch.int64), torch.zeros(0),
                                size=(M, K))
    C = torch.full((M, N + 3), 7.0, device="cuda")
    srt.csr.spmm(A, wide[:, 3:3 + N], C[:, 1:1 + N], _parts_cache=parts)
    torch.cuda.synchronize()
    got = C.cpu().numpy()
    assert np.array_equal(np.ascontiguousarray(got[:, 1:1 + N]).view(np.uint32), ref.view(np.uint32))
    assert (got[:, 0] == 7.0).all() and (got[:, 1 + N:] == 7.0).all()
    # entries outside the matrix are left out: the product without them
    out = rng.random(len(ci)) < 0.1
    bad = ci.copy()
    bad[out] = rng.choice([-1, K, K + 7, -1000], int(out.sum())).astype(index_dtype)
    keep = np.concatenate([[0], np.cumsum(~out)])
    ref = cb.csr_exec(keep[rp].astype(np.int64), ci[~out].astype(np.int64), v[~out], M, B)
    got = srt.csr.spmm(A, torch.from_numpy(B).cuda(), _parts_cache=(parts[0], torch.from_numpy(bad).cuda(), parts[2]))
    assert np.array_equal(got.cpu().numpy(), ref)


def test_csr_short_rows_with_row_pointers_out_of_order(srt):
    """Row pointers that fall or leave [0, nnz]: clamped, as by the other kernel
    (the same rows with enough entries behind them that it takes them)."""
    import torch
    M, K, N, nnz = 4099, 200, 130, 20000
    g = torch.Generator().manual_seed(3)
    rp = torch.sort(torch.randint(0, nnz, (M + 1,), generator=g)).values
    rp[5], rp[100], rp[200], rp[4000], rp[-1] = -7, 3, nnz + 9, 0, nnz + 100
    ci = torch.randint(0, K, (16 * M,), generator=g)
    v = torch.randn(16 * M, generator=g)
    B = torch.rand((K, N), generator=g).cuda()
    A = torch.sparse_csr_tensor(torch.zeros(M + 1, dtype=torch.int64), torch.zeros(0, dtype=torch.int64), torch.zeros(0),
                                size=(M, K))
    short = srt.csr.spmm(A, B, _parts_cache=(rp.cuda(), ci[:nnz].cuda(), v[:nnz].cuda()))
    # the same ranges, written out, in arrays of 16 entries a row
    lo = rp[:-1].clamp(0, nnz)
    fixed = torch.stack([lo, torch.maximum(rp[1:].clamp(max=nnz), lo)])
    lengths = fixed[1] - fixed[0]
    at = torch.cat([torch.arange(int(a), int(b)) for a, b in zip(fixed[0].tolist(), fixed[1].tolist())])
    ptr = torch.cat([torch.zeros(1, dtype=torch.int64), torch.cumsum(lengths, 0)])
    pad = 9 * M
    long = srt.csr.spmm(A, B, _parts_cache=(ptr.cuda(), torch.cat([ci[at], ci[:pad]]).cuda(),
                                            torch.cat([v[at], v[:pad]]).cuda()))
    assert torch.equal(short, long)


@pytest.mark.parametrize("K,N", [(1, 1), (1, 255), (32, 257), (33, 3299), (33, 3300), (64, 6400), (256, 25601), (257, 25700)])
def test_fp8_scales_of_few_rows(srt, K, N):
    """Both kernels of the column scales, around the lines between them: the
    exact scale of every column of a view with rows 4-byte aligned, zero, NaN
    and infinite columns among them."""
    import torch
    print("fp8 scales of few rows", K, N, flush=True)
    g = torch.Generator(device="cuda").manual_seed(K + N)
    B = torch.full((K, N + 5), float("nan"), device="cuda")[:, 3:3 + N]
    B.copy_(torch.randn((K, N), generator=g, device="cuda") * torch.exp(4 * torch.randn((1, N), generator=g, device="cuda")))
    if N > 8:
        B[:, 3] = 0
        B[K // 2, 4] = float("nan")
        B[K - 1, 5] = float("-inf")
        B[:, 6] = -0.0
    A = torch.zeros((16, K))
    A[0, 0] = 1
    _, t = srt.precision.PanelPlan.from_dense(A, "fp8").prepare_b(B)
    top = torch.where(B.isnan(), torch.zeros_like(B), B.abs()).amax(dim=0).double()
    scale = torch.where(top > 0, (top / 448.0).float(), torch.ones_like(t))
    assert torch.equal(t.view(torch.int32), scale.view(torch.int32))


@pytest.mark.parametrize("K,N,ld", [(748, 11215, 11215), (640, 13120, 13121), (1100, 7627, 7630)])
def test_prepared_b_of_many_unaligned_rows(srt, K, N, ld):
    """Tiles of k that 8 does not divide, and rows that start inside a line."""
    import torch
    print("prepared B, unaligned rows", K, N, flush=True)
    g = torch.Generator(device="cuda").manual_seed(K + N)
    B = torch.full((K, ld), float("nan"), device="cuda")[:, ld - N:]
    B.copy_(torch.randn((K, N), generator=g, device="cuda"))
    ldk = -(-K // 32) * 32
    A = torch.zeros((16, K))
    A[0, 0] = 1
    Bt, _ = srt.precision.PanelPlan.from_dense(A, "bf16").prepare_b(B)
    ref = torch.zeros((N, ldk), dtype=torch.bfloat16, device="cuda")
    ref[:, :K] = B.t().to(torch.bfloat16)
    assert torch.equal(Bt.view(torch.int16), ref.view(torch.int16))
    Bq, t = srt.precision.PanelPlan.from_dense(A, "fp8").prepare_b(B)
    scale = (B.abs().amax(dim=0).double() / 448.0).float()
    assert torch.equal(t, scale)
    q = torch.zeros((N, ldk), dtype=torch.uint8, device="cuda")
    q[:, :K] = (B.double() / scale.double()).float().t().contiguous().to(torch.float8_e4m3fn).view(torch.uint8)
    assert torch.equal(Bq, q)
