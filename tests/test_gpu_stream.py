"""Streamed execution (M_r = 1, tiles of B rows in LDS): bit-identical to the
sequential fused multiply-add chain over each row's nonzeros in column order
(the oracle's CSR executor) at the edges of tiles, slices, waves and quads."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _plan(srt, torch, A, n, index_dtype=np.int64, **cfg):
    rp, ci, v = srt.workloads.to_csr(A, index_dtype)
    return srt.MatMulSpecialized(A.shape[0], A.shape[1], n, torch.from_numpy(v), torch.from_numpy(rp),
                                 torch.from_numpy(ci), tile_config=srt.TileConfig(b_staging=3, **cfg),
                                 mapping_id=srt.named_mapping(1, "identity"))


def _chain(srt, cb, A, B):
    rp, ci, v = srt.workloads.to_csr(A)
    return cb.csr_exec(rp, ci, v, A.shape[0], B)


def _same(C, ref):
    assert np.array_equal(np.isnan(C), np.isnan(ref))
    ok = ~np.isnan(ref)
    assert np.array_equal(C.view(np.uint32)[ok], ref.view(np.uint32)[ok])


# tile edges: V = 4 holds 64 rows at 16 waves (32 at 8), V = 2 128, V = 1 256
CASES = [(1, 1, 1), (17, 63, 5), (64, 64, 256), (33, 65, 257), (130, 129, 64), (70, 255, 131), (257, 300, 510),
         (40, 513, 1023), (300, 777, 333), (16, 2048, 96)]


@pytest.mark.parametrize("V,W,R", [(1, 16, 1), (1, 4, 8), (2, 16, 2), (2, 8, 4), (4, 16, 8), (4, 16, 1), (4, 4, 2),
                                   (4, 8, 4), (0, 0, 0)])
@pytest.mark.parametrize("M,K,N", CASES)
def test_bitexact_at_the_edges(srt, oracle, M, K, N, V, W, R):
    import torch
    _, cb = oracle
    rng = np.random.default_rng(M * 7 + K * 3 + N)
    A = (rng.standard_normal((M, K)) * (rng.random((M, K)) < 0.3)).astype(np.float32)
    A[:: max(1, M // 5)] = 0  # empty rows
    A[M // 2] = rng.standard_normal(K)  # a full one
    B = rng.uniform(-1, 1, (K, N)).astype(np.float32)
    print("case", M, K, N, V, W, R, flush=True)
    plan = _plan(srt, torch, A, N, np.int32 if N % 2 else np.int64, vec_width=V, waves_per_block=W, chunk_cols=R)
    real = plan.get_config()
    assert real.b_staging == 3 and (not V or (real.vec_width, real.waves_per_block, real.chunk_cols) == (V, W, R))
    wide = torch.full((K, N + 5), 9.0, device="cuda")  # strided, unaligned rows
    wide[:, 3:3 + N] = torch.from_numpy(B).cuda()
    C = torch.full((M, N + 3), float("nan"), device="cuda")
    plan(C[:, 1:], wide[:, 3:3 + N], n=N)
    torch.cuda.synchronize()
    got = C.cpu().numpy()
    _same(np.ascontiguousarray(got[:, 1:1 + N]), _chain(srt, cb, A, B))
    assert np.isnan(got[:, 0]).all() and np.isnan(got[:, 1 + N:]).all()


def test_values_that_are_not_numbers(srt, oracle):
    """Padding leaves infinities, NaN and signed zeros as the chain has them."""
    import torch
    _, cb = oracle
    rng = np.random.default_rng(5)
    A = (rng.standard_normal((64, 200)) * (rng.random((64, 200)) < 0.2)).astype(np.float32)
    B = rng.uniform(-1, 1, (200, 70)).astype(np.float32)
    A[3, 7], A[4, 9], A[5, :] = np.inf, -np.inf, 0
    A[5, 11] = np.float32(-1e-30)
    B[20, 3], B[21, 4], B[11] = np.inf, np.nan, np.float32(1e-30)  # row 5: -0 by underflow
    plan = _plan(srt, torch, A, 70)
    C = torch.empty((64, 70), device="cuda")
    plan(C, torch.from_numpy(B).cuda())
    _same(C.cpu().numpy(), _chain(srt, cb, A, B))


def test_other_widths_groups_and_graphs(srt, oracle):
    """One plan at other widths, rebuilt for one, captured, in a group, as a hybrid."""
    import torch
    _, cb = oracle
    A = srt.workloads.magnitude_pruned(200, 150, 0.7, seed=3)
    plan = _plan(srt, torch, A, 256)
    B = srt.workloads.dense_b(150, 300, seed=4)
    Bt = torch.from_numpy(B).cuda()
    ref = _chain(srt, cb, A, B)
    C = torch.empty((200, 300), device="cuda")
    for n in (300, 1, 64, 257):
        plan(C, Bt, n=n)
        _same(np.ascontiguousarray(C.cpu().numpy()[:, :n]), np.ascontiguousarray(ref[:, :n]))
    plan.allocate_executor(8)
    plan(C, Bt)
    _same(C.cpu().numpy(), ref)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        plan(C, Bt)
    for _ in range(3):
        C.zero_()
        g.replay()
        torch.cuda.synchronize()
        _same(C.cpu().numpy(), ref)
    two = _plan(srt, torch, A, 300)
    C2 = torch.empty_like(C)
    grp = srt.cnn.GroupedPlans([plan, two], [Bt, Bt], [C, C2])  # the gather schedules, built on demand
    C.zero_()
    grp()
    torch.cuda.synchronize()
    _same(C.cpu().numpy(), ref)  # the bits of its own launch
    assert torch.equal(C, C2)
    grp.close()
    rp, ci, v = srt.workloads.to_csr(A)
    h = srt.MatMulSpecialized(200, 150, 300, torch.from_numpy(v), torch.from_numpy(rp), torch.from_numpy(ci),
                              mapping_id=srt.named_mapping(1, "identity"), dense_threshold=0.35)
    dense = h.dense_panels()["rows"]
    assert 0 < len(dense) < 13
    h(C, Bt)
    rest = np.ones(200, dtype=bool)
    for r in dense:
        rest[r:r + 16] = False
    got = C.cpu().numpy()
    _same(np.ascontiguousarray(got[rest]), np.ascontiguousarray(ref[rest]))
    assert np.all(np.abs(got - cb.dense_f64(A, B)) <= srt_bound(A, B))


def srt_bound(A, B):
    """FP32 summation bound of a chain: 2 L 2^-24 (|A| |B|)."""
    L = int((A != 0).sum(axis=1).max())
    return 2 * L * 2.0 ** -24 * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64)) + 1e-30


def test_rule_takes_streams_for_much_work(srt):
    at = srt.autotune
    assert at.streamed_launch(4096, 1024, 838860, 2048)[2] < at.gather_seconds(4096, 1024, 838860, 2048)
    assert at.streamed_launch(512, 512, 13107, 8)[2] > at.gather_seconds(512, 512, 13107, 8)


def test_alternating_widths_reuse_their_schedules(srt, oracle):
    """allocate_executor between two widths builds each launch shape once."""
    import torch
    _, cb = oracle
    A = srt.workloads.magnitude_pruned(1024, 1024, 0.5, seed=6)
    B = srt.workloads.dense_b(1024, 64, seed=7)
    ref = _chain(srt, cb, A, B)
    plan = _plan(srt, torch, A, 64)
    Bt, C = torch.from_numpy(B).cuda(), torch.empty((1024, 64), device="cuda")
    shapes, free = set(), None
    for i in range(24):
        plan.allocate_executor(2048 if i % 2 == 0 else 64)
        c = plan.get_config()
        shapes.add((c.vec_width, c.chunk_cols))
        plan(C, Bt)
        torch.cuda.synchronize()
        _same(C.cpu().numpy(), ref)
        if i == 3:
            free = torch.cuda.mem_get_info()[0]
    assert len(shapes) == 2
    assert torch.cuda.mem_get_info()[0] >= free  # a further copy of the entries is 5 MB


def test_tuned_plans_group(srt, oracle):
    """Tuned plans of sizes the table does not hold, some streamed, some not, in
    one group: the bits of their own launches, captured and re-bound."""
    import torch
    sizes = [(300, 220, 0.9, 100), (4096, 1024, 0.8, 640), (129, 500, 0.8, 33), (4096, 500, 0.75, 1000), (64, 64, 0.9, 5)]
    plans, Bs, Cs, refs = [], [], [], []
    for i, (M, K, s, N) in enumerate(sizes):
        g = torch.Generator(device="cuda").manual_seed(i)
        A = torch.randn((M, K), generator=g, device="cuda") * (torch.rand((M, K), generator=g, device="cuda") >= s)
        p = srt.autotune.tuned_plan(A.to_sparse_csr(), N)
        B = torch.rand((K, N + 3), generator=g, device="cuda")[:, 1:1 + N]
        C = torch.full((M, N), float("nan"), device="cuda")
        ref = torch.empty_like(C)
        p(ref, B)
        plans.append(p), Bs.append(B), Cs.append(C), refs.append(ref)
    streamed = [p.get_config().b_staging == 3 for p in plans]
    assert any(streamed) and not all(streamed)
    g = srt.cnn.GroupedPlans(plans, Bs, Cs)
    g()
    torch.cuda.synchronize()
    for C, ref in zip(Cs, refs):
        assert torch.equal(C, ref)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        g()
    for _ in range(3):
        for C in Cs:
            C.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for C, ref in zip(Cs, refs):
            assert torch.equal(C, ref)
    del graph
    n = [max(1, s[3] // 3) for s in sizes]
    n[1], n[4] = 0, 0  # nothing to do for a streamed one and another
    part = [torch.full((s[0], max(k, 1)), 7.0, device="cuda") for s, k in zip(sizes, n)]
    g.rebind(Bs, part, n=n)
    g()
    torch.cuda.synchronize()
    for C, ref, k in zip(part, refs, n):
        assert torch.equal(C[:, :k], ref[:, :k]) and (k or bool((C == 7.0).all()))
    g.close()
    only = srt.cnn.GroupedPlans([p for p, s in zip(plans, streamed) if s], [b for b, s in zip(Bs, streamed) if s],
                                [c for c, s in zip(Cs, streamed) if s])
    for C in Cs:
        C.zero_()
    only()
    torch.cuda.synchronize()
    for C, ref, s in zip(Cs, refs, streamed):
        assert torch.equal(C, ref) if s else not bool(C.any())
    assert only.info()["workgroups"] > 0
    # what cannot share a launch is still refused beside a streamed plan
    other = srt.MatMulSpecialized.from_csr(torch.eye(64).to_sparse_csr(), 5, mapping_id=srt.named_mapping(8, "orig"))
    with pytest.raises(srt.SrtError, match="executors"):
        srt.cnn.GroupedPlans([plans[1], plans[4], other], [Bs[1], Bs[4], Bs[4]], [Cs[1], Cs[4], Cs[4]])


def test_gather_schedule_is_built_on_the_plan_s_device_only(srt):
    """A problem table entry of a streamed plan, asked for with another GPU
    current: refused, and built when its own is."""
    import ctypes as ct

    import torch
    if torch.cuda.device_count() < 2:
        pytest.skip("needs two GPUs")
    A = srt.workloads.magnitude_pruned(64, 100, 0.7, seed=3)
    plan = _plan(srt, torch, A, 64)
    out = (ct.c_uint8 * 128)()
    fill = srt._lib.lib().srt_exec_problem_fill
    with torch.cuda.device(1):
        assert fill(plan._h, None, 64, None, 64, 0, 1, 0, ct.byref(out)) == srt._lib.SRT_ERR_INVALID
    assert fill(plan._h, None, 64, None, 64, 0, 1, 0, ct.byref(out)) == 0
