"""Where a plan streams, and in which launch shape.

The time model of the streamed executor is restated here; a streamed plan
whose lane width and rows per wave are left open takes the model's choice, the
one `autotune.tuned_plan` takes.  A plan of the 1-row mapping that leaves the
executor open streams only where that is estimated to pay.
"""
import random

import pytest

COST = {1: (7000.0, 2.8, 4000.0), 2: (5600.0, 4.7, 2500.0), 4: (4800.0, 8.5, 2000.0)}


def model(M, K, nnz, N):
    best = (1, 1, float("inf"))
    for V, (staging, per_entry, per_tile) in COST.items():
        tiles = -(-max(K, 1) // (256 // V))
        for R in (1, 2, 4, 8):
            groups = -(-M // (16 * R)) * -(-max(N, 1) // (64 * V))
            entries = 16 * R * (nnz / max(1, M * tiles) + 1.5)
            t = 2.2e-6 + -(-groups // 256) * tiles * max(staging, per_entry * entries + per_tile) / 2.4e9
            if t < best[2]:
                best = (V, R, t)
    return best


def test_estimate_is_the_model(srt):
    r = random.Random(1)
    sizes = [(0, 0, 0, 0), (1, 1, 0, 1), (4096, 1024, 838860, 2048)]
    sizes += [(int(2 ** r.uniform(0, 15)), int(2 ** r.uniform(0, 15)), int(2 ** r.uniform(0, 26)), int(2 ** r.uniform(0, 14)))
              for _ in range(300)]
    for s in sizes:
        V, R, t = srt.autotune.streamed_launch(*s)
        want = model(*s)
        assert abs(t - want[2]) <= 1e-9 * want[2]
        assert (V, R) == want[:2]
    with pytest.raises(srt.SrtError):
        srt.autotune.streamed_launch(-1, 1, 1, 1)


@pytest.mark.parametrize("M,K,s,N,streams", [
    (4096, 1024, 0.8, 2048, True), (7669, 3554, 0.8781, 284, True), (12609, 214, 0.944, 309, True),
    # slower streamed: 47 us (41 gathered), 24.0 (21.3), 6.4 (5.6), 6.2 (5.1)
    (3150, 1957, 0.9663, 852, False), (1779, 138, 0.9534, 7704, False), (2725, 223, 0.9804, 299, False),
    (503, 36, 0.9897, 5314, False), (3835, 2508, 0.7, 3, False), (512, 512, 0.95, 8, False)])
def test_tuned_rule_streams_with_a_margin(srt, M, K, s, N, streams):
    assert srt.autotune.stream_pays(M, K, int((1 - s) * M * K), N) == streams


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,s,N,cfg,streams", [
    (38, 7159, 0.9989, 365, {}, False),   # all of B for a few rows' entries: 37 us, 4.9 gathered
    (145, 4000, 0.998, 3, {}, False),
    (4096, 1024, 0.8, 2048, {}, True),
    (4096, 1024, 0.8, 16, {}, False),
    (4096, 1024, 0.8, 2048, dict(nsplit=1), True),
    (4096, 1024, 0.8, 2048, dict(nsplit=4), False),
    (4096, 1024, 0.8, 2048, dict(chunk_cols=64), False),
    (4096, 1024, 0.8, 2048, dict(b_staging=2), False),
    (38, 7159, 0.9989, 365, dict(b_staging=3), True)])
def test_open_plans_stream_where_it_pays(srt, M, K, s, N, cfg, streams):
    import torch
    csr = (torch.rand(M, K, device="cuda") >= s).float().to_sparse_csr()
    plan = srt.MatMulSpecialized.from_csr(csr, N, mapping_id=srt.named_mapping(1, "identity"),
                                          tile_config=srt.TileConfig(**cfg))
    real = plan.get_config()
    assert (real.b_staging == 3) == streams
    if streams:
        V, R, _ = srt.autotune.streamed_launch(M, K, csr.values().numel(), N)
        assert (real.vec_width, real.chunk_cols, real.waves_per_block) == (V, R, 16)
    if cfg.get("nsplit", 0) > 1 or cfg.get("chunk_cols"):
        assert (real.nsplit, real.chunk_cols) == (cfg.get("nsplit", real.nsplit), cfg.get("chunk_cols", real.chunk_cols))


@pytest.mark.gpu
def test_a_streamed_configuration_on_another_mapping(srt):
    """Its rows per wave are not taken for packed columns per wave."""
    import torch
    csr = (torch.rand(2048, 1024, device="cuda") >= 0.8).float().to_sparse_csr()
    cfg = srt.MatMulSpecialized.from_csr(csr, 512, mapping_id=srt.named_mapping(1, "identity"),
                                         tile_config=srt.TileConfig(b_staging=3)).get_config()
    assert cfg.b_staging == 3 and cfg.chunk_cols <= 8 and cfg.nsplit == 1
    real = srt.MatMulSpecialized.from_csr(csr, 512, mapping_id=srt.named_mapping(4, "orig"), tile_config=cfg).get_config()
    same = srt.TileConfig(vec_width=cfg.vec_width, waves_per_block=cfg.waves_per_block)
    want = srt.MatMulSpecialized.from_csr(csr, 512, mapping_id=srt.named_mapping(4, "orig"), tile_config=same).get_config()
    assert (real.b_staging, real.chunk_cols, real.nsplit) == (2, want.chunk_cols, want.nsplit)
