"""The work a program gives this framework, as cases that can be timed.

Every case is a sparse weight matrix times a dense matrix, through a public entry point.  Sizes are those of the
package's own workloads (pruned feed-forward layers, 1x1 convolutions of a ResNet-50, resident serving weights) and
generic ones between them.

* ``ffn``      ``autotune.tuned_plan``: the call the README shows; one layer of a pruned feed-forward block at a given
               number of tokens, from a decode step (N of a few tokens) to a prefill (N in the thousands);
* ``plain``    ``MatMulSpecialized.from_csr`` with its default mapping and launch, int32 indices, ragged sizes;
* ``hybrid``   ``MatMulSpecialized`` with ``dense_threshold``: dense 16-row panels on matrix cores, the rest not;
* ``csr``      ``csr.spmm``: a matrix used as it is, without packing;
* ``panels``   ``precision.PanelPlan`` (BF16 or FP8): the fp32 activations are converted on each call;
* ``cnn``      ``cnn.CnnFp32``: the sixteen 1x1 convolutions of a network in one grouped launch;
* ``serving``  ``serving.Server.run_batch``: one batch of BF16 requests over resident weights.
"""
import importlib
import math
import random

import torch

srt = importlib.import_module("sparse-register-tiling_amd")


def listed():
    return [
        # the smallest layer of the pruned feed-forward set: a call is all latency
        {"name": "ffn_small", "kind": "ffn", "M": 512, "K": 512, "sparsity": 0.95, "N": 128},
        # the layer the package quotes its headline figure on
        {"name": "ffn_up", "kind": "ffn", "M": 2048, "K": 512, "sparsity": 0.90, "N": 512},
        # a down projection, mildly pruned: the heaviest of the set per token
        {"name": "ffn_down", "kind": "ffn", "M": 1024, "K": 4096, "sparsity": 0.70, "N": 512},
        # prefill: thousands of tokens through one up projection
        {"name": "ffn_prefill", "kind": "ffn", "M": 4096, "K": 1024, "sparsity": 0.80, "N": 2048},
        # decode: eight sequences, one token each
        {"name": "ffn_decode", "kind": "ffn", "M": 4096, "K": 1024, "sparsity": 0.90, "N": 8},
        # sizes that divide nothing, default mapping and launch
        {"name": "plain_ragged", "kind": "plain", "M": 1000, "K": 777, "sparsity": 0.80, "N": 333},
        # a matrix with many panels dense enough for matrix cores
        {"name": "hybrid_down", "kind": "hybrid", "M": 1024, "K": 4096, "sparsity": 0.60, "N": 512,
         "threshold": 0.25},
        # an unpacked CSR matrix
        {"name": "csr_up", "kind": "csr", "M": 2048, "K": 512, "sparsity": 0.90, "N": 256, "index": "int64"},
        # reduced-precision panels, the activations converted in the call
        {"name": "panels_bf16", "kind": "panels", "M": 4096, "K": 1024, "sparsity": 0.60, "N": 512, "dtype": "bf16"},
        {"name": "panels_fp8", "kind": "panels", "M": 1024, "K": 4096, "sparsity": 0.50, "N": 512, "dtype": "fp8"},
        # one image through the 1x1 convolutions of a ResNet-50
        {"name": "cnn_batch1", "kind": "cnn", "batch": 1},
        # a batch of requests of mixed widths over four resident weights
        {"name": "serving_batch", "kind": "serving", "requests": 24, "n_max": 256, "mix": 0},
    ]


#: nnz * N of the costliest listed case: no drawn case costs more.
MOST = 4096 * 1024 * 0.2 * 2048


def _between(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi]; odd ones among them."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    r = rng.random()
    return max(lo, min(hi, v if r < 0.5 else -(-v // 8) * 8 if r < 0.75 else -(-v // 64) * 64))


def draw(rng):
    kind = rng.choice(["ffn", "ffn", "ffn", "plain", "plain", "hybrid", "csr", "panels", "panels", "cnn", "serving"])
    if kind == "cnn":
        return {"kind": "cnn", "batch": rng.randint(1, 4)}
    if kind == "serving":
        return {"kind": "serving", "requests": rng.randint(4, 48), "n_max": _between(rng, 16, 512),
                "mix": rng.randint(1, 1 << 20)}
    while True:
        c = {"kind": kind, "M": _between(rng, 256, 4096), "K": _between(rng, 128, 4096),
             "sparsity": round(rng.uniform(0.5, 0.75) if kind in ("hybrid", "panels") else rng.uniform(0.65, 0.97), 3),
             "N": _between(rng, 1 if kind in ("ffn", "plain", "csr") else 32, 4096)}
        dense = kind in ("hybrid", "panels")
        cost = c["M"] * c["K"] * c["N"] * (0.2 if dense else 1.0 - c["sparsity"])
        if cost <= (0.5 if dense else 1.0) * MOST:
            break
    if kind == "hybrid":
        c["threshold"] = rng.choice([0.2, 0.25, 0.3, 0.35, 0.4])
    if kind == "csr":
        c["index"] = rng.choice(["int32", "int64"])
    if kind == "panels":
        c["dtype"] = rng.choice(["bf16", "fp8"])
    return c


# ------------------------------------------------------------------ inputs
def _generator(seed, salt=0):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + salt) % (1 << 62))


def _pruned(M, K, sparsity, seed, salt=0):
    """A magnitude-pruned weight matrix (dense, on the GPU): normal entries, log-normal row scales, the largest kept."""
    g = _generator(seed, salt)
    W = torch.randn((M, K), generator=g, device="cuda")
    W *= torch.exp(0.5 * torch.randn((M, 1), generator=g, device="cuda"))
    keep = max(1, int(round((1.0 - sparsity) * M * K)))
    cut = torch.topk(W.abs().reshape(-1), keep).values[-1]
    return torch.where(W.abs() >= cut, W, torch.zeros_like(W))


def _activations(K, N, seed, salt=1):
    return torch.rand((K, N), generator=_generator(seed, salt), device="cuda") * 2 - 1


def _csr(A, index=torch.int64):
    rows, cols = torch.nonzero(A, as_tuple=True)
    rp = torch.zeros(A.shape[0] + 1, dtype=torch.int64, device=A.device)
    rp[1:] = torch.cumsum(torch.bincount(rows, minlength=A.shape[0]), 0)
    return torch.sparse_csr_tensor(rp.to(index), cols.to(index), A[rows, cols], size=tuple(A.shape))


def _requests(case):
    """(weight, N) of each request: any weight, widths spread over their logarithm, as arrivals mix them."""
    r = random.Random(int(case["mix"]))
    return [(r.randrange(len(SERVED)), max(1, int(round(math.exp(r.uniform(0.0, math.log(case["n_max"])))))))
            for _ in range(int(case["requests"]))]


SERVED = [(1024, 1024), (1024, 1024), (4096, 1024), (1024, 4096)]


def _served_weights(seed):
    return [_pruned(M, K, 0.9, seed, 10 + i).to(torch.bfloat16).to(torch.float32) for i, (M, K) in enumerate(SERVED)]


def _served_operands(case, seed):
    return [_activations(SERVED[w][1], n, seed, 100 + i).to(torch.bfloat16) for i, (w, n) in enumerate(_requests(case))]


def _cnn_weights(seed):
    """Dense copies of the layers' weights: each entry kept on its own, a sparsity per layer."""
    r, out = random.Random(int(seed)), []
    for i, (_, _, M, K) in enumerate(srt.cnn.RN50_1X1):
        s, g = r.uniform(0.80, 0.98), _generator(seed, 200 + i)
        keep = torch.rand((M, K), generator=g, device="cuda") >= s
        out.append((s, torch.randn((M, K), generator=g, device="cuda") * keep))
    return out


def _cnn_activations(case, seed):
    return [_activations(K, hw * case["batch"], seed, 300 + i) for i, (_, hw, _, K) in enumerate(srt.cnn.RN50_1X1)]


# ------------------------------------------------------------------ a program's state, a pass
def prepare(case, seed):
    kind = case["kind"]
    if kind == "serving":
        server = srt.serving.Server(srt.serving.RegTileWeights(_served_weights(seed)))
        return {"kind": kind, "server": server, "asked": _requests(case), "B": _served_operands(case, seed)}
    if kind == "cnn":
        layers = [srt.cnn.CnnLayer(name, hw, M, K, s, _csr(W).cpu())
                  for (name, hw, M, K), (s, W) in zip(srt.cnn.RN50_1X1, _cnn_weights(seed))]
        return {"kind": kind, "net": srt.cnn.CnnFp32(layers, case["batch"], _cnn_activations(case, seed))}
    A = _pruned(case["M"], case["K"], case["sparsity"], seed)
    st = {"kind": kind, "B": _activations(case["K"], case["N"], seed),
          "C": torch.empty((case["M"], case["N"]), device="cuda")}
    if kind == "ffn":
        st["plan"] = srt.autotune.tuned_plan(_csr(A), case["N"])
    elif kind == "plain":
        st["plan"] = srt.MatMulSpecialized.from_csr(_csr(A, torch.int32), case["N"])
    elif kind == "hybrid":
        st["plan"] = srt.MatMulSpecialized.from_csr(_csr(A), case["N"], mapping_id=srt.named_mapping(4, "orig"),
                                                    dense_threshold=case["threshold"])
    elif kind == "csr":
        st["A"] = _csr(A, getattr(torch, case["index"]))
    else:
        st["plan"] = srt.precision.PanelPlan.from_csr(_csr(A), case["dtype"])
    return st


def run(st):
    kind = st["kind"]
    if kind == "serving":
        batch = [srt.serving.Request(rid=i, weight=w, B=B) for i, ((w, _), B) in enumerate(zip(st["asked"], st["B"]))]
        st["server"].run_batch(batch)
        return [r.C for r in batch]
    if kind == "cnn":
        return st["net"]()
    if kind == "csr":
        return srt.csr.spmm(st["A"], st["B"], st["C"])
    if kind == "panels":
        Bq, scales = st["plan"].prepare_b(st["B"])
        return {"C": st["plan"](st["C"], Bq, scales), "Bq": Bq, "scales": scales}
    return st["plan"](st["C"], st["B"])


# ------------------------------------------------------------------ what a pass cannot do without, and its values
def work(case):
    if case["kind"] == "serving":
        asked = _requests(case)
        nnz = [0.1 * M * K for M, K in SERVED]
        return {"bytes": sum(nnz[w] * 4 for w in {w for w, _ in asked})
                + sum(n * (2 * SERVED[w][1] + 4 * SERVED[w][0]) for w, n in asked),
                "flops": sum(2 * nnz[w] * n for w, n in asked)}
    if case["kind"] == "cnn":
        layers = [(M, K, hw * case["batch"]) for _, hw, M, K in srt.cnn.RN50_1X1]
        return {"bytes": sum(4 * (0.11 * M * K + K * n + M * n) for M, K, n in layers),
                "flops": sum(2 * 0.11 * M * K * n for M, K, n in layers)}
    M, K, N = case["M"], case["K"], case["N"]
    nnz = (1.0 - case["sparsity"]) * M * K
    b = 4 * (nnz + K * N + M * N)
    if case["kind"] == "panels":  # the converted operand is an output too
        b += K * N * (2 if case["dtype"] == "bf16" else 1)
    return {"bytes": b, "flops": 2 * nnz * N}


def exact(case, seed):
    if case["kind"] == "serving":
        W = [w.double() for w in _served_weights(seed)]
        return [W[w] @ B.double() for (w, _), B in zip(_requests(case), _served_operands(case, seed))]
    if case["kind"] == "cnn":
        return [W.double() @ X.double() for (_, W), X in zip(_cnn_weights(seed), _cnn_activations(case, seed))]
    C = _pruned(case["M"], case["K"], case["sparsity"], seed).double() @ _activations(case["K"], case["N"], seed).double()
    return {"C": C, "Bq": None, "scales": None} if case["kind"] == "panels" else C
