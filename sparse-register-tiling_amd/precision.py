"""Precision form: BF16 and FP8-e4m3 SpMM on MFMA over 16-row dense panels.

No counterpart in the reference (its executors are FP32 only,
tools/codegen/gen_vector_specialized.py:266-349).  A is cut into 16-row panels
and 32-column blocks; every block holding a nonzero is stored dense in the
MFMA operand layout (the reference's ILP padding, sbench/ilp_pad/
nano_solver.py:76-116, taken to dense 16-row panels) and empty blocks are
skipped.  Accumulation is FP32.  FP8 uses per-row scales of A and per-column
scales of B, both computed in FP64 on the device:

    C_ij = s_i * t_j * sum_k e4m3(A_ik / s_i) * e4m3(B_kj / t_j)

    plan = PanelPlan.from_csr(A_csr, dtype="bf16")      # or "fp8"
    Bt, t = plan.prepare_b(B)                             # fp32 -> transposed bf16 / e4m3 (+ scales)
    plan(C, Bt, t)                                        # C = A . B  (fp32)
"""
from __future__ import annotations

import ctypes as ct
import functools
from typing import Dict, Optional, Tuple

import numpy as np
import torch

from . import _lib
from .native import current_raw_stream, ptr, stream_handle

DTYPES = {"bf16": _lib.SRT_DT_BF16, "fp8": _lib.SRT_DT_FP8}
# launch shapes: index -> (N tile, waves per workgroup, panels per wave)
SHAPES = {0: (64, 4, 2), 1: (128, 4, 2), 2: (64, 4, 1), 3: (128, 2, 2), 4: (32, 4, 1), 5: (128, 4, 1),
          6: (64, 8, 1), 7: (128, 8, 1), 8: (64, 16, 1), 9: (32, 8, 1)}


def _index_tensor(x, device) -> torch.Tensor:
    t = torch.as_tensor(x, device=device)
    if t.dtype not in (torch.int32, torch.int64):
        t = t.to(torch.int64)
    return t.contiguous()


# Time model of default_launch, in us: (a launch; a K block of one
# workgroup's chain, by shape; 10 KB of operand tiles of the CU with most
# workgroups; the second launch of a K split; a million floats of partial tiles).  Least squares over 66 problem
# sizes (256..4096 rows, 128..4096 deep, 32..2048 columns) times the three shapes
# times K splits of 1..32.  On average its choice takes 1.03 of the fastest
# launch's time; 64-column tiles with the K range split up to 256 workgroups,
# which it replaces, took 1.23 (512 x 512 x 100: 8.1 us, now 6.7; 2048 x 512 x
# 512: 14.2, now 7.9; 4096 x 1024 x 1024: 19.7 both).  Workgroups past a full
# chip count as a round of their own: 240 x 6214 x 4258 takes 54.0 us in 134
# workgroups of 64 columns, 60.0 in 268 of 32.
_LAUNCH_US = 5.39
_CHAIN_US = ((6, .151), (9, .103), (4, .091))
_TILE_US, _SPLIT_US, _PARTIAL_US = .101, 1.49, 1.52


def _split_limit(num_panels: int, k_blocks: int, n: int, target_groups: int = 256) -> int:
    """K splits that fill the chip with 64-column tiles of 8 panels: the most a
    default launch uses.  The fewer columns, the more splits."""
    nt, wp, pw = SHAPES[6]
    groups = -(-num_panels // (wp * pw)) * -(-n // nt)
    ks = 1
    while groups * ks * 2 <= target_groups and ks * 2 <= max(1, k_blocks // 4):
        ks *= 2
    return ks


@functools.lru_cache(maxsize=4096)
def default_launch(num_panels: int, k_blocks: int, n: int, target_groups: int = 256) -> Tuple[int, int]:
    """(shape, ksplit) of the least modelled time: wide tiles read B and A less
    often, narrow ones give more workgroups and a shorter chain per K block, a
    K split shortens the chain for a second launch and the partial tiles.
    target_groups: workgroups that fill the chip."""
    limit = _split_limit(num_panels, k_blocks, n, target_groups)
    best = None
    for shape, chain in _CHAIN_US:
        nt, wp, pw = SHAPES[shape]
        groups = -(-num_panels // (wp * pw)) * -(-n // nt)
        ks = 1
        while ks <= limit:
            steps = -(-k_blocks // ks)
            rounds = groups * ks / target_groups
            rounds = -(-groups * ks // target_groups) if rounds > 1 else rounds
            t = _LAUNCH_US + chain * steps + _TILE_US * rounds * steps * (wp * pw * 1024 + nt * 64) * 1e-4
            if ks > 1:
                t += _SPLIT_US + _PARTIAL_US * (ks + 1) * num_panels * 16 * n * 1e-6
            if best is None or t < best[0]:
                best = (t, shape, ks)
            ks *= 2
    return best[1], best[2]


@functools.lru_cache(maxsize=4096)
def split_reservation(num_panels: int, k_blocks: int) -> Tuple[int, int]:
    """(columns, K splits) of the largest workspace a default launch of any
    width can need: one reservation covers them all, at most 256 tiles of
    128 x 64 floats (8 MiB).  (0, 1) where no width is split."""
    best, columns = (0, 1), SHAPES[6][0]
    while True:
        ks = _split_limit(num_panels, k_blocks, columns)
        if ks == 1:
            return best
        if ks * columns > best[0] * best[1]:
            best = (columns, ks)
        columns += SHAPES[6][0]


class PanelPlan:
    """Packed 16-row panels of A on the device for BF16 or FP8 MFMA."""

    def __init__(self, m: int, k: int, Lx, Lp, Li, dtype: str = "bf16",
                 stream: Optional[torch.cuda.Stream] = None):
        if dtype not in DTYPES:
            raise ValueError("dtype must be 'bf16' or 'fp8'")
        device = torch.device("cuda", torch.cuda.current_device())
        Lp_t = _index_tensor(Lp, device)
        Li_t = _index_tensor(Li, device).to(Lp_t.dtype)
        Lx_t = torch.as_tensor(Lx, device=device, dtype=torch.float32).contiguous()
        if Lp_t.numel() != m + 1:
            raise ValueError("Lp must have m + 1 = %d entries" % (m + 1))
        if Li_t.numel() != Lx_t.numel():
            raise ValueError("Li and Lx must have the same length")
        self.m, self.k, self.dtype = int(m), int(k), dtype
        h = ct.c_void_p()
        _lib.call("srt_mfma_plan_create", self.m, self.k, ptr(Lx_t), ptr(Lp_t), ptr(Li_t),
                  Lp_t.element_size(), DTYPES[dtype], stream_handle(stream), ct.byref(h))
        self._h = h
        self.device = device
        self._reserved = 0  # floats of the K-split workspace
        self._lib = _lib.lib()
        st = self.stats()
        self._panels, self._k_blocks = st["num_panels"], st["k_blocks"]

    @classmethod
    def from_csr(cls, csr: torch.Tensor, dtype: str = "bf16") -> "PanelPlan":
        csr = csr.to_sparse_csr() if csr.layout != torch.sparse_csr else csr
        return cls(csr.shape[0], csr.shape[1], csr.values(), csr.crow_indices(), csr.col_indices(), dtype)

    @classmethod
    def from_dense(cls, A, dtype: str = "bf16") -> "PanelPlan":
        A = torch.as_tensor(A, dtype=torch.float32).cpu()
        return cls.from_csr(A.to_sparse_csr(), dtype)

    # -- operands -----------------------------------------------------------
    def prepare_b(self, B: torch.Tensor, stream: Optional[torch.cuda.Stream] = None
                  ) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
        """fp32 device B (K x N) -> (Bt, FP8 column scales or None): Bt is the
        B operand transposed to N x ldk (k contiguous, ldk = K rounded up to
        32, zeros past K) in the plan's dtype -- torch.bfloat16, or raw e4m3
        bytes (uint8)."""
        if not (B.is_cuda and B.dtype == torch.float32 and B.dim() == 2 and B.stride(1) == 1):
            raise ValueError("B must be a row-major 2-D float32 CUDA tensor")
        rows, cols = B.shape
        ldk = -(-rows // 32) * 32
        if self.dtype == "bf16":
            out = torch.empty((cols, ldk), dtype=torch.bfloat16, device=B.device)
            scales = None
        else:
            out = torch.empty((cols, ldk), dtype=torch.uint8, device=B.device)
            scales = torch.empty(cols, dtype=torch.float32, device=B.device)
        s = current_raw_stream(torch.cuda.current_device()) if stream is None else stream.cuda_stream
        rc = self._lib.srt_mfma_convert_b(DTYPES[self.dtype], rows, cols, B.data_ptr(), B.stride(0), out.data_ptr(), ldk,
                                          None if scales is None else scales.data_ptr(), s)
        if rc:
            _lib.check(rc)
        return out, scales

    def reserve(self, n_max: int, ksplit_max: int) -> None:
        """Workspace for K-split launches (allocates; do it before graph capture).
        A smaller one stays alive for the graphs that captured it."""
        _lib.call("srt_mfma_plan_reserve", self._h, int(n_max), int(ksplit_max))
        if ksplit_max > 1:
            self._reserved = max(self._reserved, int(ksplit_max) * self.m * int(n_max))

    def __call__(self, C: torch.Tensor, Bq: torch.Tensor, col_scales: Optional[torch.Tensor] = None,
                 n: Optional[int] = None, shape: Optional[int] = None, ksplit: Optional[int] = None,
                 stream: Optional[torch.cuda.Stream] = None) -> torch.Tensor:
        want = torch.bfloat16 if self.dtype == "bf16" else torch.uint8
        if Bq.dtype != want or not Bq.is_cuda or Bq.stride(1) != 1:
            raise ValueError("B must be the transposed CUDA %s operand from prepare_b" % want)
        if not (C.is_cuda and C.dtype == torch.float32 and C.stride(1) == 1):
            raise ValueError("C must be a row-major float32 CUDA tensor")
        n = Bq.shape[0] if n is None else int(n)
        if Bq.shape[1] < -(-self.k // 32) * 32 or C.shape[0] < self.m or C.shape[1] < n or Bq.shape[0] < n:
            raise ValueError("shape mismatch")
        chosen = ksplit is None
        if shape is None or chosen:
            dshape, dks = default_launch(self._panels, self._k_blocks, n)
            shape = dshape if shape is None else shape
            ksplit = dks if chosen else ksplit
        if ksplit > 1 and ksplit * self.m * n > self._reserved:
            if chosen:  # for every width at once
                self.reserve(*split_reservation(self._panels, self._k_blocks))
            else:
                self.reserve(n, ksplit)
        s = current_raw_stream(torch.cuda.current_device()) if stream is None else stream.cuda_stream
        rc = self._lib.srt_mfma_plan_execute(self._h, C.data_ptr(), C.stride(0), Bq.data_ptr(), Bq.stride(0),
                                             None if col_scales is None else col_scales.data_ptr(), n, int(shape),
                                             int(ksplit), s)
        if rc:
            _lib.check(rc)
        return C

    # -- inspection -----------------------------------------------------------
    def stats(self) -> Dict[str, int]:
        s = _lib.MfmaStatsC()
        _lib.call("srt_mfma_plan_stats_get", self._h, ct.byref(s))
        return {f[0]: getattr(s, f[0]) for f in s._fields_}

    def row_scales(self) -> np.ndarray:
        out = np.zeros(max(1, self.m), dtype=np.float32)
        _lib.call("srt_mfma_plan_row_scales", self._h, out.ctypes.data_as(ct.c_void_p))
        return out[:self.m]

    def blocks(self) -> Dict[str, np.ndarray]:
        """Host copies: slot [P, KB] (-1 = empty block), blk_kb, blocks [n, 512]
        (uint16 BF16 bits or uint8 e4m3 codes, MFMA operand order)."""
        st = self.stats()
        P, KB, nb = st["num_panels"], st["k_blocks"], st["stored_blocks"]
        slot = np.zeros(max(1, P * KB), dtype=np.int32)
        kb = np.zeros(max(1, nb), dtype=np.int32)
        blk = np.zeros((max(1, nb), 512), dtype=np.uint16 if self.dtype == "bf16" else np.uint8)
        _lib.call("srt_mfma_plan_copy_blocks", self._h, slot.ctypes.data_as(ct.c_void_p),
                  kb.ctypes.data_as(ct.c_void_p), blk.ctypes.data_as(ct.c_void_p))
        return {"slot": slot[:P * KB].reshape(P, KB), "blk_kb": kb[:nb], "blocks": blk[:nb]}

    def close(self) -> None:
        if getattr(self, "_h", None):
            _lib.lib().srt_mfma_plan_destroy(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


def spmm(A_csr: torch.Tensor, B: torch.Tensor, dtype: str = "bf16") -> torch.Tensor:
    """One-shot C = A . B in the precision form (packs, converts B, runs)."""
    plan = PanelPlan.from_csr(A_csr, dtype)
    Bq, t = plan.prepare_b(B)
    C = torch.empty((plan.m, B.shape[1]), dtype=torch.float32, device=B.device)
    return plan(C, Bq, t)
