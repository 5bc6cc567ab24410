"""Host side of csr.spmm: which tensors of the matrix reach the kernel."""
import importlib

import pytest


class Index:
    """A tensor as `_parts` sees one, on a device that need not exist."""

    def __init__(self, dtype, device, log):
        self.dtype, self.device, self.log = dtype, device, log
        self.is_cuda = device is not None

    def get_device(self):
        return -1 if self.device is None else self.device

    def is_contiguous(self):
        return True

    def contiguous(self):
        return self

    def cuda(self):
        return self.to(device="cuda")

    def to(self, *args, **kw):
        self.log.append(self.device)
        return Index(kw.get("dtype", self.dtype), 0, self.log)


@pytest.mark.parametrize("device,moved", [(0, False), (1, True), (None, True)])
def test_a_matrix_elsewhere_is_moved_to_the_current_device(monkeypatch, device, moved):
    """A matrix of another GPU (or the host) is copied to the current device
    and never passed by its own pointers; one that is there is used as it is."""
    import torch
    csr = importlib.import_module("sparse-register-tiling_amd").csr
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    log = []

    class A:
        layout, is_cuda = torch.sparse_csr, device is not None

        def dim(self):
            return 2

        def get_device(self):
            return -1 if device is None else device

        def crow_indices(self):
            return Index(torch.int64, device, log)

        col_indices = crow_indices

        def values(self):
            return Index(torch.float32, device, log)

    parts = csr._parts(A())
    assert [p.get_device() for p in parts] == [0, 0, 0]
    assert bool(log) == moved
