"""Launches for host tensors are refused before any address reaches the GPU."""

import pytest
import torch

from flagsparse_amd import _csc, _lib, _plan
from flagsparse_amd._matrix import CsrHandle


class _NoLaunch:
    """Stands for the library: every launch fails the test."""

    def __getattr__(self, name):
        if name.endswith("_workspace"):
            return lambda *a: 0
        return lambda *a: pytest.fail(f"{name} was called with host addresses")


def test_stream_of_a_host_device():
    with pytest.raises(ValueError, match="cuda device"):
        _lib.stream_ptr(torch.device("cpu"))


@pytest.mark.parametrize("call", [
    lambda h, v, p: h.spmm(v, torch.ones(3, 2)), lambda h, v, p: h.spmm(v, torch.ones(2, 2), transpose=True),
    lambda h, v, p: h.spmv(v, torch.ones(3)), lambda h, v, p: h.sddmm(torch.ones(2, 2), torch.ones(3, 2)),
    lambda h, v, p: _csc.gather_values(v, p), lambda h, v, p: _csc.csr_to_csc_perm(h.indptr, h.indices, 2, 3),
    lambda h, v, p: _plan.build_plan(h.indptr, 2, _plan.spmm_config(4)),
    lambda h, v, p: _plan.inspect_csr(h.indptr, h.indices, 2, 3),
])
def test_host_tensors(monkeypatch, call):
    monkeypatch.setattr(_lib, "load", lambda: _NoLaunch())
    h = CsrHandle(torch.tensor([0, 1, 2], dtype=torch.int32), torch.tensor([0, 1, 3], dtype=torch.int32), (2, 3))
    with pytest.raises(ValueError, match="cuda device"):
        call(h, torch.ones(3), torch.arange(3, dtype=torch.int32))


def test_index_of_a_device(monkeypatch):
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 5)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 100 + index, raising=False)
    for _ in range(2):
        assert _lib.stream_ptr(torch.device("cuda:3")) == 103 and _lib.stream_ptr(torch.device("cuda:0")) == 100
        assert _lib.stream_ptr(torch.device("cuda")) == _lib.stream_ptr() == 105
        with pytest.raises(ValueError, match="cuda device"):
            _lib.stream_ptr(torch.device("cpu:0"))
