"""What a COO SpMM does to the tensor passed as `out`, with the kernel replaced
by one that writes the addresses it is given."""

import ctypes

import pytest
import torch
from torch.autograd import forward_ad

from flagsparse_amd import spmm_coo

A = torch.tensor([[1.0, 2.0, 0.0], [0.0, -3.0, 4.0]])


class _Kernel:
    """CsrHandle.spmm of A: reads and writes plain memory."""

    def spmm(self, data, B, out=None):
        C = A @ B.clone()
        if out is None:
            return C
        ctypes.memmove(out.data_ptr(), C.data_ptr(), C.numel() * C.element_size())
        return out


@pytest.fixture
def canonical():
    c = object.__new__(spmm_coo._CanonicalCoo)
    c.data, c.shape, c.handle = torch.ones(4), (2, 3), _Kernel()
    return c


def _B():
    return torch.arange(12.0).view(3, 4) - 5


@pytest.mark.parametrize("make", [lambda: torch.empty(2, 4), lambda: torch._neg_view(torch.empty(2, 4)),
                                  lambda: torch.empty(4, 2).t(), lambda: torch.empty(2, 9)[:, 1:5]],
                         ids=["plain", "negated", "transposed", "strided"])
def test_out_holds_the_product(canonical, make):
    out = make()
    C = canonical.spmm(_B(), "row", out=out)
    assert C is out and torch.equal(out, A @ _B())


def test_out_in_the_memory_of_B(canonical):
    B = _B()
    out = B.view(-1)[2:10].view(2, 4)
    ref = A @ B
    assert torch.equal(canonical.spmm(B, "row", out=out), ref)


def test_backward_sees_that_out_was_overwritten(canonical):
    w = torch.ones(2, 4, requires_grad=True)
    out = torch.ones(2, 4)
    loss = (w * out).sum()  # saves out
    canonical.spmm(_B(), "row", out=out)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()


def test_out_drops_its_tangent(canonical):
    with forward_ad.dual_level():
        out = forward_ad.make_dual(torch.ones(2, 4), torch.ones(2, 4))
        canonical.spmm(_B(), "row", out=out)
        primal, tangent = forward_ad.unpack_dual(out)
        assert torch.equal(primal, A @ _B()) and (tangent is None or not tangent.any())
