"""Dense widths around the 16-byte vector (one vector, one element to either
side, several vectors plus a remainder, more than one lane group) and dense
operands off 16-byte boundaries: the last lane's vector is moved back inside
the row, so every width runs the vector loads."""

import numpy as np
import pytest
import torch

import flagsparse_amd as fs
from flagsparse_amd import synthetic
from oracle import oracle

from ._helpers import assert_rel, device_csr, np_dtype_round

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16, torch.float16],
                         ids=["f32", "f64", "bf16", "f16"])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 8, 9, 31, 75, 129, 257, 515])
def test_any_dense_width(device, dtype, n):
    """Values against the oracle, and nothing written beside the result."""
    m, k = 211, 190
    ip, ix, v = synthetic.random_csr(m, k, 0.08, seed=n)
    data, idx, ptr = device_csr(ip, ix, v, device, dtype)
    h = fs.CsrMatrix(idx, ptr, (m, k)).handle
    rng = np.random.default_rng(n)
    Bn, dCn = rng.standard_normal((k, n)), rng.standard_normal((m, n))
    # operands start one element past a 16-byte boundary
    B = torch.empty(k * n + 1, dtype=dtype, device=device)[1:].view(k, n).copy_(torch.tensor(Bn))
    dC = torch.empty(m * n + 1, dtype=dtype, device=device)[1:].view(m, n).copy_(torch.tensor(dCn))
    guarded = torch.full((m * n + 2,), 7.0, dtype=dtype, device=device)
    C = guarded[1:-1].view(m, n)
    h.spmm(data, B, out=C)
    assert guarded[0] == 7.0 and guarded[-1] == 7.0
    vr, Br, dCr = np_dtype_round(v, dtype), np_dtype_round(Bn, dtype), np_dtype_round(dCn, dtype)
    assert_rel(C, oracle.spmm(ip, ix, vr, Br, (m, k)), dtype, "spmm")
    dots = oracle.sddmm(ip, ix, dCr, Br)
    assert_rel(h.sddmm(dC, B), dots, dtype, "sddmm")
    fused = h.spmm_trans_sddmm(data, dC, B)
    if n <= 64 * (16 // data.element_size()):
        dB, dv = fused
        assert torch.equal(dB, h.spmm(data, dC, transpose=True))
        assert_rel(dB, oracle.spmm(ip, ix, vr, dCr, (m, k), "trans"), dtype, "dB")
        assert_rel(dv, dots, dtype, "dvalues")
    else:
        assert fused is None


def test_ragged_width_keeps_infinities(device):
    """A column that two lanes load counts once, also when it is infinite: a
    product with a masked zero would turn it into NaN."""
    m, k, n = 64, 50, 5
    ip, ix, v = synthetic.random_csr(m, k, 0.2, seed=3)
    data, idx, ptr = device_csr(ip, ix, np.abs(v) + 1.0, device)
    h = fs.CsrMatrix(idx, ptr, (m, k)).handle
    X, Y = torch.ones(m, n, device=device), torch.ones(k, n, device=device)
    X[:, 3] = float("inf")
    assert torch.all(torch.isposinf(h.sddmm(X, Y)))
    dB, dv = h.spmm_trans_sddmm(data, X, Y)
    assert torch.all(torch.isposinf(dv))
    used = torch.zeros(k, dtype=torch.bool, device=device)
    used[idx.long()] = True
    assert torch.all(torch.isposinf(dB[used][:, 3])) and torch.isfinite(dB[used][:, [0, 1, 2, 4]]).all()


@pytest.mark.parametrize("n", [111, 112, 128])
@pytest.mark.parametrize("rows", [49151, 49152, 56173])  # B of 24 MiB at 128 columns, at 112
def test_spmm_where_wide_rows_change_kernels(device, rows, n):
    """Dense operands on either side of 24 MiB whose rows fill their lane group or not."""
    g = torch.Generator(device="cpu").manual_seed(rows + n)
    lengths = torch.randint(0, 40, (700,), generator=g)
    lengths[3] = 900  # segments
    ptr = torch.zeros(701, dtype=torch.int32)
    ptr[1:] = lengths.cumsum(0)
    idx = torch.randint(0, rows, (int(ptr[-1]),), generator=g, dtype=torch.int32)
    val = torch.randn(idx.numel(), generator=g)
    B = torch.randn(rows, n, generator=g)
    h = fs.CsrMatrix(idx.to(device), ptr.to(device), (700, rows)).handle
    C = h.spmm(val.to(device), B.to(device)).cpu().double()
    row = torch.repeat_interleave(torch.arange(700), lengths)
    ref = torch.zeros(700, n, dtype=torch.float64).index_add_(0, row, val.double()[:, None] * B.double()[idx.long()])
    assert (C - ref).abs().max() <= 1e-5 * ref.abs().max()
