"""The transposed products' two ways to the values: read through the
permutation inside the kernel (values of at most 2 MiB) or gathered first.
Both give the same bits; the gather itself at its remainders."""

import numpy as np
import pytest
import torch

import flagsparse_amd as fs
from flagsparse_amd import _matrix
from flagsparse_amd._csc import gather_values

from ._helpers import device_csr, long_row_matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16], ids=["f32", "f64", "bf16"])
@pytest.mark.parametrize("n", [1, 8, 31, 64, 200])
def test_permuted_and_gathered_values_agree(device, dtype, n, monkeypatch):
    ip, ix, v = long_row_matrix(600, 900, [3, 599], 800, 7, seed=n)  # long columns of A^T: segments
    data, idx, ptr = device_csr(ip, ix, v, device, dtype)
    h = fs.CsrMatrix(idx, ptr, (600, 900)).handle
    dC = torch.randn(600, n, device=device).to(dtype)
    B = torch.randn(900, n, device=device).to(dtype)
    results = []
    for in_kernel in (False, True):
        monkeypatch.setattr(_matrix, "_permuted_in_kernel", lambda *a, _v=in_kernel: _v)
        fused = h.spmm_trans_sddmm(data, dC, B)
        assert (fused is None) == (n > 64 * (16 // data.element_size()))  # wider than one lane group
        results.append((h.spmm(data, dC, transpose=True), *(fused or ())))
    for a, b in zip(*results):
        assert torch.equal(a, b)
    monkeypatch.undo()
    # values change between calls, the handle stays
    assert torch.equal(h.spmm(data * 2, dC, transpose=True), results[0][0] * 2)


@pytest.mark.parametrize("dtype", [torch.uint8, torch.bfloat16, torch.float32, torch.float64, torch.complex128])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 70001, (8 << 20) // 8, (8 << 20) // 8 + 1])
def test_gather_remainders(device, dtype, n):
    x = torch.tensor(np.random.default_rng(n).integers(0, 100, n + 1), device=device).to(dtype)[1:]  # off alignment
    for perm_dtype in (torch.int32, torch.int64):
        p = torch.randperm(n, device=device).to(perm_dtype)
        assert torch.equal(gather_values(x, p), x[p.long()])
