"""The SpMM with values wider than the dense operands (the COO product's
numerics): long rows whose partials are kept in the wide type, ragged widths,
64-bit row pointers, an `out` that is B's own memory, and the pairs of types
that have no kernel."""

import numpy as np
import pytest
import torch

import flagsparse_amd as fs
from flagsparse_amd._matrix import CsrHandle
from oracle import oracle

from ._helpers import device_csr, long_row_matrix, np_dtype_round

pytestmark = pytest.mark.gpu

# one rounding of the storage type on top of a wider sum: half an ulp of the
# largest element, plus the wide sum's own rounding
STORE_EPS = {torch.float32: 2.0**-24, torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}
WIDE = {torch.float32: torch.float64, torch.bfloat16: torch.float32, torch.float16: torch.float32}


@pytest.mark.parametrize("dtype", list(WIDE), ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("index_dtype", [torch.int32, torch.int64], ids=["i32", "i64"])
@pytest.mark.parametrize("n", [1, 3, 8, 50, 129])
def test_wide_values(device, dtype, index_dtype, n):
    m, k = 400, 3000
    ip, ix, v = long_row_matrix(m, k, [0, 77, 399], 1700, 6, seed=n)
    data, idx, ptr = device_csr(ip, ix, v, device, WIDE[dtype], index_dtype)
    Bn = np.random.default_rng(n).standard_normal((k, n))
    B = torch.tensor(Bn, dtype=dtype, device=device)
    C = CsrHandle(idx, ptr, (m, k)).spmm(data, B)
    assert C.dtype == dtype
    ref = oracle.spmm(ip, ix, np_dtype_round(v, WIDE[dtype]), np_dtype_round(Bn, dtype), (m, k))
    err = np.abs(C.double().cpu().numpy() - ref)
    # f32 sums of 1700 products under the 16-bit types: 1700 * 2^-24 of sum |a b|
    sums = oracle.spmm(ip, ix, np.abs(np_dtype_round(v, WIDE[dtype])), np.abs(np_dtype_round(Bn, dtype)), (m, k))
    acc = 1700 * 2.0**-24 if WIDE[dtype] == torch.float32 else 1700 * 2.0**-53
    assert np.all(err <= STORE_EPS[dtype] * np.abs(ref) + 2 * acc * sums + 1e-30)


def test_out_is_bs_memory(device):
    """out= may be B itself: the product is formed beside it first."""
    rng = np.random.default_rng(5)
    n = 300
    row, col = rng.integers(0, n, 2500), rng.integers(0, n, 2500)
    data = torch.tensor(rng.standard_normal(2500), dtype=torch.float32, device=device)
    r, c = (torch.tensor(t, dtype=torch.int32, device=device) for t in (row, col))
    B = torch.randn(n, 40, device=device)
    want = fs.flagsparse_spmm_coo(data, r, c, B, (n, n))
    out = B.clone()
    assert fs.flagsparse_spmm_coo(data, r, c, out, (n, n), out=out) is out
    assert torch.equal(out, want)


def test_pairs_without_a_kernel(device):
    ip, ix, v = long_row_matrix(40, 60, [0], 30, 4, seed=1)
    data, idx, ptr = device_csr(ip, ix, v, device, torch.float32)
    h = CsrHandle(idx, ptr, (40, 60))
    with pytest.raises(TypeError, match="no kernel"):
        h.spmm(data, torch.randn(60, 8, dtype=torch.float64, device=device))
    with pytest.raises(TypeError, match="no kernel"):
        h.spmm(data.double(), torch.randn(60, 8, dtype=torch.float16, device=device))
