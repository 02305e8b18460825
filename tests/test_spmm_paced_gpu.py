"""The SpMM's two loops are bitwise equal: the same product with a dense operand
just below and just at the sizes where the rule changes loops (32 MiB for rows
that fill a group of 32 lanes, 56 MiB for groups of 16, 32 and full ones of 64)."""

import pytest
import torch

import flagsparse_amd as fs
from flagsparse_amd import _lib, _plan

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _shares(dtype, n, rows):
    lanes = _plan.lanes_for_dense(n, torch.empty(0, dtype=dtype).element_size())
    return _lib.load().fsp_spmm_shares_nonzeros(_lib.value_code(dtype), lanes, n, n, rows, 0)


@pytest.mark.parametrize("index", [torch.int32, torch.int64], ids=["i32", "i64"])
@pytest.mark.parametrize("dtype,n,limit", [(torch.float32, 40, 56), (torch.float32, 64, 56), (torch.float32, 128, 32),
                                           (torch.float32, 256, 56), (torch.float64, 32, 56), (torch.float64, 64, 32),
                                           (torch.bfloat16, 128, 56), (torch.float16, 200, 56)])
def test_loops_agree(device, dtype, n, limit, index):
    row_bytes = n * torch.empty(0, dtype=dtype).element_size()
    rows = -(-limit * MIB // row_bytes)
    assert _shares(dtype, n, rows - 1) == 1 and _shares(dtype, n, rows) == 0
    g = torch.Generator().manual_seed(n)
    lengths = torch.randint(0, 70, (2000,), generator=g)
    lengths[77] = 1500  # segments
    ptr = torch.zeros(2001, dtype=torch.int64)
    ptr[1:] = lengths.cumsum(0)
    idx = torch.randint(0, rows - 1, (int(ptr[-1]),), generator=g)
    val = torch.randn(idx.numel(), generator=g).to(dtype).to(device)
    B = torch.randn(rows, n, device=device).to(dtype)
    results = []
    for k, it in ((rows - 1, torch.int32), (rows - 1, index), (rows, index)):
        h = fs.CsrMatrix(idx.to(it).to(device), ptr.to(it).to(device), (2000, k)).handle
        results.append(h.spmm(val, B[:k]))
        results.append(h.spmm(val, B[:k], max_blocks=8))
    for C in results[1:]:
        assert torch.equal(C, results[0])
