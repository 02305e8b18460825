"""SpMV rows that take a whole workgroup: the edges of that bin and of the long
rows' segments, every value type, plain and transposed, capped and XCD-mapped
grids, and the loops that run such a plan with one wave a row."""
import math

import pytest
import torch

import flagsparse_amd as fs
from flagsparse_amd import _plan
from flagsparse_amd._lib import FlagSparseLibraryError

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 1023, 1024, 1025, 1279, 2048, 2049, 4095, 4096, 4097, 8191, 8192, 8193, 12288, 12289, 20001, 3, 0]
# unit roundoff of the result, and of the sum: a lane adds at most 64 products
# (4096 nonzeros on 64 lanes), the trees and the segments at most 22 more
ROUND = {torch.float32: 2.0**-24, torch.float64: 0.0, torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}
SUM = {torch.float32: 100 * 2.0**-53, torch.float64: 100 * 2.0**-53, torch.bfloat16: 100 * 2.0**-24,
       torch.float16: 100 * 2.0**-24}


def _matrix(dtype, index, n_cols, seed=5):
    g = torch.Generator().manual_seed(seed)
    ptr = torch.zeros(len(LENGTHS) + 1, dtype=torch.int64)
    ptr[1:] = torch.tensor(LENGTHS).cumsum(0)
    nnz = int(ptr[-1])
    idx = torch.randint(0, n_cols, (nnz,), generator=g)
    data = torch.randn(nnz, generator=g).to(dtype)
    return data, idx.to(index), ptr.to(index)


def _check(y, data, rows, cols, x, n_out, dtype):
    prod = data.double() * x.double()[cols.long()]
    ref = torch.tensor([math.fsum(prod[rows == r].tolist()) for r in range(n_out)], dtype=torch.float64)
    mag = torch.zeros(n_out, dtype=torch.float64).index_add_(0, rows, prod.abs())
    bound = ROUND[dtype] * ref.abs() * 1.01 + SUM[dtype] * mag
    assert ((y.cpu().double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("index", [torch.int32, torch.int64])
@pytest.mark.parametrize("dtype", list(ROUND))
def test_rows_at_the_edges(dtype, index):
    n_cols = 50000
    data, idx, ptr = _matrix(dtype, index, n_cols)
    x = torch.randn(n_cols, generator=torch.Generator().manual_seed(6)).to(dtype)
    rows = torch.repeat_interleave(torch.arange(len(LENGTHS)), torch.tensor(LENGTHS))
    d, i, p, xd = (t.cuda() for t in (data, idx, ptr, x))
    cfg = _plan.spmv_wide_config()
    h = fs.CsrMatrix(i, p, (len(LENGTHS), n_cols)).handle
    plan = h.plan(cfg)
    assert plan.bin_counts[-1] == sum(1024 < n <= 4096 for n in LENGTHS)
    assert plan.n_segments == sum(-(-n // 4096) for n in LENGTHS if n > 4096)
    for kwargs in ({}, {"max_blocks": 3}, {"xcd_groups": 8, "max_blocks": 6}, {"variant": 1}):
        y = h.spmv(d, xd, config=cfg, **kwargs)
        _check(y, data, rows, idx, x, len(LENGTHS), dtype)
    if dtype in (torch.float32, torch.float64):
        prepared = fs.prepare_spmv_csr(d, i, p, (len(LENGTHS), n_cols))
        assert prepared.plan().config == cfg
        y = fs.flagsparse_spmv_csr(x=xd, prepared=prepared)
        _check(y, data, rows, idx, x, len(LENGTHS), dtype)


@pytest.mark.parametrize("variant", [0, 2, 3])
def test_transposed_and_lds(variant):
    n_rows = 3000  # x of the transposed product, small enough for LDS
    data, idx, ptr = _matrix(torch.float32, torch.int32, n_rows, seed=7)
    # A = (the matrix above)^T, so that the long rows are columns of A
    t = torch.sparse_csr_tensor(ptr, idx, torch.arange(1, data.numel() + 1, dtype=torch.float64),
                                (len(LENGTHS), n_rows), check_invariants=False).to_sparse_coo()
    r, c = t._indices()
    order = torch.sort(c * len(LENGTHS) + r, stable=True).indices
    a_ptr = torch.zeros(n_rows + 1, dtype=torch.int64)
    a_ptr[1:] = torch.bincount(c, minlength=n_rows).cumsum(0)
    h = fs.CsrMatrix(r[order].int().cuda(), a_ptr.int().cuda(), (n_rows, len(LENGTHS))).handle
    x = torch.randn(n_rows, generator=torch.Generator().manual_seed(8))
    y = h.spmv(data[order].cuda(), x.cuda(), transpose=True, config=_plan.spmv_wide_config(), variant=variant)
    _check(y, data[order], r[order], c[order], x, len(LENGTHS), torch.float32)


def test_other_kernels_refuse_a_workgroup_per_row():
    data, idx, ptr = _matrix(torch.float32, torch.int32, 500)
    h = fs.CsrMatrix(idx.cuda(), ptr.cuda(), (len(LENGTHS), 500)).handle
    with pytest.raises(FlagSparseLibraryError, match="lanes 256"):
        h.spmm(data.cuda(), torch.zeros(500, 8, device="cuda"), config=_plan.spmv_wide_config())
