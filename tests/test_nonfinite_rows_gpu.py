"""Infinite and NaN values stay in the rows that hold them.  A workgroup that
walks several row tiles has the next tile's values in registers while other
rows of its wave still run: rows of unequal length, capped and XCD-mapped
grids, every loop and value type, compared bit for bit with the product of the
same matrix without those values."""

import pytest
import torch

import flagsparse_amd as fs
from flagsparse_amd import _plan
from flagsparse_amd.autotune import TuneParams
from flagsparse_amd.batch import CsrBatch

pytestmark = pytest.mark.gpu

BAD = (float("inf"), float("-inf"), float("nan"))


def _matrix(n_rows, n_cols, seed):
    """Rows of 0 to 60 nonzeros, one of 900 (segments), and the rows to spoil."""
    g = torch.Generator().manual_seed(seed)
    lengths = torch.randint(0, 61, (n_rows,), generator=g)
    lengths[n_rows // 3] = 900
    ptr = torch.zeros(n_rows + 1, dtype=torch.int64)
    ptr[1:] = lengths.cumsum(0)
    idx = torch.randint(0, n_cols, (int(ptr[-1]),), generator=g)
    row = torch.repeat_interleave(torch.arange(n_rows), lengths)
    spoiled = torch.rand(n_rows, generator=g) < 0.3
    return ptr, idx, row, spoiled, torch.randn(idx.numel(), generator=g)


def _spoil(val, where, seed):
    bad = torch.tensor(BAD, dtype=val.dtype)[torch.randint(0, 3, val.shape, generator=torch.Generator().manual_seed(seed))]
    return torch.where(where, bad, val)


@pytest.mark.parametrize("grid", [{}, {"max_blocks": 4}, {"max_blocks": 24, "xcd_groups": 8}], ids=["all", "cap", "xcd"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n", [1, 16, 31, 64, 200])
@pytest.mark.parametrize("unroll", [4, 8])
def test_rows_keep_their_values(device, grid, dtype, n, unroll):
    m, k = 3000, 500
    ptr, idx, row, spoiled, val = _matrix(m, k, n)
    val = val.to(dtype)
    h = fs.CsrMatrix(idx.int().to(device), ptr.int().to(device), (m, k)).handle
    B = torch.randn(k, n, device=device).to(dtype)
    cfg = _plan.spmm_config(_plan.lanes_for_dense(n, val.element_size()), unroll=unroll)
    clean = h.spmm(val.to(device), B, config=cfg, **grid)
    mixed = h.spmm(_spoil(val, spoiled[row], n).to(device), B, config=cfg, **grid)
    keep = ~spoiled.to(device)
    assert torch.isfinite(clean).all() and torch.equal(mixed[keep], clean[keep])
    has = torch.zeros(m, dtype=torch.bool)
    has[row] = True
    assert not torch.isfinite(mixed[(spoiled & has).to(device)]).any()


@pytest.mark.parametrize("grid", [{}, {"max_blocks": 4}], ids=["all", "cap"])
@pytest.mark.parametrize("in_kernel", [False, True], ids=["gathered", "permuted"])
def test_columns_of_the_transposed_product(device, grid, in_kernel):
    m, k, n = 3000, 500, 64
    ptr, idx, row, _, val = _matrix(m, k, 5)
    h = fs.CsrMatrix(idx.int().to(device), ptr.int().to(device), (m, k)).handle
    spoiled = torch.rand(k, generator=torch.Generator().manual_seed(6)) < 0.3
    dC = torch.randn(m, n, device=device)
    clean = h.spmm(val.to(device), dC, transpose=True, values_via_perm=in_kernel, **grid)
    bad = _spoil(val, spoiled[idx], 7).to(device)
    mixed = h.spmm(bad, dC, transpose=True, values_via_perm=in_kernel, **grid)
    keep = ~spoiled.to(device)
    assert torch.equal(mixed[keep], clean[keep])
    dB, dv = h.spmm_trans_sddmm(bad, dC, torch.randn(k, n, device=device))
    assert torch.equal(dB[keep], clean[keep]) and torch.isfinite(dv).all()


def test_wide_values(device):
    m, k, n = 3000, 500, 64
    ptr, idx, row, spoiled, val = _matrix(m, k, 8)
    h = fs.CsrMatrix(idx.int().to(device), ptr.int().to(device), (m, k)).handle
    B = torch.randn(k, n, device=device)
    val = val.double()
    clean = h.spmm(val.to(device), B, max_blocks=4)
    mixed = h.spmm(_spoil(val, spoiled[row], 9).to(device), B, max_blocks=4)
    keep = ~spoiled.to(device)
    assert torch.equal(mixed[keep], clean[keep])


def test_systems_of_a_batch(device):
    """One system of a batch that has diverged leaves the others alone."""
    mats, bad = [], []
    for s in range(24):
        ptr, idx, _, _, val = _matrix(200, 200, 100 + s)
        mats.append([t.to(device) for t in (val, idx.int(), ptr.int())] + [(200, 200)])
        bad.append(torch.full_like(mats[-1][0], float("nan")) if s % 3 == 1 else mats[-1][0])
    batch = CsrBatch.from_matrices([tuple(m) for m in mats])
    B = torch.randn(24 * 200, 32, device=device)
    for xg in (0, 8):
        p = TuneParams(blocks_per_cu=8, xcd_groups=xg)
        # fewer workgroups than tiles, as a tuned launch of a large batch has
        capped = dict(config=p.spmm_config(8), lanes_n=8, max_blocks=40, xcd_groups=xg)
        for run in (lambda d: batch.spmm(B, data=d, params=p), lambda d: batch.handle.spmm(d, B, **capped)):
            clean, mixed = batch.split(run(batch.data)), batch.split(run(torch.cat(bad)))
            for s in range(24):
                if s % 3 != 1:
                    assert torch.equal(mixed[s], clean[s])
