"""The C entries fsp_csr_inspect and fsp_csr_row_bins called directly (the
package builds its plans with fsp_csr_build_plan): figures and stable bins
against numpy, and the same rows and figures as fsp_csr_build_plan's."""

import ctypes

import numpy as np
import pytest
import torch

from flagsparse_amd import _lib, _plan

pytestmark = pytest.mark.gpu


def _row_bins(p, n_rows, uppers):
    lib, nb = _lib.load(), len(uppers) + 1
    ws_bytes = ctypes.c_int64(0)
    _lib.check(lib.fsp_csr_row_bins_workspace(n_rows, nb, ctypes.byref(ws_bytes)), "workspace")
    rows = torch.full((n_rows + 1,), -7, dtype=torch.int32, device=p.device)
    offsets = torch.full((nb + 2,), -7, dtype=torch.int64, device=p.device)
    ws = torch.empty(ws_bytes.value, dtype=torch.uint8, device=p.device)
    _lib.check(lib.fsp_csr_row_bins(_lib.index_code(p.dtype), p.data_ptr(), n_rows, nb,
                                    (ctypes.c_int64 * nb)(*uppers, 0), rows.data_ptr(), offsets.data_ptr(),
                                    ws.data_ptr(), ws_bytes.value, _lib.stream_ptr(p.device)), "fsp_csr_row_bins")
    assert int(rows[-1]) == -7 and int(offsets[-1]) == -7
    return rows[:-1].cpu().numpy(), offsets[:-1].cpu().numpy()


def _inspect(p, i, n_rows):
    stats = torch.empty(6, dtype=torch.int64, device=p.device)
    _lib.check(_lib.load().fsp_csr_inspect(_lib.index_code(p.dtype), p.data_ptr(), _lib.index_code(i.dtype),
                                           _lib.ptr(i), n_rows, i.numel(), stats.data_ptr(),
                                           _lib.stream_ptr(p.device)), "fsp_csr_inspect")
    return stats.tolist()


@pytest.mark.parametrize("pt", [torch.int32, torch.int64], ids=["p32", "p64"])
@pytest.mark.parametrize("it", [torch.int32, torch.int64], ids=["i32", "i64"])
@pytest.mark.parametrize("n_rows", [0, 1, 63, 1024, 1025, 30000])
def test_entries(device, pt, it, n_rows):
    rng = np.random.default_rng(n_rows)
    lengths = rng.integers(0, 40, n_rows)
    if n_rows > 60:
        lengths[rng.choice(n_rows, 9, replace=False)] = rng.integers(65, 5000, 9)
    indptr = np.concatenate([[0], np.cumsum(lengths)])
    cols = rng.integers(0, 1000, int(indptr[-1]))
    p = torch.tensor(indptr, dtype=pt, device=device)
    i = torch.tensor(cols, dtype=it, device=device)
    uppers = (0, 8, 16, 64)
    bins = np.searchsorted(uppers, lengths, side="left")
    rows, offsets = _row_bins(p, n_rows, uppers)
    assert np.array_equal(rows, np.argsort(bins, kind="stable"))
    assert np.array_equal(offsets, np.concatenate([[0], np.cumsum(np.bincount(bins, minlength=5))]))
    plan = _plan.build_plan(p, n_rows, _plan.PlanConfig((1, 2, 4, 8), uppers, 64, 4))
    if not plan.identity:
        assert np.array_equal(plan.rows.cpu().numpy(), rows)
    want = [0, int(indptr[-1]), 0, int(cols.min()) if cols.size else 2**63 - 1,
            int(cols.max()) if cols.size else -2**63, int(lengths.max()) if n_rows else 0]
    assert _inspect(p, i, n_rows) == want


def test_figures_of_a_broken_pointer(device):
    p = torch.tensor([3, 9, 4, 4, 2, 8], dtype=torch.int32, device=device)
    i = torch.tensor([5, -4, 7], dtype=torch.int32, device=device)
    assert _inspect(p, i, 5) == [3, 8, 2, -4, 7, 6]
    stats, plan = _plan.inspect_csr(p, i, 5, 3, _plan.spmm_config(16))
    assert plan is None and list(stats.values()) == [3, 8, 2, -4, 7, 6]
