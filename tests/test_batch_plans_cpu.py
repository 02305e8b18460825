"""The per-matrix plans of a batch are sized for the matrix, not for the batch."""

import numpy as np
import torch

from flagsparse_amd import _plan
from flagsparse_amd._matrix import CsrHandle
from flagsparse_amd.batch import CsrBatch


def test_plan_bounds(monkeypatch):
    b = object.__new__(CsrBatch)
    b.n_mats, b._per_matrix, b.total_cols = 2, None, 7
    b.row_offsets, b.col_offsets, b.nnz_offsets = np.array([0, 2, 5]), np.array([0, 3, 7]), np.array([0, 3, 11])
    b.indices = b.local_indices = torch.zeros(11, dtype=torch.int32)
    b.indptr = torch.tensor([0, 1, 3, 5, 8, 11], dtype=torch.int32)
    b.local_indptr = torch.tensor([0, 1, 3, 0, 2, 5, 8], dtype=torch.int32)
    seen = []
    monkeypatch.setattr(_plan, "build_plan", lambda indptr, n_rows, config, nnz=None: seen.append((n_rows, nnz)))
    for h, hg, *_ in b._matrices():
        h.plan(_plan.spmv_config())
        hg.plan(_plan.spmv_config())
    assert seen == [(2, 3), (2, 3), (3, 8), (3, 8)]


def test_handle_saved_without_the_bound(monkeypatch):
    state = {"indices": torch.zeros(4, dtype=torch.int32), "indptr": torch.tensor([0, 1, 4], dtype=torch.int32),
             "shape": (2, 3), "n_rows": 2, "n_cols": 3, "nnz": 4, "_plans": {}, "_csc": None, "_csc_plans": {}}
    h = object.__new__(CsrHandle)
    for name, value in state.items():  # what unpickling an older handle sets
        setattr(h, name, value)
    seen = []
    monkeypatch.setattr(_plan, "build_plan", lambda indptr, n_rows, config, nnz=None: seen.append((n_rows, nnz)))
    h.plan(_plan.spmv_config())
    assert seen == [(2, 4)]
