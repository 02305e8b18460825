"""Strides in the meta of flagsparse_spmm_coo: those of B in the compute dtype."""

import pytest
import torch

from flagsparse_amd import spmm_coo


class _Canonical:
    def __init__(self, *args):
        pass

    def spmm(self, B, dense_layout, out=None):
        return torch.zeros(2, B.shape[1], dtype=B.dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16])
@pytest.mark.parametrize("layout", ["row", "col"])
@pytest.mark.parametrize("make", [lambda d: torch.zeros(3, 5, dtype=d), lambda d: torch.zeros(5, 3, dtype=d).t(),
                                  lambda d: torch.zeros(5, 8, dtype=d).t()[:3], lambda d: torch.zeros(3, 9, dtype=d)[:, :5],
                                  lambda d: torch.zeros(1, 3, dtype=d).t()], ids=["row", "col", "col_padded",
                                                                                  "row_padded", "one"])
def test_b_stride(monkeypatch, dtype, layout, make):
    B = make(dtype)

    def inputs(data, row, col, B, shape, dense_layout):
        return data, row, col, spmm_coo._materialize_dense_layout(B, dense_layout), 2, 3, int(B.shape[1])

    monkeypatch.setattr(spmm_coo, "_prepare_spmm_coo_inputs", inputs)
    monkeypatch.setattr(spmm_coo, "_CanonicalCoo", _Canonical)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    i = torch.zeros(1, dtype=torch.int64)
    _, meta = spmm_coo.flagsparse_spmm_coo(torch.ones(1, dtype=dtype), i, i, B, (2, 3), return_meta=True,
                                           dense_layout=layout)
    held = spmm_coo._materialize_dense_layout(B, layout)
    compute = {torch.float32: torch.float64, torch.bfloat16: torch.float32}.get(dtype, dtype)
    assert meta["b_stride"] == tuple(held.to(compute).stride())
