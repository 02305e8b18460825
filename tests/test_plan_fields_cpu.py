"""A plan whose fields change after a launch, and what dataclasses does with it."""

import dataclasses

import pytest
import torch

from flagsparse_amd import _plan


def _plan_of(rows):
    none = torch.empty(0, dtype=torch.int64)
    return _plan.CsrPlan(
        config=_plan.spmv_config(), n_rows=3, rows=torch.tensor(rows, dtype=torch.int32), bin_counts=[2, 1, 0, 0, 0],
        identity=False, seg_row=none.int(), seg_begin=none, seg_end=none, long_rows=none.int(), long_seg_ptr=none,
        n_segments=0, n_long_rows=0)


@pytest.mark.parametrize("field,value,read", [
    ("rows", torch.tensor([1, 0, 2], dtype=torch.int32), lambda st, p: (st.bins[0].rows, p.rows.data_ptr())),
    ("bin_counts", [1, 2, 0, 0, 0], lambda st, p: (st.bins[0].count, 1)),
    ("identity", True, lambda st, p: (st.bins[0].rows, None)),
    ("config", _plan.spmv_config(unroll=8), lambda st, p: (st.unroll, 8)),
    ("row_len", 7, lambda st, p: (st.row_len, 7)),
])
def test_changed_field_reaches_the_next_launch(field, value, read):
    plan = _plan_of([2, 0, 1])
    plan.struct()
    setattr(plan, field, value)
    got, want = read(plan.struct(), plan)
    assert got == want


def test_dataclass_functions_after_a_launch():
    plan = _plan_of([2, 0, 1])
    plan.struct()
    state = dataclasses.asdict(plan)
    assert set(state) == {f.name for f in dataclasses.fields(plan)} and torch.equal(state["rows"], plan.rows)
    other = dataclasses.replace(plan, rows=plan.rows.clone())
    assert other.struct().bins[0].rows == other.rows.data_ptr() != plan.rows.data_ptr()
