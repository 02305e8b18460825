"""Copies and pickles of a plan that has already been launched with."""
import copy
import io
import pickle

import pytest
import torch

from flagsparse_amd import _plan


def _pickled(plan):
    return pickle.loads(pickle.dumps(plan))


def _saved(plan):
    f = io.BytesIO()
    torch.save(plan, f)
    f.seek(0)
    return torch.load(f, weights_only=False)


def _older(plan):  # a state without the cached structs
    state = {k: v for k, v in vars(plan).items() if k != "_structs"}
    new = object.__new__(_plan.CsrPlan)
    new.__setstate__(state)
    return new


@pytest.mark.parametrize("how", [copy.copy, copy.deepcopy, _pickled, _saved, _older])
def test_copy_has_its_own_struct(how):
    none = torch.empty(0, dtype=torch.int64)
    plan = _plan.CsrPlan(
        config=_plan.spmv_config(), n_rows=3, rows=torch.tensor([2, 0, 1], dtype=torch.int32),
        bin_counts=[2, 1, 0, 0, 0], identity=False, seg_row=none.int(), seg_begin=none, seg_end=none,
        long_rows=none.int(), long_seg_ptr=none, n_segments=0, n_long_rows=0)
    plan.struct(max_blocks=4)
    other = how(plan)
    other.rows = other.rows.clone()
    st = other.struct(max_blocks=4)
    assert st.bins[0].rows == other.rows.data_ptr() and st.bins[1].rows == other.rows.data_ptr() + 8
    assert other.bin_sizes == plan.bin_sizes and other.config == plan.config
    assert plan.struct(max_blocks=4).bins[0].rows == plan.rows.data_ptr()
