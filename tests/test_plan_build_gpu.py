"""fsp_csr_build_plan against numpy: figures, stable row bins and long-row
segments, on both sides of the one-workgroup limit (8192 rows, 131072
nonzeros), with more long rows than a workgroup's scan takes at once, and the
same plan whatever bound on the nonzeros the buffers were sized for."""

import numpy as np
import pytest
import torch

from flagsparse_amd import _plan

pytestmark = pytest.mark.gpu


def _expect(lengths, indptr, cfg):
    bins = np.searchsorted(np.asarray(cfg.uppers), lengths, side="left")  # smallest b with length <= uppers[b]
    nb = len(cfg.uppers) + 1
    order = [np.flatnonzero(bins == b) for b in range(nb)]
    seg_row, seg_begin, seg_end, ptr = [], [], [], [0]
    for r in order[-1]:
        n = -(-int(lengths[r]) // cfg.seg_len)
        for j in range(n):
            seg_row.append(r)
            seg_begin.append(indptr[r] + int(lengths[r]) * j // n)
            seg_end.append(indptr[r] + int(lengths[r]) * (j + 1) // n)
        ptr.append(ptr[-1] + n)
    return order, seg_row, seg_begin, seg_end, ptr


@pytest.mark.parametrize("pt", [torch.int32, torch.int64], ids=["p32", "p64"])
@pytest.mark.parametrize("n_rows,mean,n_long", [(1, 3, 1), (63, 5, 0), (1024, 4, 3), (1025, 4, 1025), (8192, 15, 40),
                                                (8193, 2, 1), (8192, 17, 0), (40000, 6, 2100)])
def test_plan_matches_numpy(device, pt, n_rows, mean, n_long):
    rng = np.random.default_rng(n_rows + mean)
    lengths = rng.integers(0, 2 * mean + 1, n_rows)
    cfg = _plan.spmm_config(16, long_threshold=64, seg_len=48)
    lengths[rng.choice(n_rows, n_long, replace=False)] = rng.integers(65, 400, n_long)
    indptr = np.concatenate([[0], np.cumsum(lengths)])
    nnz = int(indptr[-1])
    cols = rng.integers(0, 1000, nnz)
    p = torch.tensor(indptr, dtype=pt, device=device)
    i = torch.tensor(cols, dtype=torch.int32, device=device)
    order, seg_row, seg_begin, seg_end, ptr = _expect(lengths, indptr, cfg)
    stats, plan = _plan.inspect_csr(p, i, n_rows, nnz, cfg)
    assert stats == {"indptr_first": 0, "indptr_last": nnz, "n_decreasing": 0, "min_col": int(cols.min()),
                     "max_col": int(cols.max()), "max_row": int(lengths.max())}
    plans = [plan, _plan.build_plan(p, n_rows, cfg), _plan.build_plan(p, n_rows, cfg, nnz + (1 << 22))]
    for q in plans:
        assert q.n_long_rows == n_long and q.n_segments == len(seg_row)
        if not q.identity:
            assert q.bin_counts == [len(o) for o in order[:-1]]
        assert np.array_equal(q.rows.cpu().numpy(), np.concatenate(order))
        if n_long:
            assert np.array_equal(q.long_rows.cpu().numpy(), order[-1])
            assert np.array_equal(q.seg_row.cpu().numpy(), seg_row)
            assert np.array_equal(q.seg_begin.cpu().numpy(), seg_begin)
            assert np.array_equal(q.seg_end.cpu().numpy(), seg_end)
            assert np.array_equal(q.long_seg_ptr.cpu().numpy(), ptr)


def test_plan_of_too_small_a_bound_is_refused(device):
    p = torch.tensor([0, 300, 600], dtype=torch.int32, device=device)
    with pytest.raises(RuntimeError, match="more nonzeros"):
        _plan.build_plan(p, 2, _plan.spmm_config(16), 300)
