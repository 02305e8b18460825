"""Plans of matrices whose nonzeros sit in a few rows: thousands of segments of
one row, on both sides of the one-workgroup limit (8192 rows, 131072
nonzeros), mixed with rows of few segments, and with room for too few."""

import numpy as np
import pytest
import torch

from flagsparse_amd import _plan

pytestmark = pytest.mark.gpu


def _pointer(n_rows, long_rows, device, pt=torch.int32):
    lengths = np.random.default_rng(n_rows).integers(0, 30, n_rows)
    for r, n in long_rows.items():
        lengths[r] = n
    indptr = np.concatenate([[0], np.cumsum(lengths)])
    return lengths, indptr, torch.tensor(indptr, dtype=pt, device=device)


@pytest.mark.parametrize("pt", [torch.int32, torch.int64], ids=["p32", "p64"])
@pytest.mark.parametrize("n_rows,long_rows", [
    (1, {0: 3_000_001}), (1, {0: 1 << 20}), (300, {7: 120_000}), (300, {7: 4_000_000, 8: 65, 299: 192, 0: 193}),
    (500, {i: 193 + i for i in range(500)}), (8193, {0: 100_000, 8192: 64 * 48 + 1}),
    (300, {0: 60_000, 5: 1024 * 48 + 1, 9: 1024 * 48, 11: 16 * 48 + 1, 12: 16 * 48, 13: 17 * 48}),
    (9000, {0: 60_000, 5: 1024 * 48 + 1, 9: 1024 * 48, 11: 16 * 48 + 1, 12: 16 * 48, 13: 17 * 48}),
    (9000, {i: 2000 + i for i in range(0, 9000, 3)}),
    (70_000, {**{i: 200 + i % 900 for i in range(0, 70_000, 31)}, 69_999: 5_000_000}),
], ids=["one", "one_wave", "small", "mixed", "all", "rows", "steps_small", "steps", "mid", "many"])
def test_segments_of_long_rows(device, pt, n_rows, long_rows):
    lengths, indptr, p = _pointer(n_rows, long_rows, device, pt)
    cfg = _plan.spmm_config(16, long_threshold=64, seg_len=48)
    rows = np.flatnonzero(lengths > 64)
    n = -(-lengths[rows] // 48)
    ptr = np.concatenate([[0], np.cumsum(n)])
    owner = np.repeat(np.arange(rows.size), n)
    j = np.arange(int(ptr[-1])) - ptr[owner]
    begin, length = indptr[rows][owner], lengths[rows][owner]
    idx = torch.zeros(int(indptr[-1]), dtype=torch.int32, device=device)
    for plan in (_plan.build_plan(p, n_rows, cfg), _plan.build_plan(p, n_rows, cfg, idx.numel() + 12345),
                 _plan.inspect_csr(p, idx, n_rows, idx.numel(), cfg)[1]):
        assert plan.n_segments == ptr[-1] and np.array_equal(plan.long_rows.cpu().numpy(), rows)
        assert np.array_equal(plan.long_seg_ptr.cpu().numpy(), ptr)
        assert np.array_equal(plan.seg_row.cpu().numpy(), rows[owner])
        assert np.array_equal(plan.seg_begin.cpu().numpy(), begin + length * j // n[owner])
        assert np.array_equal(plan.seg_end.cpu().numpy(), begin + length * (j + 1) // n[owner])


@pytest.mark.parametrize("n_rows", [300, 9000])
def test_too_small_a_bound(device, n_rows):
    _, indptr, p = _pointer(n_rows, {5: 50_000, 6: 400}, device)
    cfg = _plan.spmm_config(16, long_threshold=64, seg_len=48)
    for nnz in (100, 5000):  # neither leaves room for the 1042 segments
        with pytest.raises(RuntimeError, match="more nonzeros"):
            _plan.build_plan(p, n_rows, cfg, nnz)


def test_time_does_not_depend_on_the_longest_row(device):
    """8 M nonzeros in one row against 8192 rows of 1024: the same number of segments."""
    cfg = _plan.spmm_config(16)
    one = torch.full((8193,), 1 << 23, dtype=torch.int32, device=device)
    one[0] = 0
    even = torch.arange(0, (1 << 23) + 1, 1024, dtype=torch.int32, device=device)

    def best(p):
        times = []
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            plan = _plan.build_plan(p, 8192, cfg, 1 << 23)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        assert plan.n_segments == 1 << 15
        return min(times)

    t_one, t_even = best(one), best(even)
    print(f"one row {t_one:.3f} ms, even rows {t_even:.3f} ms", flush=True)
    assert t_one < 5 * t_even  # 20 ms against 0.3 when one thread wrote a row's segments
