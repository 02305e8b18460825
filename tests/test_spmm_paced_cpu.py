"""The rule that says which SpMM loop a launch takes, at its edges (no launch)."""

import pytest

from flagsparse_amd import _lib

MIB = 1 << 20
F32, F64, BF16 = _lib.FSP_F32, _lib.FSP_F64, _lib.FSP_BF16


@pytest.mark.parametrize("value,lanes,n,ld,rows,backward,shares", [
    (F32, 2, 8, 8, 1000, 0, 0),  # two lanes
    (F32, 4, 16, 16, 1000, 0, 1),
    (F32, 8, 32, 32, 400 * MIB // 128, 0, 1),  # eight lanes are never paced
    (F32, 16, 64, 64, 56 * MIB // 256 - 1, 0, 1), (F32, 16, 64, 64, 56 * MIB // 256, 0, 0),
    (F32, 16, 64, 128, 28 * MIB // 256, 0, 0),  # the gaps between rows count
    (F32, 16, 64, 64, 400 * MIB // 256, 1, 1),  # the backward
    (F32, 32, 100, 100, 52 * MIB // 400, 0, 1), (F32, 32, 112, 112, 52 * MIB // 448, 0, 0),  # 25 and 28 of 32 lanes
    (F64, 32, 64, 64, 32 * MIB // 512 - 1, 0, 1), (F64, 32, 64, 64, 32 * MIB // 512, 0, 0),
    (F64, 64, 128, 128, 56 * MIB // 1024 - 1, 0, 1), (F64, 64, 128, 128, 56 * MIB // 1024, 0, 0),
    (F64, 64, 75, 75, 400 * MIB // 600, 0, 1),  # 38 of 64 lanes
    (F64, 64, 300, 300, 57 * MIB // 2400, 0, 0),  # more than one column tile
    (BF16, 16, 128, 128, 56 * MIB // 256, 0, 0),
    (F32, 8, 32, 32, (1 << 32) // 128 - 2, 0, 1), (F32, 8, 32, 32, (1 << 32) // 128 - 1, 0, 0),  # 32-bit offsets
    (F32, 16, 3, 3, 10, 0, 0), (F32, 16, 64, 63, 10, 0, 0), (F32, 12, 64, 64, 10, 0, 0), (F32, 128, 64, 64, 10, 0, 0),
    (F32, 16, 64, 64, -1, 0, 0),
])
def test_rule(value, lanes, n, ld, rows, backward, shares):
    assert _lib.load().fsp_spmm_shares_nonzeros(value, lanes, n, ld, rows, backward) == shares
