"""The BSR SpMM's wave-per-block-row kernel where its loops turn: block rows of
0, 1, 63, 64, 65 and 130 blocks (64 block columns are held per chunk), dense
widths on either side of 2, 4 and 8 tiles of 16 columns, one and two block rows
per wave with an odd number of block rows."""

import numpy as np
import pytest
import torch

import flagsparse_amd as fs

pytestmark = pytest.mark.gpu


def _matrix(counts, nbc, seed, device):
    rng = np.random.default_rng(seed)
    ptr = np.concatenate([[0], np.cumsum(counts)])
    col = np.concatenate([np.sort(rng.choice(nbc, c, replace=False)) for c in counts] + [np.zeros(0, np.int64)])
    data = rng.standard_normal((int(ptr[-1]), 16, 16))
    return (torch.tensor(data, dtype=torch.float32, device=device),
            torch.tensor(col.astype(np.int64), dtype=torch.int32, device=device),
            torch.tensor(ptr, dtype=torch.int32, device=device))


def _reference(data, col, ptr, B, rows, nbc):
    """float64 product and the same of the absolute values, from the operands the kernel multiplies."""
    n = B.shape[1]
    Bp = torch.zeros(nbc * 16, n, dtype=torch.float64, device=B.device)
    Bp[: B.shape[0]] = B
    out = []
    owner = torch.repeat_interleave((ptr[1:] - ptr[:-1]).long())
    for a, b in ((data, Bp), (data.abs(), Bp.abs())):
        C = torch.zeros(ptr.numel() - 1, 16, n, dtype=torch.float64, device=B.device)
        C.index_add_(0, owner, torch.bmm(a, b.view(nbc, 16, n)[col.long()]))
        out.append(C.view(-1, n)[:rows])
    return out


@pytest.mark.parametrize("n", [1, 16, 17, 33, 48, 64, 65, 128, 130, 257])
@pytest.mark.parametrize("kind", ["bf16", "f16", "fp8"])
@pytest.mark.parametrize("many", [False, True], ids=["one_row", "two_rows"])
def test_sweep_edges(device, n, kind, many):
    nbc = 200
    counts = [0, 1, 63, 64, 65, 130, 2, 199, 0]
    if many:  # at least 4096 block rows: two per wave, the last one alone
        counts = counts + [int(c) for c in np.random.default_rng(n).integers(0, 4, 4096)]
    rows, K = len(counts) * 16 - 5, nbc * 16 - 3
    data, col, ptr = _matrix(counts, nbc, n, device)
    B = torch.tensor(np.random.default_rng(7).standard_normal((K, n)), dtype=torch.float32, device=device)
    # 16 * 199 f32 terms, each sum rounded once per block pair at most: n_terms * 2^-24
    terms = 16 * max(counts) * 2.0**-24
    if kind == "fp8":
        codes, scales = fs.quantize_bsr_fp8(data)
        C = fs.flagsparse_spmm_bsr(codes, col, ptr, B, (rows, K), scales=scales)
        a = codes.view(torch.float8_e4m3fn).double() * scales.double()[:, None, None]
        am = B.abs().max()
        b = ((B * (448.0 / am)).to(torch.float8_e4m3fn).double() * (am.double() / 448.0))
        slack = 4 * terms + 2.0**-20  # the scales are float32 products
    else:
        dt = torch.bfloat16 if kind == "bf16" else torch.float16
        C = fs.flagsparse_spmm_bsr(data.to(dt), col, ptr, B, (rows, K))
        a, b = data.to(dt).double(), B.to(dt).double()
        slack = 4 * terms
    ref, mag = _reference(a, col, ptr, b, rows, nbc)
    assert torch.all((C.double() - ref).abs() <= slack * mag + 1e-30)
