"""BSR SpMM with a packed B on either side of 4 GiB: below it every launch takes
bsr_spmm_sweep_kernel, beyond it bsr_spmm_kernel with 64-bit addresses.  The
blocks' columns lie at both ends of B.  Both are compared with the product over
the referenced rows of B alone, which has the same blocks in the same order and
takes the sweep kernel: bit for bit, and bf16 / f16 with float64."""

import pytest
import torch

import flagsparse_amd as fs

pytestmark = pytest.mark.gpu

N, BLOCK_ROWS, PER_ROW = 128, 37, 7
BEYOND, BELOW = (1 << 24) + 1024, (1 << 24) - 32  # rows of a 16-bit B; 256 packed bytes each


@pytest.mark.parametrize("kind,K", [("bf16", BEYOND), ("f16", BEYOND), ("fp8", 2 * BEYOND), ("bf16", BELOW),
                                    ("fp8", 2 * BELOW)])
def test_packed_b_around_4gib(device, kind, K):
    packed = K * N * (1 if kind == "fp8" else 2)
    assert (packed > 1 << 32) == (K in (BEYOND, 2 * BEYOND)) and abs(packed - (1 << 32)) < 1 << 20
    nbc = K // 16
    g = torch.Generator(device=device).manual_seed(K % 1000)
    cols = []
    for _ in range(BLOCK_ROWS):  # four blocks anywhere, three in the last 64 block columns, one of them the last
        lo = torch.randperm(nbc - 64, generator=g, device=device)[:4]
        hi = nbc - 64 + torch.randperm(63, generator=g, device=device)[:2]
        cols.append(torch.cat([lo, hi, torch.tensor([nbc - 1], device=device)]).sort().values)
    col = torch.cat(cols)
    ptr = torch.arange(0, BLOCK_ROWS * PER_ROW + 1, PER_ROW, dtype=torch.int32, device=device)
    blocks = torch.randn(col.numel(), 16, 16, generator=g, device=device)
    dt = torch.float16 if kind == "f16" else torch.bfloat16
    B = torch.randn(K, N, generator=g, device=device, dtype=dt)
    uniq, small = torch.unique(col, return_inverse=True)
    scales = None
    if kind == "fp8":
        B[uniq[0] * 16, 0] = 64.0  # the largest element of both operands, so both have one scale
        blocks, scales = fs.quantize_bsr_fp8(blocks)
    else:
        blocks = blocks.to(dt)
    C = fs.flagsparse_spmm_bsr(blocks, col.int(), ptr, B, (BLOCK_ROWS * 16, K), scales=scales)
    rows = (uniq[:, None] * 16 + torch.arange(16, device=device)).view(-1)
    B_small = B[rows]
    del B
    torch.cuda.empty_cache()
    C_small = fs.flagsparse_spmm_bsr(blocks, small.int(), ptr, B_small, (BLOCK_ROWS * 16, rows.numel()), scales=scales)
    assert torch.equal(C, C_small)
    if kind == "fp8":  # the fp8 MFMA sums below float32 precision; held to the oracle at smaller sizes
        return
    a, b, slack = blocks.double(), B_small.double(), 4 * 16 * PER_ROW * 2.0**-24
    owner = torch.repeat_interleave(torch.arange(BLOCK_ROWS, device=device), PER_ROW)
    ref, mag = (torch.zeros(BLOCK_ROWS, 16, N, dtype=torch.float64, device=device).index_add_(
        0, owner, torch.bmm(x, y.view(-1, 16, N)[small])).view(-1, N) for x, y in ((a, b), (a.abs(), b.abs())))
    assert torch.all((C.double() - ref).abs() <= slack * mag + 1e-30)
