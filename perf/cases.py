"""Performance cases of the public entry points.

A case is a dict of plain values.  ``listed()`` names twelve of them and says
what each stands for, ``draw`` gives further ones of the same ranges,
``prepare`` builds what a program holds before a call (inputs on the GPU and
the prepared object it keeps), ``run`` is one pass through the public API,
``work`` the bytes and operations of a pass and ``exact`` its result in
64 bits from plain torch.

Keys: ``kind`` is the entry point family, ``pattern`` the sparsity
("uniform": every row ``mean`` nonzeros; "power_law": row lengths of exponent
2.1 capped at 4096, uniform columns; "graph": a symmetric Chung-Lu graph of
exponent 2.3, so hub rows and hub columns), ``n`` the dense width.
"""

import math

import torch

import flagsparse_amd as fs
from flagsparse_amd.batch import CsrBatch
from flagsparse_amd.synthetic import power_law_scale

DEVICE = "cuda"
DTYPES = {"f32": torch.float32, "f64": torch.float64, "bf16": torch.bfloat16, "f16": torch.float16}
INDEX = {"i32": torch.int32, "i64": torch.int64}
BYTES = {"f32": 4, "f64": 8, "bf16": 2, "f16": 2, "fp8": 1, "i32": 4, "i64": 8}
CHUNK = 1 << 24  # nonzeros per step of exact()


def listed():
    return [
        # the smallest call: one prepared SpMV of an iterative solver on a cache-resident matrix, launch-bound
        {"name": "spmv_small", "kind": "spmv", "pattern": "uniform", "rows": 16384, "cols": 16384, "mean": 16,
         "dtype": "f32", "index": "i32", "op": "non"},
        # prepared SpMV of a web / recommendation matrix: skewed rows, x beyond LDS
        {"name": "spmv_power_law", "kind": "spmv", "pattern": "power_law", "rows": 262144, "cols": 262144,
         "mean": 24, "dtype": "f32", "index": "i32", "op": "non"},
        # the largest: a tall matrix streamed from HBM once per pass
        {"name": "spmv_tall", "kind": "spmv", "pattern": "uniform", "rows": 1 << 24, "cols": 16384, "mean": 16,
         "dtype": "f32", "index": "i32", "op": "non"},
        # one unprepared SpMM call: validation, plan and product each time the matrix changes
        {"name": "spmm_call", "kind": "spmm_call", "pattern": "power_law", "rows": 4096, "cols": 4096, "mean": 16,
         "dtype": "f32", "index": "i32", "op": "non", "n": 32},
        # the SpMM the framework is benchmarked on: prepared, f32, N = 64
        {"name": "spmm_power_law", "kind": "spmm", "pattern": "power_law", "rows": 262144, "cols": 262144,
         "mean": 24, "dtype": "f32", "index": "i32", "op": "non", "n": 64},
        # ragged sizes in double precision: a block of 75 right-hand sides, 64-bit indices
        {"name": "spmm_ragged", "kind": "spmm", "pattern": "power_law", "rows": 100003, "cols": 70001, "mean": 24,
         "dtype": "f64", "index": "i64", "op": "non", "n": 75},
        # graph convolution in bf16 against the transposed adjacency, through the route API
        {"name": "spmm_trans", "kind": "spmm", "pattern": "graph", "rows": 200000, "cols": 200000, "mean": 14,
         "dtype": "bf16", "index": "i32", "op": "trans", "n": 128},
        # edge scores of an attention layer on the same graph
        {"name": "sddmm_graph", "kind": "sddmm", "pattern": "graph", "rows": 200000, "cols": 200000, "mean": 14,
         "dtype": "f32", "index": "i32", "n": 128},
        # a training step of a graph layer: forward, gradients of values and features
        {"name": "train_graph", "kind": "train", "pattern": "graph", "rows": 200000, "cols": 200000, "mean": 14,
         "dtype": "bf16", "index": "i32", "n": 128},
        # block-sparse weights on the matrix cores
        {"name": "bsr_spmm", "kind": "bsr", "rows": 65536, "cols": 65536, "mean": 40, "dtype": "bf16", "n": 128},
        # many small systems in one launch
        {"name": "batch_spmm", "kind": "batch", "op": "spmm", "mats": 1024, "rows": 8192, "mean": 34, "n": 32,
         "dtype": "f32"},
        # COO input prepared once, as a data pipeline hands it over (float32 is computed in float64)
        {"name": "coo_spmm", "kind": "coo", "pattern": "power_law", "rows": 150001, "cols": 90001, "mean": 20,
         "dtype": "f32", "index": "i64", "op": "non", "n": 100},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges."""
    kind = rng.choice(["spmv", "spmv", "spmv", "spmm_call", "spmm", "spmm", "spmm", "sddmm", "train", "bsr", "batch",
                       "coo"])
    if kind == "bsr":
        rows = _log_int(rng, 1000, 65536)
        cols = _log_int(rng, 2000, 65536)
        return {"kind": kind, "rows": rows, "cols": cols, "mean": min(_log_int(rng, 4, 48), -(-cols // 16)),
                "dtype": rng.choice(["bf16", "f16", "fp8"]), "n": _log_int(rng, 16, 256)}
    if kind == "batch":
        op = rng.choice(["spmv", "spmm"])
        return {"kind": kind, "op": op, "mats": _log_int(rng, 32, 1024), "rows": _log_int(rng, 500, 8192),
                "mean": rng.randint(6, 34), "n": 1 if op == "spmv" else _log_int(rng, 4, 64),
                "dtype": rng.choice(["f32", "f32", "f64"])}
    if kind == "spmv" and rng.random() < 0.25:  # tall matrices
        pattern, rows, cols = rng.choice(["uniform", "power_law"]), _log_int(rng, 1 << 20, 1 << 23), \
            _log_int(rng, 3000, 1 << 18)
    elif kind == "spmm_call":
        pattern, rows, cols = rng.choice(["uniform", "power_law"]), _log_int(rng, 300, 16384), \
            _log_int(rng, 300, 16384)
    elif kind in ("train", "sddmm"):
        pattern = "graph"
        rows = cols = _log_int(rng, 3000, 200000)
    else:
        pattern = rng.choice(["uniform", "power_law", "graph"])
        rows = _log_int(rng, 2000, 262144)
        cols = rows if pattern == "graph" else _log_int(rng, 2000, 262144)
    dtype = {"sddmm": ["f32", "f64"], "coo": ["f32", "f32", "bf16", "f64"],
             "train": ["bf16", "f32", "f16"]}.get(kind, ["f32", "f32", "f64", "bf16", "f16"])
    case = {"kind": kind, "pattern": pattern, "rows": rows, "cols": cols, "mean": rng.randint(6, 30),
            "dtype": rng.choice(dtype), "index": "i32" if kind == "sddmm" else rng.choice(["i32", "i64"])}
    if kind in ("spmv", "spmm_call", "spmm", "coo"):
        case["op"] = rng.choice(["non", "non", "trans"])
    if kind != "spmv":
        case["n"] = rng.choice([8, 16, 32, 64, 128]) if rng.random() < 0.5 else _log_int(rng, 3, 160)
    return case


# ------------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _uniform(shape, dtype, g):
    """U[-1, 1] in the storage dtype."""
    t = torch.rand(shape, generator=g, dtype=torch.float64 if dtype == torch.float64 else torch.float32,
                   device=DEVICE)
    return t.mul_(2).sub_(1).to(dtype)


def _normal(shape, dtype, g):
    t = torch.randn(shape, generator=g, dtype=torch.float64 if dtype == torch.float64 else torch.float32,
                    device=DEVICE)
    return t.to(dtype)


def _starts(lengths):
    ptr = torch.zeros(lengths.numel() + 1, dtype=torch.int64, device=DEVICE)
    torch.cumsum(lengths, 0, out=ptr[1:])
    return ptr


def _spread(lengths, widths, g):
    """(row pointer, columns): row r takes one uniform column from each of
    lengths[r] equal strata of its widths[r] columns, so its columns are
    distinct and ascending."""
    ptr = _starts(lengths)
    nnz = int(ptr[-1])
    owner = torch.repeat_interleave(lengths, output_size=nnz)
    j = torch.arange(nnz, device=DEVICE) - ptr[owner]
    L = lengths[owner]
    W = widths[owner] if torch.is_tensor(widths) else widths
    lo = torch.div(j * W, L, rounding_mode="floor")
    hi = torch.div((j + 1) * W, L, rounding_mode="floor")
    del j, L, owner
    pick = torch.rand(nnz, generator=g, device=DEVICE)
    return ptr, torch.minimum(lo + (pick * (hi - lo)).to(torch.int64), hi - 1)


def _pattern(case, g):
    """(row pointer, columns), int64."""
    rows, cols, mean = case["rows"], case["cols"], case["mean"]
    if case["pattern"] == "uniform":
        return _spread(torch.full((rows,), min(mean, cols), dtype=torch.int64, device=DEVICE), cols, g)
    if case["pattern"] == "power_law":
        cap = min(4096, cols)
        xm = power_law_scale(2.1, mean, cap)
        u = 1.0 - torch.rand(rows, generator=g, dtype=torch.float64, device=DEVICE)
        return _spread(torch.floor(xm * u ** (-1.0 / 1.1)).clamp_(max=cap).to(torch.int64), cols, g)
    w = (1.0 - torch.rand(rows, generator=g, dtype=torch.float64, device=DEVICE)) ** (-1.0 / 1.3)
    w = torch.minimum(w, w.sum().sqrt())
    cdf = torch.cumsum(w, 0) / w.sum()
    m = min(rows * mean // 2, rows * (rows - 1) // 4)
    key = torch.empty(0, dtype=torch.int64, device=DEVICE)
    while key.numel() < m:  # m distinct undirected edges (the same number for every seed)
        ends = torch.searchsorted(cdf, torch.rand(2, m + m // 4 + 64, generator=g, dtype=torch.float64, device=DEVICE))
        lo, hi = ends.clamp_(max=rows - 1).sort(0).values
        key = torch.unique(torch.cat([key, (lo * rows + hi)[lo < hi]]))
    key = key[torch.randperm(key.numel(), generator=g, device=DEVICE)[:m]]
    key = torch.cat([key, key % rows * rows + key // rows]).sort().values
    return _starts(torch.bincount(key // rows, minlength=rows)), key % rows


def _csr(case, g):
    """(values, columns, row pointer) in the case's types."""
    ptr, col = _pattern(case, g)
    it = INDEX[case["index"]]
    return _uniform((col.numel(),), DTYPES[case["dtype"]], g), col.to(it), ptr.to(it)


def _coo(case, g):
    """The nonzeros in no particular order."""
    val, col, ptr = _csr(case, g)
    order = torch.randperm(col.numel(), generator=g, device=DEVICE)
    return val[order], _rows_of(ptr)[order].to(col.dtype), col[order]


def _blocks(case, g):
    """(blocks, block columns, block row pointer); fp8 blocks as float32, before quantisation."""
    nbr, nbc = -(-case["rows"] // 16), -(-case["cols"] // 16)
    ptr, col = _spread(torch.full((nbr,), min(case["mean"], nbc), dtype=torch.int64, device=DEVICE), nbc, g)
    dt = torch.float32 if case["dtype"] == "fp8" else DTYPES[case["dtype"]]
    return _normal((col.numel(), 16, 16), dt, g), col.to(torch.int32), ptr.to(torch.int32)


def _batch(case, g):
    """(values, local columns, local row pointers, row offsets, nonzero offsets): square matrices of
    log-uniform size, row lengths uniform around ``mean``."""
    lo, hi = 64, max(65, case["rows"])
    u = (torch.randperm(case["mats"], generator=g, device=DEVICE).double() + 0.5) / case["mats"]
    size = torch.exp(math.log(lo) + u * math.log((hi + 1) / lo)).to(torch.int64).clamp_(lo, hi)
    offs = _starts(size)
    mat = torch.repeat_interleave(size)
    per = torch.randint(4, 2 * case["mean"] - 3, (mat.numel(),), generator=g, device=DEVICE)
    per = torch.minimum(per, size[mat])
    ptr, col = _spread(per, size[mat], g)
    nnz = ptr[offs]
    local = torch.zeros(mat.numel() + case["mats"], dtype=torch.int64, device=DEVICE)
    local[torch.arange(mat.numel(), device=DEVICE) + mat + 1] = ptr[1:] - nnz[mat]
    val = _uniform((col.numel(),), DTYPES[case["dtype"]], g)
    return val, col.to(torch.int32), local.to(torch.int32), offs, nnz, ptr, offs[mat]


def _dense_rows(case):
    return case["rows"] if case.get("op") == "trans" else case["cols"]


def prepare(case, seed):
    """Inputs and the prepared object a program keeps across calls."""
    g = _generator(seed)
    kind = case["kind"]
    shape = (case["rows"], case["cols"]) if "cols" in case else None
    s = {"kind": kind, "shape": shape, "op": case.get("op")}
    if kind == "bsr":
        blocks, bcol, bptr = _blocks(case, g)
        s["scales"] = None
        if case["dtype"] == "fp8":
            blocks, s["scales"] = fs.quantize_bsr_fp8(blocks)
        s.update(blocks=blocks, bcol=bcol, bptr=bptr, B=_normal((case["cols"], case["n"]), torch.float32, g))
        return s
    dt = DTYPES[case["dtype"]]
    if kind == "batch":
        val, col, local, offs, nnz, _, _ = _batch(case, g)
        s["batch"] = CsrBatch(val, col, local, offs, nnz_offsets=nnz)
        total = s["batch"].total_cols
        if case["op"] == "spmv":
            s["x"] = _uniform((total,), dt, g)
            s["batch"].params("spmv")  # tuned once, as a serving program does at start-up
        else:
            s["x"] = _normal((total, case["n"]), dt, g)
            s["batch"].params("spmm", case["n"])
        return s
    if kind == "coo":
        val, row, col = _coo(case, g)
        s["prepared"] = fs.prepare_spmm_coo_route(val, row, col, shape, op=case["op"])
        s["B"] = _normal((_dense_rows(case), case["n"]), dt, g)
        return s
    val, col, ptr = _csr(case, g)
    if kind == "spmv":
        s["prepared"] = fs.prepare_spmv_csr(val, col, ptr, shape, op=case["op"])
        s["x"] = _uniform((_dense_rows(case),), dt, g)
    elif kind == "spmm_call":
        s.update(csr=(val, col, ptr), B=_normal((_dense_rows(case), case["n"]), dt, g))
    elif kind == "spmm":
        s["route"] = case["op"] != "non" or case["dtype"] in ("bf16", "f16")
        make = fs.prepare_spmm_csr_route if s["route"] else fs.prepare_spmm_csr_opt
        s["prepared"] = make(val, col, ptr, shape, **({"op": case["op"]} if s["route"] else {}))
        s["B"] = _normal((_dense_rows(case), case["n"]), dt, g)
    elif kind == "sddmm":
        s["prepared"] = fs.prepare_sddmm_csr(col, ptr, shape)
        s.update(val=val, X=_normal((case["rows"], case["n"]), dt, g), Y=_normal((case["cols"], case["n"]), dt, g))
    elif kind == "train":
        s["matrix"] = fs.CsrMatrix(col, ptr, shape).prepare_backward()
        s["val"] = val.requires_grad_()
        s["B"] = _normal((case["cols"], case["n"]), dt, g).requires_grad_()
        s["dC"] = _normal((case["rows"], case["n"]), dt, g)
    return s


def run(s):
    """One pass through the public API."""
    kind = s["kind"]
    if kind == "spmv":
        return fs.flagsparse_spmv_csr(x=s["x"], prepared=s["prepared"])
    if kind == "spmm_call":
        return fs.flagsparse_spmm_csr(*s["csr"], s["B"], s["shape"], op=s["op"])
    if kind == "spmm":
        if s["route"]:
            return fs.flagsparse_spmm_csr_run(s["prepared"], s["B"])
        return fs.flagsparse_spmm_csr_opt(B=s["B"], prepared=s["prepared"])
    if kind == "sddmm":
        return fs.flagsparse_sddmm_csr(data=s["val"], x=s["X"], y=s["Y"], alpha=1.25, beta=0.5, prepared=s["prepared"])
    if kind == "train":
        C = fs.spmm_csr_autograd(s["val"], s["B"], s["matrix"])
        d_val, d_B = torch.autograd.grad(C, (s["val"], s["B"]), s["dC"])
        return C.detach(), d_val, d_B
    if kind == "bsr":
        return fs.flagsparse_spmm_bsr(s["blocks"], s["bcol"], s["bptr"], s["B"], s["shape"], scales=s["scales"])
    if kind == "batch":
        return s["batch"].spmv(s["x"]) if s["op"] == "spmv" else s["batch"].spmm(s["x"])
    return fs.flagsparse_spmm_coo_run(s["prepared"], s["B"])


def work(case):
    """Bytes (each input read once, each output written once) and operations of one pass."""
    kind, n = case["kind"], case.get("n", 1)
    if kind == "bsr":
        nbr, nbc = -(-case["rows"] // 16), -(-case["cols"] // 16)
        nnzb = nbr * min(case["mean"], nbc)
        b = nnzb * (256 * BYTES[case["dtype"]] + 4 + (4 if case["dtype"] == "fp8" else 0)) + 4 * (nbr + 1)
        return {"bytes": b + 4 * n * (case["cols"] + case["rows"]), "flops": 512 * nnzb * n}
    e = BYTES[case["dtype"]]
    if kind == "batch":
        lo, hi = 64, max(65, case["rows"])
        total = case["mats"] * (hi - lo) / math.log(hi / lo)
        nnz = total * (case["mean"])
        return {"bytes": nnz * (e + 4) + 4 * total + 2 * total * n * e, "flops": 2 * nnz * n}
    i = BYTES[case["index"]]
    nnz = case["rows"] * min(case["mean"], case["cols"])
    dense = (case["rows"] + case["cols"]) * n * e
    csr = nnz * (e + i) + (case["rows"] + 1) * i
    if kind == "coo":
        return {"bytes": nnz * (e + 2 * i) + dense, "flops": 2 * nnz * n}
    if kind == "sddmm":
        return {"bytes": csr + nnz * e + dense, "flops": 2 * nnz * n}
    if kind == "train":  # A, B and dC in; C, dB and dvalues out
        return {"bytes": csr + nnz * e + 2 * dense, "flops": 6 * nnz * n}
    return {"bytes": csr + dense, "flops": 2 * nnz * n}


# -------------------------------------------------------------------- exact
def _rows_of(ptr):
    return torch.repeat_interleave((ptr[1:] - ptr[:-1]).to(torch.int64))


def _product(val, row, col, B, n_out):
    """sum over nonzeros of val * B[col] into row, in float64."""
    B = B.double()
    C = torch.zeros((n_out,) + tuple(B.shape[1:]), dtype=torch.float64, device=DEVICE)
    step = max(1, CHUNK // max(1, B.shape[1] if B.ndim == 2 else 1))
    for p in range(0, val.numel(), step):
        v = val[p:p + step].double()
        C.index_add_(0, row[p:p + step].long(),
                     (v[:, None] if B.ndim == 2 else v) * B[col[p:p + step].long()])
    return C


def _dots(row, col, X, Y):
    out = torch.empty(row.numel(), dtype=torch.float64, device=DEVICE)
    step = max(1, CHUNK // X.shape[1])
    for p in range(0, row.numel(), step):
        out[p:p + step] = (X[row[p:p + step].long()].double() * Y[col[p:p + step].long()].double()).sum(1)
    return out


def exact(case, seed):
    """run()'s outputs in float64, from plain torch."""
    g = _generator(seed)
    kind = case["kind"]
    if kind == "bsr":
        blocks, bcol, bptr = _blocks(case, g)
        B = _normal((case["cols"], case["n"]), torch.float32, g).double()
        nbr, nbc = bptr.numel() - 1, -(-case["cols"] // 16)
        Bp = torch.zeros((nbc * 16, case["n"]), dtype=torch.float64, device=DEVICE)
        Bp[: case["cols"]] = B
        Bp = Bp.view(nbc, 16, case["n"])
        C = torch.zeros((nbr, 16, case["n"]), dtype=torch.float64, device=DEVICE)
        brow = _rows_of(bptr)
        for p in range(0, bcol.numel(), 8192):
            C.index_add_(0, brow[p:p + 8192], torch.bmm(blocks[p:p + 8192].double(), Bp[bcol[p:p + 8192].long()]))
        return C.view(nbr * 16, case["n"])[: case["rows"]]
    dt = DTYPES[case["dtype"]]
    if kind == "batch":
        val, col, _, offs, _, ptr, base = _batch(case, g)
        row = _rows_of(ptr)
        total = int(offs[-1])
        x = _uniform((total,), dt, g) if case["op"] == "spmv" else _normal((total, case["n"]), dt, g)
        return _product(val, row, col.long() + base[row], x, total)
    if kind == "coo":
        val, row, col = _coo(case, g)
    else:
        val, col, ptr = _csr(case, g)
        row = _rows_of(ptr)
    if kind == "sddmm":
        X, Y = _normal((case["rows"], case["n"]), dt, g), _normal((case["cols"], case["n"]), dt, g)
        return 1.25 * _dots(row, col, X, Y) + 0.5 * val.double()
    if kind == "train":
        B = _normal((case["cols"], case["n"]), dt, g)
        dC = _normal((case["rows"], case["n"]), dt, g)
        return (_product(val, row, col, B, case["rows"]), _dots(row, col, dC, B),
                _product(val, col, row, dC, case["cols"]))
    n_out = case["rows"]
    if case["op"] == "trans":
        row, col, n_out = col, row, case["cols"]
    B = _uniform((_dense_rows(case),), dt, g) if kind == "spmv" else _normal((_dense_rows(case), case["n"]), dt, g)
    return _product(val, row, col, B, n_out)
