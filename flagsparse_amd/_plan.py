"""Row-length work plans for the CSR kernels (prepare-time, cached).

A plan bins the rows of a CSR (or CSC) index structure by length on the GPU
(a stable multi-split, rows stay ascending inside a bin) and cuts rows longer
than the last bin into nnz-balanced segments, both in ``fsp_csr_build_plan``.
The kernels then run every bin and every segment in one launch; rows that
were split get a second, deterministic pass that adds their segment partials
in order.  Building a plan costs one device->host copy, of the validation
figures, the bin boundaries and the number of segments; running with a plan
costs no host sync.

Bin layouts per kernel family (``unroll`` = nonzeros per lane per trip):

* SpMV: lanes per row L in {4, 8, 16, 32, 64}; a row of length n goes to the
  smallest L with n <= L * unroll, L = 64 up to ``long_threshold`` (untuned
  pipelined loop: up to 1024, then a workgroup's 256 lanes).
* SpMM / SDDMM with G lanes along the dense dimension: nonzero slots per row
  S in {1, 2, ..., 64 / G}; smallest S with n <= S * unroll * slot_scale,
  S = 64 / G up to ``long_threshold``.  SDDMM uses half the lanes of a full
  K slice (``sddmm_lanes``) and walks K in two passes.

The reference rebuilds its buckets with ``torch.nonzero`` on every call
(spmv_csr.py:371-420, 910-911) or with atomic count / compact kernels
(spmm_csr.py:3022-3072, 3114-3115).
"""

import ctypes
from dataclasses import dataclass
from functools import lru_cache

import torch

from . import _lib

# Defaults, overridable per call (the autotuner picks per shape class).
SPMV_UNROLL = 4
SPMV_LONG_THRESHOLD = 4096
SPMV_SEG_LEN = 4096
SPMV_WIDE_ROW = 1024  # the pipelined loop's rows above this take a workgroup
SPMV_WIDE_LANES = 256
SPMM_UNROLL = 4
SPMM_LONG_THRESHOLD = 256
SPMM_SEG_LEN = 256
SDDMM_UNROLL = 4
SDDMM_LONG_THRESHOLD = 256
SDDMM_SEG_LEN = 256
# Rows per wave over slots per row: measured best on MI355X for power-law rows
# (mean 14-24 nonzeros) in f32 and bf16 (SpMM); SDDMM is best with one slot
# per row up to the long threshold.
SLOT_SCALE = 4
SDDMM_SLOT_SCALE = 1


@dataclass(frozen=True)
class PlanConfig:
    """Row-bin thresholds of one plan (hashable: it keys the plan cache)."""

    lanes: tuple  # lanes (SpMV) or slots (SpMM/SDDMM) of each regular bin
    uppers: tuple  # inclusive upper row length of each regular bin
    seg_len: int  # segment length of rows above the last upper bound
    unroll: int


# SpMV variant 2 stages x in LDS: x of at most this many bytes, and only for
# matrices large enough that every workgroup's one copy of x (a persistent
# grid of two 1024-thread workgroups per CU) is small beside the nonzeros
LDSX_MAX_BYTES = 65536
LDSX_MIN_NNZ = 1 << 20


def chunk_aligned(*tensors):
    """True when every tensor's storage starts on a 4-element boundary (the
    vector-chunk SpMV loop reads 4-element chunks)."""
    return all(t.data_ptr() % (4 * t.element_size()) == 0 for t in tensors)


def spmv_default_variant(x_len, elem_bytes, nnz, chunk_ok=False):
    """SpMV loop used without tuning: when x fits in LDS and the matrix is
    large, 4 (vector chunks, needs 4-element aligned index / value arrays and
    unroll 4 or 8) or else 2 (x in LDS); otherwise 0 (software-pipelined)."""
    if 0 < x_len * elem_bytes <= LDSX_MAX_BYTES and nnz >= LDSX_MIN_NNZ:
        return 4 if chunk_ok else 2
    return 0


@lru_cache(maxsize=256)
def spmv_config(unroll=SPMV_UNROLL, long_threshold=SPMV_LONG_THRESHOLD, seg_len=SPMV_SEG_LEN):
    lanes = (4, 8, 16, 32, 64)
    uppers = [min(l * unroll, long_threshold) for l in lanes[:-1]] + [long_threshold]
    return _dedupe(lanes, uppers, seg_len, unroll)


@lru_cache(maxsize=1)
def spmv_wide_config():
    """Bins of the software-pipelined loop without tuning: as spmv_config, but
    rows of more than 1024 nonzeros and the segments of long ones take a
    workgroup each.  f32, 100000 rows of 10 on average: power-law up to 4096 /
    with 20 rows of 9000, microseconds: one wave a row 15.6 / 20.4; a workgroup
    above 256: 11.2, above 512: 10.7 / 12.6, above 1024: 10.5 / 12.6, above 2048:
    11.1.  The tuner's candidates have no such bin, so a tuned plan keeps one
    wave a row."""
    base = spmv_config(long_threshold=SPMV_WIDE_ROW)
    return PlanConfig(base.lanes + (SPMV_WIDE_LANES,), base.uppers + (SPMV_LONG_THRESHOLD,), SPMV_SEG_LEN, SPMV_UNROLL)


def spmv_plan_config(x_len, elem_bytes, nnz):
    """Bins for the loop that spmv_default_variant picks."""
    return spmv_config() if spmv_default_variant(x_len, elem_bytes, nnz) else spmv_wide_config()


@lru_cache(maxsize=1024)
def rows_config(lanes_dense, unroll, long_threshold, seg_len, slot_scale=1):
    """SpMM / SDDMM bins for `lanes_dense` lanes along the dense dimension.

    A row of length n gets the fewest slots S with n <= S * unroll *
    slot_scale: slot_scale > 1 packs more rows into a wave (more independent
    rows in flight, more trips per row)."""
    max_slots = max(1, 64 // int(lanes_dense))
    lanes = []
    s = 1
    while s <= max_slots:
        lanes.append(s)
        s *= 2
    uppers = [min(l * unroll * slot_scale, long_threshold) for l in lanes[:-1]] + [long_threshold]
    return _dedupe(tuple(lanes), uppers, seg_len, unroll)


def spmm_config(lanes_dense, unroll=SPMM_UNROLL, long_threshold=SPMM_LONG_THRESHOLD, seg_len=SPMM_SEG_LEN,
                slot_scale=SLOT_SCALE):
    return rows_config(lanes_dense, unroll, long_threshold, seg_len, slot_scale)


def sddmm_config(lanes_dense, unroll=SDDMM_UNROLL, long_threshold=SDDMM_LONG_THRESHOLD, seg_len=SDDMM_SEG_LEN,
                 slot_scale=SDDMM_SLOT_SCALE):
    return rows_config(lanes_dense, unroll, long_threshold, seg_len, slot_scale)


def _dedupe(lanes, uppers, seg_len, unroll):
    # Drop bins made empty by a small long_threshold (upper not increasing).
    keep_l, keep_u = [], []
    prev = -1
    for l, u in zip(lanes, uppers):
        if u > prev:
            keep_l.append(l)
            keep_u.append(u)
            prev = u
    return PlanConfig(tuple(keep_l), tuple(keep_u), int(max(1, seg_len)), int(unroll))


def sddmm_lanes(k, elem_bytes):
    """SDDMM lanes along K: half of a full 16-byte-per-lane slice once that
    slice spans 8 lanes or more (two passes over K per nonzero keep twice the
    nonzero slots in a wave; measured 1.6-1.7x faster on power-law graphs
    with K = 64 / 128 in f32 and bf16 on MI355X)."""
    g = lanes_for_dense(k, elem_bytes)
    return g // 2 if g >= 8 else g


def lanes_for_dense(n_dense, elem_bytes):
    """Lanes along a dense dimension of n_dense elements read 16 bytes at a time."""
    vec = max(1, 16 // int(elem_bytes))
    vcols = -(-int(n_dense) // vec)
    g = 1
    while g < 64 and g < vcols:
        g *= 2
    return g


def _index_code(t):
    return _lib.index_code(t.dtype)


@dataclass(init=False)
class CsrPlan:
    """Device work plan of one index structure (see module docstring)."""

    config: PlanConfig
    n_rows: int
    rows: torch.Tensor  # int32 [n_rows], regular bins then the long bin
    bin_counts: list  # host counts of the regular bins
    identity: bool  # the single regular bin holds rows 0..n_rows-1
    seg_row: torch.Tensor
    seg_begin: torch.Tensor
    seg_end: torch.Tensor
    long_rows: torch.Tensor
    long_seg_ptr: torch.Tensor
    n_segments: int
    n_long_rows: int
    row_len: int = 0  # > 0: every row has exactly this many nonzeros
    indptr_base: int = 0  # indptr[0] when row_len > 0

    def __init__(self, config, n_rows, rows, bin_counts, identity, seg_row, seg_begin, seg_end, long_rows, long_seg_ptr,
                 n_segments, n_long_rows, row_len=0, indptr_base=0):
        # (an assignment each would cost an unprepared call 3 us)
        self.__dict__.update(
            config=config, n_rows=n_rows, rows=rows, bin_counts=bin_counts, identity=identity, seg_row=seg_row,
            seg_begin=seg_begin, seg_end=seg_end, long_rows=long_rows, long_seg_ptr=long_seg_ptr,
            n_segments=n_segments, n_long_rows=n_long_rows, row_len=row_len, indptr_base=indptr_base, _structs={})

    # _structs: the C plans made so far.  They hold the addresses of this plan's
    # own tensors, so a field that is assigned drops them, and a copy, a pickle
    # or a plan that was saved before there were any starts without them.
    def __setattr__(self, name, value):
        object.__setattr__(self, name, value)
        object.__setattr__(self, "_structs", {})

    def __getstate__(self):
        state = dict(self.__dict__)
        state.pop("_structs", None)
        return state

    def __setstate__(self, state):
        self.__dict__.update(state, _structs={})

    @property
    def bin_sizes(self):
        return list(self.bin_counts) + [self.n_long_rows]

    def partials(self, n_dense, acc_dtype, device):
        """Scratch of n_segments x n_dense partial sums for ONE launch.

        A fresh buffer from torch's stream-ordered caching allocator on the
        current stream (the stream the launch goes to), so calls that share a
        plan on different streams never share partials; under graph capture it
        comes from the graph's private pool."""
        if self.n_segments == 0:
            return None
        return torch.empty(self.n_segments * max(1, int(n_dense)), dtype=acc_dtype, device=device)

    def struct(self, partials=None, max_blocks=0, xcd_groups=0, variant=0):
        """The C plan.  max_blocks > 0 makes the launch persistent: at most
        that many workgroups, each walking a contiguous run of row tiles;
        xcd_groups > 1 cuts each bin's tiles into that many contiguous regions
        served by the workgroups b with b % xcd_groups == region (8 = one
        region per XCD).  variant selects the SpMV loop (0 pipelined, 1 plain,
        2 plain and 3 pipelined with x staged in LDS, 4 vector chunks with x
        in LDS)."""
        key = (max_blocks, xcd_groups, variant)
        base = self._structs.get(key)
        if base is None:
            base = self._structs[key] = self._struct(max_blocks, xcd_groups, variant)
        # a copy per launch: calls on other threads and streams set their own partials
        st = _lib.FspCsrPlan.from_buffer_copy(base)
        if partials is not None:
            st.partials_dev = partials.data_ptr()
            st.partials_bytes = partials.numel() * partials.element_size()
        return st

    def _struct(self, max_blocks, xcd_groups, variant):
        st = _lib.FspCsrPlan()
        st.n_bins = len(self.bin_counts)
        st.unroll = self.config.unroll
        st.max_blocks = int(max_blocks)
        st.xcd_groups = int(xcd_groups)
        st.variant = int(variant)
        off = 0
        for i, (lanes, count) in enumerate(zip(self.config.lanes, self.bin_counts)):
            st.bins[i].lanes = int(lanes)
            st.bins[i].count = int(count)
            if self.identity or count == 0:
                st.bins[i].rows = None
            else:
                st.bins[i].rows = self.rows.data_ptr() + 4 * off
            off += count
        st.n_segments = self.n_segments
        st.n_long_rows = self.n_long_rows
        st.row_len = self.row_len
        st.indptr_base = self.indptr_base
        if self.n_segments:
            st.seg_row_dev = self.seg_row.data_ptr()
            st.seg_begin_dev = self.seg_begin.data_ptr()
            st.seg_end_dev = self.seg_end.data_ptr()
            st.long_rows_dev = self.long_rows.data_ptr()
            st.long_seg_ptr_dev = self.long_seg_ptr.data_ptr()
        return st


_N_STATS = 6  # figures ahead of the bin offsets in fsp_csr_build_plan's meta
_KEEP_BYTES = 1 << 20


def _build(indptr, indices, n_rows, nnz, config, meanwhile=None):
    """fsp_csr_build_plan and the one host readback: (figures, plan arrays).
    The plan arrays are None without `config`; they are usable only if the
    figures describe a valid CSR of at most nnz nonzeros.  meanwhile() is
    called between the copy of the figures and the wait for it: what it
    launches runs while the host waits and goes on."""
    device = indptr.device
    lib = _lib.load()
    n_bins = len(config.uppers) + 1 if config is not None else 0  # regular bins + the long bin
    n_meta = _N_STATS + (n_bins + 2 if n_bins else 0)
    ws_bytes = ctypes.c_int64(0)
    _lib.check(lib.fsp_csr_build_plan_workspace(n_rows, nnz, n_bins, ctypes.byref(ws_bytes)),
               "fsp_csr_build_plan_workspace")
    max_long = max_seg = 0
    uppers, seg_len, buf32 = None, 1, None
    if n_bins:
        seg_len = config.seg_len
        max_long = min(n_rows, nnz // (config.uppers[-1] + 1))
        max_seg = max_long + nnz // seg_len if max_long else 0
        uppers = (ctypes.c_int64 * n_bins)(*config.uppers, 0)
        buf32 = torch.empty(n_rows + max_seg, dtype=torch.int32, device=device)
    # int64 words: meta | segment begins | segment ends | segment ranges | workspace
    o_end, o_ptr = n_meta + max_seg, n_meta + 2 * max_seg
    o_ws = o_ptr + (max_long + 1 if max_long else 0)
    buf = torch.empty(o_ws + -(-ws_bytes.value // 8), dtype=torch.int64, device=device)
    at64, at32 = buf.data_ptr(), (buf32.data_ptr() if buf32 is not None else 0)
    _lib.check(
        lib.fsp_csr_build_plan(
            _index_code(indptr), indptr.data_ptr(), 0 if indices is None else _index_code(indices),
            None if indices is None else _lib.ptr(indices), n_rows, nnz, n_bins, uppers, seg_len, at64, at32, max_seg,
            at32 + 4 * n_rows, at64 + 8 * n_meta, at64 + 8 * o_end, max_long, at64 + 8 * o_ptr, at64 + 8 * o_ws,
            ws_bytes.value, _lib.stream_ptr(device),
        ),
        "fsp_csr_build_plan",
    )
    if meanwhile is None:
        host = buf[:n_meta].tolist()  # the one host sync
    else:
        stream = torch.cuda.current_stream(device)
        figures = buf[:n_meta].to("cpu", non_blocking=True)
        copied = stream.record_event()
        meanwhile()
        copied.synchronize()  # the one host sync, behind the copy only
        host = figures.tolist()
    if not n_bins:
        return host, None
    off, n_seg = host[_N_STATS:-1], host[-1]
    n_long = off[n_bins] - off[n_bins - 1]
    segments = None
    if 0 < n_long <= max_long and 0 < n_seg <= max_seg:
        segments = (buf32[n_rows:n_rows + n_seg], buf[n_meta:n_meta + n_seg], buf[o_end:o_end + n_seg],
                    buf[o_ptr:o_ptr + n_long + 1], n_seg)
    return host, (buf32[:n_rows], off, segments)


def _row_len_if_constant(n_rows, first, last, max_len):
    """The common row length when every row has max_len nonzeros (n_rows
    rows of at most max_len summing to last - first), else 0."""
    if n_rows > 0 and max_len > 0 and max_len * n_rows == last - first:
        return int(max_len)
    return 0


def build_plan(indptr, n_rows, config, nnz=None):
    """Bin the rows described by `indptr` (device tensor, int32/int64).  nnz:
    an upper bound on their nonzeros (read from indptr when not given)."""
    n_rows = int(n_rows)
    if nnz is None:
        ends = indptr[:n_rows + 1:max(1, n_rows)].tolist()
        nnz = max(0, ends[-1] - ends[0])
    host, arrays = _build(indptr, None, n_rows, int(nnz), config)
    first, last, max_len = host[0], host[1], host[5]
    return _finish_plan(indptr, n_rows, config, arrays, _row_len_if_constant(n_rows, first, last, max_len), first)


def inspect_csr(indptr, indices, n_rows, nnz, config=None, meanwhile=None):
    """Validation figures of a CSR and, with `config`, its row-bin plan, for
    ONE host readback.  Returns (stats, plan): stats has indptr_first,
    indptr_last, n_decreasing, min_col, max_col (None without nonzeros) and
    max_row; plan is None without `config` or when the row pointer is not a
    valid CSR (the caller raises on the stats first)."""
    n_rows, nnz = int(n_rows), int(nnz)
    host, arrays = _build(indptr, indices, n_rows, nnz, config, meanwhile)
    stats = {
        "indptr_first": host[0],
        "indptr_last": host[1],
        "n_decreasing": host[2],
        "min_col": host[3] if nnz else None,
        "max_col": host[4] if nnz else None,
        "max_row": host[5] if n_rows else 0,
    }
    plan = None
    if config is not None and host[0] == 0 and host[1] == nnz and host[2] == 0:
        plan = _finish_plan(indptr, n_rows, config, arrays,
                            _row_len_if_constant(n_rows, host[0], host[1], stats["max_row"]), host[0])
    return stats, plan


def _copies(*tensors):
    """Copies that are written when this returns, as everything else of a plan
    is: the next launch may be on another stream."""
    out = [t.clone() for t in tensors]
    if out[0].is_cuda:
        torch.cuda.current_stream(out[0].device).synchronize()
    return out


def _finish_plan(indptr, n_rows, config, arrays, row_len=0, indptr_base=0):
    """The plan from the arrays of _build for a valid CSR.
    row_len > 0 (every row that long, indptr[i] = indptr_base + i * row_len)
    is kept for a single-bin plan: its kernels then compute row bounds."""
    device = indptr.device
    rows, off, segments = arrays
    nb = len(config.uppers) + 1
    counts = [off[i + 1] - off[i] for i in range(nb)]
    regular = counts[:-1]
    n_long = counts[-1]
    identity = n_long == 0 and sum(1 for c in regular if c) <= 1
    if identity and n_rows:
        # one non-empty regular bin holding every row, in order: drop the list
        regular = [n_rows if c else 0 for c in regular]
    n_seg = 0
    if segments is not None:
        seg_row, seg_begin, seg_end, long_seg_ptr, n_seg = segments
        long_rows = rows[off[nb - 1]: off[nb]]
        held = seg_begin.untyped_storage().nbytes()
        if held > _KEEP_BYTES and held > 8 * 8 * n_seg:  # few segments of what was provided for
            rows, seg_row, long_rows, seg_begin, seg_end, long_seg_ptr = _copies(
                rows, seg_row, long_rows, seg_begin, seg_end, long_seg_ptr)
    else:
        if n_long:
            raise RuntimeError("the row pointer holds more nonzeros than the plan was built for")
        seg_row = long_rows = torch.empty(0, dtype=torch.int32, device=device)
        seg_begin = seg_end = long_seg_ptr = torch.empty(0, dtype=torch.int64, device=device)
        if rows.untyped_storage().nbytes() > 4 * n_rows + _KEEP_BYTES:
            rows, = _copies(rows)
    return CsrPlan(
        config=config,
        n_rows=n_rows,
        rows=rows,
        bin_counts=regular,
        identity=bool(identity),
        seg_row=seg_row,
        seg_begin=seg_begin,
        seg_end=seg_end,
        long_rows=long_rows,
        long_seg_ptr=long_seg_ptr,
        n_segments=n_seg,
        n_long_rows=int(n_long),
        row_len=int(row_len) if identity else 0,
        indptr_base=int(indptr_base) if identity and row_len else 0,
    )
