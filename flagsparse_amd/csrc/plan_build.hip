// Validation figures, row bins and long-row segments of a CSR in one go, all
// on the device, so that the host reads one small buffer back and needs no
// second round trip for the rows that are cut into segments.
//
// A small structure (kSmallRows rows, kSmallNnz nonzeros) takes ONE launch of
// one 1024-thread workgroup: at that size the work is a few microseconds and
// every further launch costs as much as all of it (an unprepared SpMM call of
// 4096 power-law rows, 65536 nonzeros, N = 32: 239 us with eight plan launches,
// six copies and a second readback for the segments, 78 us now).  Larger ones
// take a counting pass over rows and columns (a workgroup per 1024 rows,
// per-workgroup results instead of atomics, so nothing has to be cleared
// first), one workgroup that reduces and scans the counts, the stable scatter
// of the row ids, and the workgroups that write the segments (20000 rows and
// one of 16 M nonzeros: 77 us in all, 39 ms with a thread per row; 50000 rows of
// 5000: 0.65 ms and 1.8).
//
// A launch more before the readback costs more than its run: with the ranges
// and the segments in kernels of their own the host's wait outgrew the time that
// it polls, and the first product on a new matrix of 9904 rows took 163 us
// instead of 140.
//
// The structure is not trusted: lengths are taken as they come, and every
// write is bounded by the sizes the caller passes.
#include "fsp_device.hpp"
#include "fsp_host.hpp"
#include "plan_kernels.hpp"

namespace fsp {

constexpr int kBuildThreads = 1024;
constexpr int kBuildWaves = kBuildThreads / 64;
constexpr int64_t kSmallRows = 8192;
constexpr int64_t kSmallNnz = 1 << 17;
constexpr int kMetaStats = 6;

// What the caller gets: meta = the six figures, n_bins + 1 bin offsets and
// the number of segments (see fsp_csr_build_plan).
struct build_out {
  int64_t* meta;
  int32_t* rows;
  int64_t max_segments;
  int32_t* seg_row;
  int64_t* seg_begin;
  int64_t* seg_end;
  int64_t max_long;
  int64_t* long_seg_ptr;
};

struct csr_figures {
  int64_t dec, longest, lo, hi;
};

__device__ __forceinline__ csr_figures no_figures() { return {0, 0, kStatsMin, kStatsMax}; }
__device__ __forceinline__ csr_figures merge(const csr_figures& a, const csr_figures& b) {
  return {a.dec + b.dec, a.longest > b.longest ? a.longest : b.longest, a.lo < b.lo ? a.lo : b.lo,
          a.hi > b.hi ? a.hi : b.hi};
}
__device__ __forceinline__ csr_figures wave_merge(csr_figures f) {
  for (int m = 32; m > 0; m >>= 1) {
    f = merge(f, csr_figures{__shfl_xor(f.dec, m), __shfl_xor(f.longest, m), __shfl_xor(f.lo, m), __shfl_xor(f.hi, m)});
  }
  return f;
}
// The figures of a workgroup, in its first wave; s has one entry per wave.
__device__ __forceinline__ csr_figures block_merge(csr_figures f, csr_figures* s, int waves) {
  f = wave_merge(f);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = f;
  __syncthreads();
  f = static_cast<int>(threadIdx.x) < waves ? s[threadIdx.x] : no_figures();
  return threadIdx.x < 64 ? wave_merge(f) : f;
}

__device__ __forceinline__ void write_figures(int64_t* meta, int64_t first, int64_t last, const csr_figures& f) {
  meta[0] = first;
  meta[1] = last;
  meta[2] = f.dec;
  meta[3] = f.lo;
  meta[4] = f.hi;
  meta[5] = f.longest;
}

// Smallest and largest column of this thread's share, four loads in flight.
template <typename IT>
__device__ __forceinline__ csr_figures column_figures(const IT* __restrict__ indices, int64_t nnz, int64_t first,
                                                      int64_t stride) {
  csr_figures f = no_figures();
  for (int64_t p = first; p < nnz; p += 4 * stride) {
    int64_t c[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) c[u] = static_cast<int64_t>(indices[p + u * stride < nnz ? p + u * stride : p]);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      f.lo = c[u] < f.lo ? c[u] : f.lo;
      f.hi = c[u] > f.hi ? c[u] : f.hi;
    }
  }
  return f;
}

// Inclusive sum over the 1024 threads of a workgroup; total in `total`.
__device__ __forceinline__ int64_t block_scan(int64_t v, int64_t* s_wave, int64_t& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int d = 1; d < 64; d <<= 1) {
    const int64_t o = __shfl_up(v, d);
    if (lane >= d) v += o;
  }
  if (lane == 63) s_wave[wave] = v;
  __syncthreads();
  int64_t before = 0;
  total = 0;
  for (int w = 0; w < kBuildWaves; ++w) {
    if (w < wave) before += s_wave[w];
    total += s_wave[w];
  }
  __syncthreads();
  return before + v;
}

// Segment j of the n that a row's [b, b + len) is cut into; `at` is below max_segments.
__device__ __forceinline__ void write_segment(const build_out& out, int64_t at, int64_t j, int64_t n, int64_t row,
                                              int64_t b, int64_t len) {
  out.seg_row[at] = static_cast<int32_t>(row);
  out.seg_begin[at] = b + len * j / n;
  out.seg_end[at] = b + len * (j + 1) / n;
}

// Segments of the long rows rows[first, n_rows): row i of them is cut evenly
// into ceil(len / seg_len) segments.  Every one of `parts` workgroups (a power of
// two) scans all rows' counts, 1024 at a time.  Rows of few segments are written
// by a lane each, every parts-th run of them by one workgroup, a run as long as
// leaves each workgroup one and at most 1024, so that a wave's lanes write side by
// side (one lane takes 0.6 us a segment: two divisions and three stores after one
// another).  Rows of more are written by a wave each, every parts-th row by one
// workgroup, and rows of very many by all workgroups together.  Against one
// thread a row in one workgroup, whole plan: 262144 power-law rows 198 -> 139 us,
// 50000 rows of 4 segments 288 -> 173, 3000 rows of 40 280 -> 80, 64 rows of 118
// 81 -> 60, one row of 62500 among 20001 40 ms -> 76 us; 2000 rows of 4 are even
// (62 and 61).
constexpr int kLaneSegments = 16;
constexpr int kWaveSegments = 1024;
template <typename PT>
__device__ __forceinline__ void write_segments(const PT* __restrict__ indptr, int64_t n_rows, int64_t first,
                                               int64_t seg_len, const build_out& out, int64_t* s_wave,
                                               int64_t* n_segments, unsigned part, unsigned parts) {
  int64_t n_long = n_rows - first;
  if (n_long > out.max_long) n_long = out.max_long;
  int run_log2 = 0;
  while (run_log2 < 10 && (n_long >> (run_log2 + 1)) >= int64_t(parts)) ++run_log2;
  int64_t carry = 0;
  for (int64_t base = 0; base < n_long; base += kBuildThreads) {  // uniform
    const int64_t i = base + threadIdx.x;
    const bool live = i < n_long;
    int64_t row = 0, b = 0, len = 0, n = 0;
    if (live) {
      row = out.rows[first + i];
      b = static_cast<int64_t>(indptr[row]);
      len = static_cast<int64_t>(indptr[row + 1]) - b;
      n = (len + seg_len - 1) / seg_len;
      if (n < 0) n = 0;
      if (n > out.max_segments) n = out.max_segments;
    }
    int64_t total;
    const int64_t at = carry + block_scan(n, s_wave, total) - n;
    carry += total;
    if (live && part == 0) out.long_seg_ptr[i] = at;
    const bool few = n <= kLaneSegments;
    const bool mine = ((few ? i >> run_log2 : i) & (parts - 1)) == part;
    if (mine && few) {
      for (int64_t j = 0; j < n && at + j < out.max_segments; ++j) write_segment(out, at + j, j, n, row, b, len);
    }
    for (uint64_t left = __ballot(!few && (mine || n > kWaveSegments)); left != 0; left &= left - 1) {  // wave-uniform
      const int from = __ffsll(static_cast<unsigned long long>(left)) - 1;
      const int64_t n_w = __shfl(n, from);
      const bool shared = n_w > kWaveSegments;
      const int64_t at_w = __shfl(at, from), row_w = __shfl(row, from), b_w = __shfl(b, from), len_w = __shfl(len, from);
      const int64_t step = shared ? int64_t(parts) * 64 : 64;
      for (int64_t j = (shared ? int64_t(part) * 64 : 0) + (threadIdx.x & 63); j < n_w && at_w + j < out.max_segments; j += step) {
        write_segment(out, at_w + j, j, n_w, row_w, b_w, len_w);
      }
    }
  }
  if (threadIdx.x == 0 && part == 0) {
    if (n_long > 0) out.long_seg_ptr[n_long] = carry;
    *n_segments = carry;
  }
}

template <typename PT, typename IT>
__global__ __launch_bounds__(kBuildThreads) void plan_small_kernel(const PT* __restrict__ indptr,
                                                                   const IT* __restrict__ indices, int64_t n_rows,
                                                                   int64_t nnz, int n_bins, bin_bounds bb,
                                                                   int64_t seg_len, build_out out) {
  __shared__ csr_figures s_fig[kBuildWaves];
  __shared__ int64_t s_wave[kBuildWaves];
  __shared__ int s_cnt[FSP_MAX_BINS];
  __shared__ int s_off[FSP_MAX_BINS + 1];
  __shared__ int s_base[FSP_MAX_BINS];
  __shared__ int s_wave_cnt[kBuildWaves][FSP_MAX_BINS];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  if (t < FSP_MAX_BINS) s_cnt[t] = 0;
  __syncthreads();
  csr_figures f = column_figures(indices, nnz, t, kBuildThreads);
  for (int64_t r = t; r < n_rows; r += kBuildThreads) {
    const int64_t len = static_cast<int64_t>(indptr[r + 1]) - static_cast<int64_t>(indptr[r]);
    f.dec += len < 0 ? 1 : 0;
    f.longest = len > f.longest ? len : f.longest;
    if (n_bins > 0) atomicAdd(&s_cnt[bin_of(len, bb, n_bins)], 1);
  }
  f = block_merge(f, s_fig, kBuildWaves);  // its barrier publishes s_cnt too
  if (t == 0) {
    write_figures(out.meta, static_cast<int64_t>(indptr[0]), static_cast<int64_t>(indptr[n_rows]), f);
    int off = 0;
    for (int b = 0; b < n_bins; ++b) {
      s_off[b] = s_base[b] = off;
      out.meta[kMetaStats + b] = off;
      off += s_cnt[b];
    }
    if (n_bins > 0) {
      s_off[n_bins] = off;
      out.meta[kMetaStats + n_bins] = off;
    }
  }
  __syncthreads();
  if (n_bins == 0) return;
  const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  for (int64_t base = 0; base < n_rows; base += kBuildThreads) {  // uniform
    const int64_t r = base + t;
    int b = -1, rank = 0;
    if (r < n_rows) b = bin_of(static_cast<int64_t>(indptr[r + 1]) - static_cast<int64_t>(indptr[r]), bb, n_bins);
    for (int j = 0; j < n_bins; ++j) {
      const uint64_t m = __ballot(b == j);
      if (b == j) rank = __popcll(m & lt_mask);
      if (lane == 0) s_wave_cnt[wave][j] = __popcll(m);
    }
    __syncthreads();
    if (b >= 0) {
      int pos = s_base[b] + rank;
      for (int w = 0; w < wave; ++w) pos += s_wave_cnt[w][b];
      out.rows[pos] = static_cast<int32_t>(r);
    }
    __syncthreads();
    if (t < n_bins) {
      int tot = 0;
      for (int w = 0; w < kBuildWaves; ++w) tot += s_wave_cnt[w][t];
      s_base[t] += tot;
    }
    __syncthreads();  // the last one also orders the row ids before their reads below
  }
  write_segments(indptr, n_rows, s_off[n_bins - 1], seg_len, out, s_wave, &out.meta[kMetaStats + n_bins + 1], 0, 1);
}

// Workgroup b counts the bins of rows [1024 b, 1024 (b + 1)) into
// counts[bin * n_row_blocks + b] and takes every gridDim-th share of the
// columns; its figures go to figures[b].
template <typename PT, typename IT>
__global__ __launch_bounds__(FSP_WG_THREADS) void plan_count_kernel(const PT* __restrict__ indptr,
                                                                    const IT* __restrict__ indices, int64_t n_rows,
                                                                    int64_t nnz, int n_bins, bin_bounds bb,
                                                                    int64_t n_row_blocks, int64_t* __restrict__ counts,
                                                                    csr_figures* __restrict__ figures) {
  __shared__ csr_figures s_fig[FSP_WAVES];
  __shared__ int s_cnt[FSP_MAX_BINS];
  if (threadIdx.x < FSP_MAX_BINS) s_cnt[threadIdx.x] = 0;
  __syncthreads();
  const int64_t blk = blockIdx.x;
  csr_figures f = column_figures(indices, nnz, blk * FSP_WG_THREADS + threadIdx.x,
                                 static_cast<int64_t>(gridDim.x) * FSP_WG_THREADS);
  if (blk < n_row_blocks) {
    for (int k = 0; k < kBinItems; ++k) {
      const int64_t r = blk * kBinRowsPerBlock + k * FSP_WG_THREADS + threadIdx.x;
      if (r < n_rows) {
        const int64_t len = static_cast<int64_t>(indptr[r + 1]) - static_cast<int64_t>(indptr[r]);
        f.dec += len < 0 ? 1 : 0;
        f.longest = len > f.longest ? len : f.longest;
        if (n_bins > 0) atomicAdd(&s_cnt[bin_of(len, bb, n_bins)], 1);
      }
    }
  }
  f = block_merge(f, s_fig, FSP_WAVES);
  if (threadIdx.x == 0) figures[blk] = f;
  if (blk < n_row_blocks && static_cast<int>(threadIdx.x) < n_bins) {
    counts[threadIdx.x * n_row_blocks + blk] = s_cnt[threadIdx.x];
  }
}

// Reduces the workgroups' figures and scans the counts in place; one workgroup.
template <typename PT>
__global__ __launch_bounds__(kBuildThreads) void plan_reduce_kernel(const PT* __restrict__ indptr, int64_t n_rows,
                                                                    int n_bins, int64_t n_row_blocks,
                                                                    int64_t* __restrict__ counts,
                                                                    const csr_figures* __restrict__ figures,
                                                                    int64_t n_figures, int64_t* __restrict__ meta) {
  __shared__ csr_figures s_fig[kBuildWaves];
  __shared__ int64_t s_wave[kBuildWaves];
  csr_figures f = no_figures();
  for (int64_t i = threadIdx.x; i < n_figures; i += kBuildThreads) f = merge(f, figures[i]);
  f = block_merge(f, s_fig, kBuildWaves);
  if (threadIdx.x == 0) {
    write_figures(meta, static_cast<int64_t>(indptr[0]), static_cast<int64_t>(indptr[n_rows]), f);
  }
  constexpr int kItems = 4;
  const int64_t n = n_row_blocks * n_bins;
  int64_t carry = 0;
  for (int64_t base = 0; base < n; base += kBuildThreads * kItems) {  // uniform
    const int64_t i0 = base + static_cast<int64_t>(threadIdx.x) * kItems;
    int64_t v[kItems], sum = 0;
#pragma unroll
    for (int k = 0; k < kItems; ++k) v[k] = i0 + k < n ? counts[i0 + k] : 0;
#pragma unroll
    for (int k = 0; k < kItems; ++k) sum += v[k];
    int64_t total;
    int64_t at = carry + block_scan(sum, s_wave, total) - sum;
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
      const int64_t i = i0 + k;
      if (i < n) {
        counts[i] = at;
        if (i % n_row_blocks == 0) meta[kMetaStats + i / n_row_blocks] = at;
      }
      at += v[k];
    }
    carry += total;
  }
  if (threadIdx.x == 0 && n_bins > 0) meta[kMetaStats + n_bins] = n_rows;
}

template <typename PT>
__global__ __launch_bounds__(kBuildThreads) void plan_segments_kernel(const PT* __restrict__ indptr, int64_t n_rows,
                                                                      int n_bins, int64_t seg_len, build_out out) {
  __shared__ int64_t s_wave[kBuildWaves];
  write_segments(indptr, n_rows, out.meta[kMetaStats + n_bins - 1], seg_len, out, s_wave,
                 &out.meta[kMetaStats + n_bins + 1], blockIdx.x, gridDim.x);
}

static inline int64_t build_row_blocks(int64_t n_rows) {
  const int64_t b = ceil_div(n_rows, int64_t(kBinRowsPerBlock));
  return b > 0 ? b : 1;
}
// Workgroups of the counting pass: one per 1024 rows, and enough for the
// columns (16 per thread) up to four per CU.
static inline int64_t build_blocks(int64_t n_rows, int64_t nnz) {
  int64_t c = ceil_div(nnz, int64_t(FSP_WG_THREADS) * 16);
  if (c > 1024) c = 1024;
  const int64_t r = build_row_blocks(n_rows);
  return c > r ? c : r;
}
// Workgroups that write the segments, of which the caller provides for
// max_segments: a power of two, one per 1024 up to 64.
static inline int64_t segment_blocks(int64_t max_segments) {
  int64_t b = 1;
  while (b < 64 && b * 1024 < max_segments) b *= 2;
  return b;
}

}  // namespace fsp

using namespace fsp;

extern "C" {

int fsp_csr_build_plan_workspace(int64_t n_rows, int64_t nnz, int32_t n_bins, int64_t* bytes) {
  if (bytes == nullptr || n_rows < 0 || nnz < 0 || n_bins < 0 || n_bins > FSP_MAX_BINS) {
    return fail(FSP_ERR_ARG, "fsp_csr_build_plan_workspace: bad arguments");
  }
  *bytes = (build_row_blocks(n_rows) * n_bins) * (int64_t)sizeof(int64_t) +
           build_blocks(n_rows, nnz) * (int64_t)sizeof(csr_figures);
  return FSP_OK;
}

int fsp_csr_build_plan(int32_t indptr_type, const void* indptr_dev, int32_t index_type, const void* indices_dev,
                       int64_t n_rows, int64_t nnz, int32_t n_bins, const int64_t* upper, int64_t seg_len,
                       int64_t* meta_dev, int32_t* rows_dev, int64_t max_segments, int32_t* seg_row_dev,
                       int64_t* seg_begin_dev, int64_t* seg_end_dev, int64_t max_long, int64_t* long_seg_ptr_dev,
                       void* ws_dev, int64_t ws_bytes, void* stream) {
  if (n_rows < 0 || nnz < 0 || n_bins < 0 || n_bins > FSP_MAX_BINS || seg_len < 1 || max_segments < 0 ||
      max_long < 0 || indptr_dev == nullptr || meta_dev == nullptr ||
      (n_bins > 0 && (upper == nullptr || (n_rows > 0 && rows_dev == nullptr))) ||
      (max_segments > 0 && (seg_row_dev == nullptr || seg_begin_dev == nullptr || seg_end_dev == nullptr)) ||
      (max_long > 0 && long_seg_ptr_dev == nullptr)) {
    return fail(FSP_ERR_ARG, "fsp_csr_build_plan: bad arguments");
  }
  if (n_bins > 0 && n_rows > (int64_t)INT32_MAX) {
    return fail(FSP_ERR_ARG, "fsp_csr_build_plan: n_rows exceeds int32 row ids");
  }
  // without columns to look at, the nonzeros only count as segments: 4096 of
  // 256 for one wave at most
  const bool small = n_rows <= kSmallRows && nnz <= (indices_dev == nullptr ? 8 * kSmallNnz : kSmallNnz);
  if (indices_dev == nullptr) nnz = 0;  // no columns to look at
  bin_bounds bb;
  for (int b = 0; b < FSP_MAX_BINS; ++b) bb.upper[b] = INT64_MAX;
  for (int b = 0; b + 1 < n_bins; ++b) bb.upper[b] = upper[b];
  const build_out out{meta_dev, rows_dev, max_segments, seg_row_dev, seg_begin_dev, seg_end_dev, max_long,
                      long_seg_ptr_dev};
  const hipStream_t s = as_stream(stream);
  const int64_t row_blocks = build_row_blocks(n_rows);
  const int64_t blocks = build_blocks(n_rows, nnz);
  if (!small) {
    int64_t need = 0;
    fsp_csr_build_plan_workspace(n_rows, nnz, n_bins, &need);
    if (ws_dev == nullptr || ws_bytes < need) {
      return fail(FSP_ERR_WORKSPACE, "fsp_csr_build_plan: workspace %lld < %lld", (long long)ws_bytes, (long long)need);
    }
  }
  FSP_DISPATCH_INDEX(indptr_type, PT, {
    const PT* ip = static_cast<const PT*>(indptr_dev);
    FSP_DISPATCH_INDEX(index_type, IT, {
      const IT* ix = static_cast<const IT*>(indices_dev);
      if (small) {
        hipLaunchKernelGGL((plan_small_kernel<PT, IT>), dim3(1), dim3(kBuildThreads), 0, s, ip, ix, n_rows, nnz,
                           n_bins, bb, seg_len, out);
        return check_launch("plan_small");
      }
      int64_t* counts = static_cast<int64_t*>(ws_dev);
      csr_figures* figures = reinterpret_cast<csr_figures*>(counts + row_blocks * n_bins);
      hipLaunchKernelGGL((plan_count_kernel<PT, IT>), dim3(static_cast<unsigned>(blocks)), dim3(FSP_WG_THREADS), 0, s,
                         ip, ix, n_rows, nnz, n_bins, bb, row_blocks, counts, figures);
      int st = check_launch("plan_count");
      if (st) return st;
      hipLaunchKernelGGL(plan_reduce_kernel<PT>, dim3(1), dim3(kBuildThreads), 0, s, ip, n_rows, n_bins, row_blocks,
                         counts, figures, blocks, meta_dev);
      st = check_launch("plan_reduce");
      if (st || n_bins == 0) return st;
      hipLaunchKernelGGL(bins_scatter_kernel<PT>, dim3(static_cast<unsigned>(row_blocks)), dim3(FSP_WG_THREADS), 0, s,
                         ip, n_rows, n_bins, bb, counts, row_blocks, rows_dev);
      st = check_launch("bins_scatter");
      if (st) return st;
      hipLaunchKernelGGL(plan_segments_kernel<PT>, dim3(static_cast<unsigned>(segment_blocks(max_segments))),
                         dim3(kBuildThreads), 0, s, ip, n_rows, n_bins, seg_len, out);
      return check_launch("plan_segments");
    });
  });
  return FSP_OK;
}

}  // extern "C"
