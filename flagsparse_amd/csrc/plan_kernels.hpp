// Row binning pieces shared by fsp_csr_row_bins and fsp_csr_build_plan.
#pragma once

#include "fsp_device.hpp"
#include "fsp_host.hpp"

namespace fsp {

// The column figures of a CSR without nonzeros.
constexpr int64_t kStatsMin = INT64_MAX;
constexpr int64_t kStatsMax = INT64_MIN;

constexpr int kBinItems = 4;                                  // rows per thread
constexpr int kBinRowsPerBlock = FSP_WG_THREADS * kBinItems;  // 1024

struct bin_bounds {
  int64_t upper[FSP_MAX_BINS];
};

__device__ __forceinline__ int bin_of(int64_t len, const bin_bounds& bb, int n_bins) {
  int b = 0;
  while (b < n_bins - 1 && len > bb.upper[b]) ++b;
  return b;
}

// Stable scatter: rows keep ascending order inside each bin.
template <typename PT>
__global__ __launch_bounds__(FSP_WG_THREADS) void bins_scatter_kernel(
    const PT* __restrict__ indptr, int64_t n_rows, int n_bins, bin_bounds bb,
    const int64_t* __restrict__ offsets, int64_t n_blocks, int32_t* __restrict__ rows_out) {
  __shared__ int s_wave_cnt[FSP_WAVES][FSP_MAX_BINS];
  __shared__ int64_t s_base[FSP_MAX_BINS];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  if (threadIdx.x < FSP_MAX_BINS) {
    s_base[threadIdx.x] =
        threadIdx.x < n_bins ? offsets[threadIdx.x * n_blocks + blockIdx.x] : 0;
  }
  __syncthreads();
  const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kBinRowsPerBlock;
  for (int k = 0; k < kBinItems; ++k) {
    const int64_t r = base + k * FSP_WG_THREADS + threadIdx.x;
    const bool valid = r < n_rows;
    int b = -1;
    if (valid) {
      const int64_t len = static_cast<int64_t>(indptr[r + 1]) - static_cast<int64_t>(indptr[r]);
      b = bin_of(len, bb, n_bins);
    }
    int my_rank = 0;
    for (int j = 0; j < n_bins; ++j) {
      const uint64_t m = __ballot(b == j);
      if (b == j) my_rank = __popcll(m & lt_mask);
      if (lane == 0) s_wave_cnt[wave][j] = __popcll(m);
    }
    __syncthreads();
    if (valid) {
      int64_t pos = s_base[b] + my_rank;
      for (int w = 0; w < wave; ++w) pos += s_wave_cnt[w][b];
      rows_out[pos] = static_cast<int32_t>(r);
    }
    __syncthreads();
    if (threadIdx.x < n_bins) {
      int tot = 0;
      for (int w = 0; w < FSP_WAVES; ++w) tot += s_wave_cnt[w][threadIdx.x];
      s_base[threadIdx.x] += tot;
    }
    __syncthreads();
  }
}

}  // namespace fsp
