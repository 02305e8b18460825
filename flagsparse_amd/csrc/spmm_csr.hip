// Entry points of the CSR SpMM: argument checks, the all-zero cases and the
// dispatch on the value type.  The kernels are in spmm_kernels.hpp.
#include <mutex>

#include "spmm_kernels.hpp"

namespace fsp {
FSP_SPMM_INSTANCES(extern, float)
FSP_SPMM_INSTANCES(extern, double)
FSP_SPMM_INSTANCES(extern, __bf16)
FSP_SPMM_INSTANCES(extern, _Float16)
FSP_SPMM_WIDE_INSTANCE(extern, float, double)
FSP_SPMM_WIDE_INSTANCE(extern, __bf16, float)
FSP_SPMM_WIDE_INSTANCE(extern, _Float16, float)
}  // namespace fsp

// Scratch of the no-allocation SpMM entry: the long-row partials live in
// this file-scope device array (one copy per GPU, held until the process
// ends).  Host code never passes the array's name to a kernel: its device
// address on each GPU comes from hipGetSymbolAddress, resolved once per device
// with that device current and kept in scratch_dev.
static __device__ __align__(256) unsigned char scratch[FSP_NOALLOC_SCRATCH_BYTES];

namespace fsp {

constexpr int kMaxScratchDevices = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_dev[kMaxScratchDevices];

// Device address of `scratch` on the current device (resolved on first use).
static int current_scratch(void* stream, void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(FSP_ERR_LAUNCH, "fsp_spmm_csr_noalloc: hipGetDevice: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxScratchDevices) return fail(FSP_ERR_ARG, "fsp_spmm_csr_noalloc: device %d", dev);
  if (stream != nullptr) {
    int sdev = -1;
    e = hipStreamGetDevice(as_stream(stream), &sdev);
    if (e != hipSuccess) {
      return fail(FSP_ERR_LAUNCH, "fsp_spmm_csr_noalloc: hipStreamGetDevice: %s", hipGetErrorString(e));
    }
    if (sdev != dev) {
      return fail(FSP_ERR_ARG, "fsp_spmm_csr_noalloc: stream belongs to device %d, current device is %d", sdev, dev);
    }
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_dev[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      return fail(FSP_ERR_LAUNCH, "fsp_spmm_csr_noalloc: hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
    }
    g_scratch_dev[dev] = p;
  }
  *out = g_scratch_dev[dev];
  return FSP_OK;
}

static int spmm_entry(int32_t value_type, int32_t index_type, int32_t indptr_type, const void* indptr_dev,
                      const void* indices_dev, const void* data_dev, int32_t perm_type, const void* perm_dev,
                      const void* B_dev, int64_t ldb, void* C_dev, int64_t ldc, int64_t n_rows, int64_t n_dense,
                      int64_t nnz, int64_t b_rows, int32_t lanes_n, const fsp_csr_plan* plan, void* stream,
                      bool wide_values = false) {
  if (n_rows < 0 || n_dense < 0 || nnz < 0 || b_rows < 0) return fail(FSP_ERR_ARG, "fsp_spmm_csr: negative size");
  int st = check_plan(plan, n_rows);
  if (st) return st;
  if (n_rows == 0 || n_dense == 0) return FSP_OK;
  if (indptr_dev == nullptr || B_dev == nullptr || C_dev == nullptr) {
    return fail(FSP_ERR_ARG, "fsp_spmm_csr: NULL pointer");
  }
  if (ldb < n_dense || ldc < n_dense) return fail(FSP_ERR_ARG, "fsp_spmm_csr: leading dimension < n_dense");
  const hipStream_t s = as_stream(stream);
  spmm_args x{indptr_dev, indices_dev, data_dev, perm_dev, B_dev, ldb, C_dev, ldc, n_rows, n_dense, lanes_n, nnz, b_rows};
  if (nnz == 0) {
    // The kernels read clamped in-range indices; with no nonzeros there are
    // none, so the all-zero result is written directly.
    FSP_DISPATCH_VALUE(value_type, T, {
      int64_t g = ceil_div(n_rows * n_dense, FSP_WG_THREADS);
      if (g > 65536) g = 65536;
      hipLaunchKernelGGL(fill_zero_rows_kernel<T>, dim3(static_cast<unsigned>(g)), dim3(FSP_WG_THREADS), 0, s,
                         static_cast<T*>(C_dev), ldc, n_rows, n_dense);
      return check_launch("fill_zero_rows");
    });
  }
  if (indices_dev == nullptr || data_dev == nullptr || b_rows == 0) {
    return fail(FSP_ERR_ARG, "fsp_spmm_csr: NULL indices/data or empty B with nonzeros");
  }
  if (wide_values) {
    switch (value_type) {
      case FSP_F32: return spmm_wide_launch<float, double>(index_type, indptr_type, x, plan, s);
      case FSP_BF16: return spmm_wide_launch<__bf16, float>(index_type, indptr_type, x, plan, s);
      default: return spmm_wide_launch<_Float16, float>(index_type, indptr_type, x, plan, s);
    }
  }
  FSP_DISPATCH_VALUE(value_type, T, { return spmm_launch<T>(index_type, indptr_type, perm_type, x, plan, s); });
  return FSP_OK;
}

}  // namespace fsp

using namespace fsp;

extern "C" int fsp_spmm_csr(int32_t value_type, int32_t index_type, int32_t indptr_type, const void* indptr_dev,
                            const void* indices_dev, const void* data_dev, int32_t perm_type, const void* perm_dev,
                            const void* B_dev, int64_t ldb, void* C_dev, int64_t ldc, int64_t n_rows,
                            int64_t n_dense, int64_t nnz, int64_t b_rows, int32_t lanes_n,
                            const fsp_csr_plan* plan, void* stream) {
  return spmm_entry(value_type, index_type, indptr_type, indptr_dev, indices_dev, data_dev, perm_type, perm_dev,
                    B_dev, ldb, C_dev, ldc, n_rows, n_dense, nnz, b_rows, lanes_n, plan, stream);
}

extern "C" int fsp_spmm_shares_nonzeros(int32_t value_type, int32_t lanes_n, int64_t n_dense, int64_t ldb,
                                        int64_t b_rows, int32_t backward) {
  const int64_t elem = value_type == FSP_F64 ? 8 : (value_type == FSP_F32 ? 4 : 2);
  if (lanes_n < 1 || lanes_n > 64 || !is_pow2(lanes_n) || n_dense < 16 / elem || ldb < n_dense || b_rows < 0) return 0;
  return spmm_shares_nonzeros(elem, ilog2(lanes_n), n_dense, ldb, b_rows, backward != 0) ? 1 : 0;
}

extern "C" int fsp_spmm_csr_wide(int32_t dense_type, int32_t index_type, int32_t indptr_type, const void* indptr_dev,
                                 const void* indices_dev, const void* data_dev, const void* B_dev, int64_t ldb,
                                 void* C_dev, int64_t ldc, int64_t n_rows, int64_t n_dense, int64_t nnz,
                                 int64_t b_rows, int32_t lanes_n, const fsp_csr_plan* plan, void* stream) {
  if (dense_type != FSP_F32 && dense_type != FSP_BF16 && dense_type != FSP_F16) {
    return fail(FSP_ERR_DTYPE, "fsp_spmm_csr_wide: dense type %d has no wider value type", (int)dense_type);
  }
  return spmm_entry(dense_type, index_type, indptr_type, indptr_dev, indices_dev, data_dev, 0, nullptr, B_dev, ldb,
                    C_dev, ldc, n_rows, n_dense, nnz, b_rows, lanes_n, plan, stream, true);
}

namespace fsp {

// data_dev in CSC order, or (csr_values) in CSR order and read through pos.
static int trans_sddmm_entry(bool csr_values, int32_t value_type, int32_t index_type, int32_t indptr_type,
                             const void* colptr_dev, const void* rowind_dev, const void* data_dev,
                             int32_t pos_type, const void* pos_dev, const void* dC_dev, int64_t lddc,
                             const void* B_dev, int64_t ldb, void* dB_dev, int64_t lddb,
                             void* dvalues_dev, int64_t n_cols, int64_t n_dense, int64_t nnz,
                             int64_t n_rows, int32_t lanes_n, const fsp_csr_plan* plan, void* stream) {
  if (n_cols < 0 || n_dense < 0 || nnz < 0 || n_rows < 0) {
    return fail(FSP_ERR_ARG, "fsp_spmm_csr_trans_sddmm: negative size");
  }
  int st = check_plan(plan, n_cols);
  if (st) return st;
  if (colptr_dev == nullptr || (nnz > 0 && (rowind_dev == nullptr || data_dev == nullptr || pos_dev == nullptr ||
                                            dvalues_dev == nullptr || dC_dev == nullptr || B_dev == nullptr)) ||
      (n_cols > 0 && n_dense > 0 && dB_dev == nullptr)) {
    return fail(FSP_ERR_ARG, "fsp_spmm_csr_trans_sddmm: NULL pointer");
  }
  if (lddc < n_dense || ldb < n_dense || lddb < n_dense) {
    return fail(FSP_ERR_ARG, "fsp_spmm_csr_trans_sddmm: leading dimension < n_dense");
  }
  const hipStream_t s = as_stream(stream);
  if (nnz == 0 || n_dense == 0) {
    // no nonzeros: dB = 0; no dense columns: every dvalue is an empty dot, 0
    FSP_DISPATCH_VALUE(value_type, T, {
      if (n_cols > 0 && n_dense > 0) {
        int64_t g = ceil_div(n_cols * n_dense, FSP_WG_THREADS);
        if (g > 65536) g = 65536;
        hipLaunchKernelGGL(fill_zero_rows_kernel<T>, dim3(static_cast<unsigned>(g)), dim3(FSP_WG_THREADS), 0, s,
                           static_cast<T*>(dB_dev), lddb, n_cols, n_dense);
        st = check_launch("fill_zero_rows");
        if (st) return st;
      }
      if (nnz > 0) {
        int64_t g = ceil_div(nnz, FSP_WG_THREADS);
        if (g > 65536) g = 65536;
        hipLaunchKernelGGL(fill_zero_rows_kernel<T>, dim3(static_cast<unsigned>(g)), dim3(FSP_WG_THREADS), 0, s,
                           static_cast<T*>(dvalues_dev), int64_t(1), nnz, int64_t(1));
        return check_launch("fill_zero_rows");
      }
      return FSP_OK;
    });
  }
  if (n_cols == 0) return FSP_OK;  // nnz > 0 needs columns: unreachable for a valid CSC
  spmm_args x{colptr_dev, rowind_dev, data_dev, csr_values ? pos_dev : nullptr, dC_dev, lddc, dB_dev, lddb, n_cols, n_dense, lanes_n,
              nnz, n_rows};
  x.Bj = B_dev;
  x.ldbj = ldb;
  x.pos = pos_dev;
  x.dvals = dvalues_dev;
  FSP_DISPATCH_VALUE(value_type, T, { return spmm_sdd_launch<T>(index_type, indptr_type, pos_type, x, plan, s); });
  return FSP_OK;
}

}  // namespace fsp

extern "C" int fsp_spmm_csr_trans_sddmm(int32_t value_type, int32_t index_type, int32_t indptr_type,
                                        const void* colptr_dev, const void* rowind_dev, const void* data_csc_dev,
                                        int32_t pos_type, const void* pos_dev, const void* dC_dev, int64_t lddc,
                                        const void* B_dev, int64_t ldb, void* dB_dev, int64_t lddb,
                                        void* dvalues_dev, int64_t n_cols, int64_t n_dense, int64_t nnz,
                                        int64_t n_rows, int32_t lanes_n, const fsp_csr_plan* plan, void* stream) {
  return trans_sddmm_entry(false, value_type, index_type, indptr_type, colptr_dev, rowind_dev, data_csc_dev, pos_type,
                           pos_dev, dC_dev, lddc, B_dev, ldb, dB_dev, lddb, dvalues_dev, n_cols, n_dense, nnz, n_rows,
                           lanes_n, plan, stream);
}

extern "C" int fsp_spmm_csr_trans_sddmm_perm(int32_t value_type, int32_t index_type, int32_t indptr_type,
                                             const void* colptr_dev, const void* rowind_dev, const void* data_dev,
                                             int32_t pos_type, const void* pos_dev, const void* dC_dev, int64_t lddc,
                                             const void* B_dev, int64_t ldb, void* dB_dev, int64_t lddb,
                                             void* dvalues_dev, int64_t n_cols, int64_t n_dense, int64_t nnz,
                                             int64_t n_rows, int32_t lanes_n, const fsp_csr_plan* plan,
                                             void* stream) {
  return trans_sddmm_entry(true, value_type, index_type, indptr_type, colptr_dev, rowind_dev, data_dev, pos_type,
                           pos_dev, dC_dev, lddc, B_dev, ldb, dB_dev, lddb, dvalues_dev, n_cols, n_dense, nnz, n_rows,
                           lanes_n, plan, stream);
}

extern "C" int fsp_spmm_csr_noalloc(int32_t value_type, int32_t index_type, int32_t indptr_type,
                                    const void* indptr_dev, const void* indices_dev, const void* data_dev,
                                    int32_t perm_type, const void* perm_dev, const void* B_dev, int64_t ldb,
                                    void* C_dev, int64_t ldc, int64_t n_rows, int64_t n_dense, int64_t nnz,
                                    int64_t b_rows, int32_t lanes_n, const fsp_csr_plan* plan, void* stream) {
  if (plan == nullptr) return fail(FSP_ERR_ARG, "fsp_spmm_csr_noalloc: plan is NULL");
  if (n_dense < 0 || plan->n_segments < 0) return fail(FSP_ERR_ARG, "fsp_spmm_csr_noalloc: negative size");
  const int64_t acc_bytes = value_type == FSP_F64 ? 8 : 4;
  // n_segments * n_dense * acc_bytes <= the scratch size, without overflow
  if (plan->n_segments > 0 && n_dense > 0 &&
      plan->n_segments > FSP_NOALLOC_SCRATCH_BYTES / acc_bytes / n_dense) {
    return fail(FSP_ERR_WORKSPACE,
                "fsp_spmm_csr_noalloc: %lld long-row segments x %lld dense columns x %lld bytes exceed the %lld-byte "
                "static scratch; use fsp_spmm_csr with a caller-supplied partials buffer",
                (long long)plan->n_segments, (long long)n_dense, (long long)acc_bytes,
                (long long)FSP_NOALLOC_SCRATCH_BYTES);
  }
  fsp_csr_plan p = *plan;
  p.partials_dev = nullptr;
  p.partials_bytes = 0;
  if (p.n_segments > 0 && n_rows > 0 && n_dense > 0 && nnz > 0) {
    const int st = current_scratch(stream, &p.partials_dev);
    if (st) return st;
    p.partials_bytes = FSP_NOALLOC_SCRATCH_BYTES;
  }
  return spmm_entry(value_type, index_type, indptr_type, indptr_dev, indices_dev, data_dev, perm_type, perm_dev,
                    B_dev, ldb, C_dev, ldc, n_rows, n_dense, nnz, b_rows, lanes_n, &p, stream);
}
