// Entry points of the CSR SpMV: argument checks, the all-zero case and the
// dispatch on the value type.  The kernels are in spmv_kernels.hpp.
#include "spmv_kernels.hpp"

namespace fsp {
FSP_SPMV_INSTANCES(extern, float)
FSP_SPMV_INSTANCES(extern, double)
FSP_SPMV_INSTANCES(extern, __bf16)
FSP_SPMV_INSTANCES(extern, _Float16)
}  // namespace fsp

using namespace fsp;

extern "C" int fsp_spmv_csr(int32_t value_type, int32_t index_type, int32_t indptr_type,
                            const void* indptr_dev, const void* indices_dev, const void* data_dev,
                            int32_t perm_type, const void* perm_dev, const void* x_dev, void* y_dev,
                            int64_t n_rows, int64_t nnz, int64_t x_len, const fsp_csr_plan* plan, void* stream) {
  if (n_rows < 0 || nnz < 0 || x_len < 0) return fail(FSP_ERR_ARG, "fsp_spmv_csr: negative n_rows, nnz or x_len");
  int st = check_plan(plan, n_rows, kWideLanes);
  if (st) return st;
  if (n_rows == 0) return FSP_OK;
  if (indptr_dev == nullptr || y_dev == nullptr) return fail(FSP_ERR_ARG, "fsp_spmv_csr: NULL indptr or y");
  if (nnz > 0 && (indices_dev == nullptr || data_dev == nullptr || x_dev == nullptr)) {
    return fail(FSP_ERR_ARG, "fsp_spmv_csr: NULL indices, data or x");
  }
  const hipStream_t s = as_stream(stream);
  if (nnz == 0) {  // y = 0: the row kernels read the first nonzero unconditionally
    FSP_DISPATCH_VALUE(value_type, T, {
      int64_t g = ceil_div(n_rows, FSP_WG_THREADS);
      if (g > 65536) g = 65536;
      hipLaunchKernelGGL(spmv_zero_kernel<T>, dim3(static_cast<unsigned>(g)), dim3(FSP_WG_THREADS), 0, s,
                         static_cast<T*>(y_dev), n_rows);
      return check_launch("spmv_zero");
    });
  }
  FSP_DISPATCH_VALUE(value_type, T, {
    return spmv_launch<T>(index_type, indptr_type, perm_type, indptr_dev, indices_dev, data_dev, perm_dev, x_dev, y_dev,
                          x_len, nnz, plan, s);
  });
  return FSP_OK;
}

extern "C" int fsp_spmv_csr_parts(int32_t value_type, int32_t index_type, int32_t indptr_type,
                                  const void* indptr_dev, const void* indices_dev, const void* data_dev,
                                  const void* x_dev, void* y_dev, int64_t nnz, int64_t n_parts,
                                  const int64_t* parts_dev, int32_t lanes, int64_t row_len,
                                  int64_t indptr_base, void* stream) {
  if (nnz < 0 || n_parts < 0 || (lanes != 4 && lanes != 8 && lanes != 16)) {
    return fail(FSP_ERR_ARG, "fsp_spmv_csr_parts: bad arguments (lanes must be 4, 8 or 16)");
  }
  if (row_len < 0 || indptr_base < 0) {
    return fail(FSP_ERR_ARG, "fsp_spmv_csr_parts: row_len %lld / indptr_base %lld negative", (long long)row_len,
                (long long)indptr_base);
  }
  if (n_parts == 0) return FSP_OK;
  if (n_parts > 0x7fffffff || parts_dev == nullptr || indptr_dev == nullptr || y_dev == nullptr ||
      (nnz > 0 && (indices_dev == nullptr || data_dev == nullptr || x_dev == nullptr))) {
    return fail(FSP_ERR_ARG, "fsp_spmv_csr_parts: NULL array or too many parts");
  }
  const hipStream_t s = as_stream(stream);
  const int ll = lanes == 4 ? 2 : (lanes == 8 ? 3 : 4);
  FSP_DISPATCH_VALUE(value_type, T, {
    return spmv_parts_launch<T>(index_type, indptr_type, indptr_dev, indices_dev, data_dev, x_dev, y_dev, nnz, n_parts,
                                parts_dev, ll, row_len, indptr_base, s);
  });
  return FSP_OK;
}
