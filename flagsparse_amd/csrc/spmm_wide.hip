// CSR SpMM kernels whose values are wider than the dense operands
// (spmm_kernels.hpp).
#include "spmm_kernels.hpp"

namespace fsp {
FSP_SPMM_WIDE_INSTANCE(, float, double)
FSP_SPMM_WIDE_INSTANCE(, __bf16, float)
FSP_SPMM_WIDE_INSTANCE(, _Float16, float)
}  // namespace fsp
