// CSR SpMM kernels of f64 values (spmm_kernels.hpp).
#include "spmm_kernels.hpp"

namespace fsp {
FSP_SPMM_INSTANCES(, double)
}  // namespace fsp
