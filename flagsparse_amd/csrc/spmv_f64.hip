// CSR SpMV kernels of f64 values (spmv_kernels.hpp).
#include "spmv_kernels.hpp"

namespace fsp {
FSP_SPMV_INSTANCES(, double)
}  // namespace fsp
