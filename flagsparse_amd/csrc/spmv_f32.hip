// CSR SpMV kernels of f32 values (spmv_kernels.hpp).
#include "spmv_kernels.hpp"

namespace fsp {
FSP_SPMV_INSTANCES(, float)
}  // namespace fsp
