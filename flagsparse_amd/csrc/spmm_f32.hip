// CSR SpMM kernels of f32 values (spmm_kernels.hpp).
#include "spmm_kernels.hpp"

namespace fsp {
FSP_SPMM_INSTANCES(, float)
}  // namespace fsp
