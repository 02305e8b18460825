// CSR SpMM kernels of f16 values (spmm_kernels.hpp).
#include "spmm_kernels.hpp"

namespace fsp {
FSP_SPMM_INSTANCES(, _Float16)
}  // namespace fsp
