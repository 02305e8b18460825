// CSR SpMM kernels of bf16 values (spmm_kernels.hpp).
#include "spmm_kernels.hpp"

namespace fsp {
FSP_SPMM_INSTANCES(, __bf16)
}  // namespace fsp
