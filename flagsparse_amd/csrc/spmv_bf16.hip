// CSR SpMV kernels of bf16 values (spmv_kernels.hpp).
#include "spmv_kernels.hpp"

namespace fsp {
FSP_SPMV_INSTANCES(, __bf16)
}  // namespace fsp
