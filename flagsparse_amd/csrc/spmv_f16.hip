// CSR SpMV kernels of f16 values (spmv_kernels.hpp).
#include "spmv_kernels.hpp"

namespace fsp {
FSP_SPMV_INSTANCES(, _Float16)
}  // namespace fsp
