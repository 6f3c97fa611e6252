// SpMV kernels: float values, c64 vectors.
#include "spmv_kernels.hpp"

namespace idrs {
IDRS_SPMV_PAIR(float, c64)
}  // namespace idrs
