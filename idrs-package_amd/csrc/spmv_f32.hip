// SpMV kernels: float values, float vectors.
#include "spmv_kernels.hpp"

namespace idrs {
IDRS_SPMV_PAIR(float, float)
}  // namespace idrs
