// SpMV kernels: float values, double vectors.
#include "spmv_kernels.hpp"

namespace idrs {
IDRS_SPMV_PAIR(float, double)
}  // namespace idrs
