// SpMV kernels: double values, c128 vectors.
#include "spmv_kernels.hpp"

namespace idrs {
IDRS_SPMV_PAIR(double, c128)
}  // namespace idrs
