// SpMV kernels: double values, double vectors.
#include "spmv_kernels.hpp"

namespace idrs {
IDRS_SPMV_PAIR(double, double)
}  // namespace idrs
