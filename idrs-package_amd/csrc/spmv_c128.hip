// SpMV kernels: c128 values, c128 vectors.
#include "spmv_kernels.hpp"

namespace idrs {
IDRS_SPMV_PAIR(c128, c128)
}  // namespace idrs
