// Launches of the SpMV kernels for one value/vector type pair; the
// definitions are in spmv_kernels.hpp, instantiated per pair in spmv_*.hip.
#pragma once

#include "matrix.hpp"
#include "spmv_epi.hpp"

namespace idrs {

// one product with the given epilogue
template <class VT, class T>
void dispatch_epi(const DevMatrix &K, const SpmvArgs<VT, T> &A, const EpiArgs<T> &E, int epi, const int *info,
                  hipStream_t st);
// one product over the tiles of a batch's partition
template <class VT, class T>
void dispatch_epi_tiles(const DevMatrix &K, const SpmvArgs<VT, T> &A, const EpiArgs<T> &E, int epi,
                        const TileCtx &tc, hipStream_t st);
// one block product of at most SPMV_COLS columns; false when K's layout has
// no block kernel (generic DIA, CRS with lanes per row)
template <class VT, class T>
bool launch_cols(const DevMatrix &K, const SpmvArgs<VT, T> &A, const ColArgs<T> &C, hipStream_t st);

}  // namespace idrs
