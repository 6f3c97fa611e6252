// Row-coded matrices: a matrix whose rows repeat (a stencil with constant or
// piecewise constant coefficients) as one byte per row and a table of its
// distinct rows.
#pragma once

#include "matrix.hpp"
#include "spmv_epi.hpp"

namespace idrs {

constexpr int ROWCODE_MAX = 256;       // distinct rows (one byte)
constexpr int ROWCODE_WIDTH = 32;      // entries of a row
constexpr int ROWCODE_ENTRIES = 2048;  // entries of the table (32 KB of LDS)
constexpr int ROWCODE_MIN_ROWS = 1 << 15;

// one entry of a distinct row: value and column - row
struct alignas(16) RowEntry {
    double val;
    int off, pad;
};

// Distinct row p: len[p] entries ent[p * width + k], in stored order.  ent32:
// the values rounded to float (the FP32-value products), held as double.
// Without values (ent holds the offsets alone) the code stands for the column
// indices of a sliced CRS matrix, whose values are read as before.
struct RowCode {
    int npat = 0, width = 0;
    bool values = true;
    unsigned char *code = nullptr;   // nrows
    RowEntry *ent = nullptr, *ent32 = nullptr;
    int *len = nullptr;
    void *mem = nullptr;   // holds them all, from the pool
    size_t bytes = 0;
    RowCode() = default;
    RowCode(const RowCode &) = delete;
    RowCode &operator=(const RowCode &) = delete;
    ~RowCode();
};

// The row code of K with the values of op (K's own without diagonal scaling),
// or of K's column offsets alone; null when K is not of a coded form or has
// more than ROWCODE_MAX distinct rows, or without memory for it.  Two passes
// over the matrix and one wait.
std::shared_ptr<RowCode> make_rowcode(const Operator &op, bool values, hipStream_t st);

// The code that the products of op use, or null: built by op_prepare_solve.  One of
// offsets alone only with 'offsets' (block products and FP32 values have no
// kernel for it).
const RowCode *op_rowcode(const Operator &op, bool offsets);

// y = xs (K' x - seed x/sdiag) + a z with the epilogue, as dispatch_epi
void rowcode_spmv(const DevMatrix &K, const RowCode &rc, bool f32, const SpmvArgs<double, double> &A,
                  const EpiArgs<double> &E, int epi, const int *info, hipStream_t st);
// the columns of a block product, as launch_cols
void rowcode_cols(const DevMatrix &K, const RowCode &rc, bool f32, const SpmvArgs<double, double> &A,
                  const ColArgs<double> &C, hipStream_t st);

}  // namespace idrs
