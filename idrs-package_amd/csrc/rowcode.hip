// Row-coded products.
//
// What bounds a stencil product is the matrix: of the 72 bytes a row of a
// 7-point product in DIA storage moves (112 in sliced CRS), 48 (88) are values
// and indices.  Where the rows repeat -- constant coefficients, or a few
// materials -- they are all in a table of at most 256 distinct rows (27 for a
// 3-D stencil on a box), kept in LDS, and a row costs one byte.  The products
// are the same operations on the same values in the same order as the DIA and
// the sliced CRS kernels', so they give the same bits.  Plain product, us:
// 200^3 DIA 96 -> 39.5 (P^T y 148 -> 92, omega 102 -> 63), 128^3 sliced CRS
// 32.7 -> 13.3.  Then it is bound by its instructions (about 250 cycles of a
// CU per 64 rows), no longer by memory.  Measured and slower: one chunk of
// rows per block 52 us (the table is read again every 256 rows), 16 chunks 45,
// the next chunk's codes read ahead 41.5, uniform wavefronts through the
// scalar cache 50.
// A CRS matrix whose values differ from row to row but whose column offsets
// repeat (a stencil with variable coefficients) keeps its sliced values and
// codes the offsets: 8 bytes an entry instead of 12 (101x97x103, 7 points, IDR(8) +
// Chebyshev(8): 33.4 -> 25.4 ms).
#include "rowcode.hpp"

#include <algorithm>
#include <climits>

namespace idrs {
namespace {

constexpr int HSLOTS = 1024;   // hash slots, at most a quarter of them filled

// the stored entries of a row, in order
struct RowSrc {
    int nrows, ncols;
    // DIA
    int ndiag, ud;
    const int *offsets;
    // CRS
    const int *rp, *col;
    const double *val;   // null: offsets alone (every value 0)
    template <class F>
    __device__ inline void each(int row, F &&f) const {
        if (rp) {
            for (int p = rp[row]; p < rp[row + 1]; p++) f(col[p] - row, val ? val[p] : 0.0);
        } else {
            for (int d = 0; d < ndiag; d++) {
                const long c = (long)row + offsets[d];
                if (c >= 0 && c < ncols)
                    f(offsets[d], d == ud ? 1.0 : val[(long)(d - (d > ud ? 1 : 0)) * nrows + row]);
            }
        }
    }
    __device__ inline unsigned long long hash(int row) const {
        unsigned long long h = 0x9E3779B97F4A7C15ULL;
        each(row, [&](int o, double v) {
            h = (h ^ (unsigned long long)__double_as_longlong(v)) * 0xBF58476D1CE4E5B9ULL;
            h ^= h >> 29;
            h = (h ^ (unsigned)o) * 0x94D049BB133111EBULL;
            h ^= h >> 32;
        });
        return h ? h : 1;
    }
};

struct Work {
    unsigned long long key[HSLOTS];   // 0: free
    int rep[HSLOTS];                  // a row of this hash
    int id[HSLOTS];
    int count, bad;
};

// Puts the hashes of one row in each 'step' rows into the table; more than
// ROWCODE_MAX of them: bad, and later rows are skipped.  Ordinary loads see nearly every
// row's hash already there; a line read before its key was written only costs
// an atomic that finds the key.  A quarter-filled table has no probe sequence
// of PROBES, so one that long means an overfull table.
constexpr int PROBES = 64;
__global__ __launch_bounds__(256) void k_find_rows(RowSrc S, long rows, long step, Work *w) {
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < rows; q += (long)gridDim.x * blockDim.x) {
        if (w->bad) return;
        // not always the first of them: on a box of 64 rows a side every 64th row
        // is a boundary row, and a kind of row that the sample misses costs an
        // atomic per row in the next pass (search at 64^3 690 us, so 230)
        const int row = (int)min(q * step + (long)((unsigned long)q * 2654435761UL % (unsigned long)step), S.nrows - 1L);
        const unsigned long long h = S.hash(row);
        unsigned s = (unsigned)h % HSLOTS;
        int probe = 0;
        for (; probe < PROBES; probe++, s = (s + 1) % HSLOTS) {
            unsigned long long k = w->key[s];
            if (k == 0) {
                k = atomicCAS(&w->key[s], 0ULL, h);
                if (k == 0) {
                    w->rep[s] = row;
                    if (atomicAdd(&w->count, 1) >= ROWCODE_MAX) atomicExch(&w->bad, 1);
                    break;
                }
            }
            if (k == h) break;
        }
        if (probe == PROBES) atomicExch(&w->bad, 1);
    }
}

// numbers the distinct rows and writes the table; too many of them, or too
// large a table: bad
__global__ __launch_bounds__(256) void k_row_table(RowSrc S, Work *w, int width, RowEntry *ent, RowEntry *ent32,
                                                   int *len) {
    __shared__ int next, skip;
    if (threadIdx.x == 0) {
        next = 0;
        skip = w->bad || w->count > ROWCODE_MAX || w->count * width > ROWCODE_ENTRIES;
        if (skip) w->bad = 1;
    }
    __syncthreads();
    if (skip) return;
    for (int s = threadIdx.x; s < HSLOTS; s += blockDim.x)
        if (w->key[s]) {
            const int p = atomicAdd(&next, 1);
            w->id[s] = p;
            int k = 0;
            S.each(w->rep[s], [&](int o, double v) {
                ent[p * width + k] = {v, o, 0};
                ent32[p * width + k] = {(double)(float)v, o, 0};
                k++;
            });
            len[p] = k;
            for (; k < width; k++) ent[p * width + k] = ent32[p * width + k] = {0.0, 0, 0};
        }
}

// every row's code, checked entry by entry against the table (bad: a row
// differs from the one of its hash)
__global__ __launch_bounds__(256) void k_code_rows(RowSrc S, Work *w, int width, const RowEntry *ent, const int *len,
                                                   unsigned char *code) {
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < S.nrows; q += (long)gridDim.x * blockDim.x) {
        if (w->bad) return;
        const int row = (int)q;
        const unsigned long long h = S.hash(row);
        unsigned s = (unsigned)h % HSLOTS;
        int probe = 0;
        while (w->key[s] != h && probe < HSLOTS) {
            s = (s + 1) % HSLOTS;
            probe++;
        }
        const int p = probe < HSLOTS ? w->id[s] : 0;
        int k = 0;
        bool ok = probe < HSLOTS;
        S.each(row, [&](int o, double v) {
            ok = ok && k < len[p] && ent[p * width + k].off == o &&
                 __double_as_longlong(ent[p * width + k].val) == __double_as_longlong(v);
            k++;
        });
        if (!ok || k != len[p]) atomicExch(&w->bad, 1);
        code[row] = (unsigned char)p;
    }
}

__global__ void k_zero_work(Work *w) {
    for (int s = threadIdx.x; s < HSLOTS; s += blockDim.x) w->key[s] = 0;
    if (threadIdx.x == 0) w->count = w->bad = 0;
}

struct PatArgs {
    const unsigned char *code;
    const RowEntry *ent;
    const int *len;
    int npat, width;
    // sliced values (entry k of a row SELL_C k further on); null: the table's
    const double *sval;
    const long *sptr;
};

// the table in LDS: entries, then lengths
struct PatLds {
    const RowEntry *ent;
    const int *len;
};
__device__ inline PatLds stage_table(const PatArgs &p, unsigned char *dyn) {
    const int ne = p.npat * p.width;
    double2 *e = (double2 *)dyn;
    int *l = (int *)(e + ne);
    for (int i = threadIdx.x; i < ne; i += blockDim.x) e[i] = ((const double2 *)p.ent)[i];
    for (int i = threadIdx.x; i < p.npat; i += blockDim.x) l[i] = p.len[i];
    __syncthreads();
    return {(const RowEntry *)e, l};
}

// (K' x)(row): the chunks of sell_row with the entries out of the table.  W:
// the table's width when it is at most 8 (0: any).
// OWN: values from the sliced copy.
template <int W, bool OWN, bool KEEP>
__device__ inline double pat_row(const PatArgs &P, const PatLds &t, int pat, const double *__restrict__ x, int row) {
    double acc = 0.0;
    const int width = W > 0 ? W : P.width;
    const int len = t.len[pat];
    const RowEntry *e = t.ent + pat * width;
    constexpr int C = W > 0 ? W : 8;
    const double *v0 = nullptr;
    if constexpr (OWN) {
        // a wavefront's rows are one slice
        const int slice = __builtin_amdgcn_readfirstlane(row / SELL_C);
        v0 = P.sval + P.sptr[slice] + row % SELL_C;
    }
    for (int k0 = 0; k0 < width; k0 += C) {
        double vv[C], xx[C];
#pragma unroll
        for (int k = 0; k < C; k++) {
            const bool ok = k0 + k < len;
            const RowEntry q = e[ok ? k0 + k : 0];
            if constexpr (OWN) vv[k] = ok ? ldp<KEEP>(v0 + (long)SELL_C * (k0 + k)) : 0.0;
            else vv[k] = q.val;
            // entries beyond the row read x(row) and are not used
            xx[k] = x[ok ? row + q.off : row];
        }
#pragma unroll
        for (int k = 0; k < C; k++)
            if (k0 + k < len) acc = fmav(vv[k], xx[k], acc);
    }
    return acc;
}

template <int EPI, int NV, int W, bool OWN, bool KEEP>
__global__ __launch_bounds__(SPMV_THREADS) void k_spmv_pat(SpmvArgs<double, double> A, PatArgs P, EpiArgs<double> E,
                                                           const int *info) {
    if (info && *info >= 0) return;
    constexpr int PC = EPI == EPI_PDOT ? NV : 1;
    extern __shared__ __align__(16) unsigned char dyn[];
    __shared__ double s_red[NV * (SPMV_THREADS / WAVE)];
    const PatLds t = stage_table(P, dyn);
    double e[NV];
#pragma unroll
    for (int i = 0; i < NV; i++) e[i] = 0.0;
    const int lb = xcd_block(blockIdx.x, gridDim.x);
    const long n = A.nrows;
    const long nchunk = (n + SPMV_THREADS - 1) / SPMV_THREADS;
    const long c0 = nchunk * lb / gridDim.x, c1 = nchunk * (lb + 1) / gridDim.x;
    const double *zp = A.z;
    for (long c = c0; c < c1; c++) {
        const long row = c * SPMV_THREADS + threadIdx.x;
        if (row >= n) continue;
        const int pat = P.code[row];
        const double zq = zp ? zp[row] : 0.0;
        double pe[PC];
        if constexpr (EPI == EPI_PDOT) epi_load_row<double, PC, KEEP>(pe, E, E.P + row * E.prow);
        if constexpr (EPI == EPI_OMEGA) epi_load<double, EPI, PC, KEEP>(pe, E, row, 0, 1);
        const double acc = pat_row<W, OWN, KEEP>(P, t, pat, A.x, (int)row);
        const double yv = finish_value(A, row, acc, zq);
        A.y[row] = yv;
        epi_accum<double, EPI, NV, PC>(e, pe, E, yv, 0, 1);
    }
    epi_store<double, EPI, NV>(e, E, s_red);
}

// grid row y: column y of the block
template <int W>
__global__ __launch_bounds__(SPMV_THREADS) void k_spmv_pat_cols(SpmvArgs<double, double> A, PatArgs P,
                                                                ColArgs<double> C) {
    extern __shared__ __align__(16) unsigned char dyn[];
    const PatLds t = stage_table(P, dyn);
    const int j = blockIdx.y;
    const int lb = xcd_block(blockIdx.x, gridDim.x);
    const long n = A.nrows;
    const long nchunk = (n + SPMV_THREADS - 1) / SPMV_THREADS;
    const long c0 = nchunk * lb / gridDim.x, c1 = nchunk * (lb + 1) / gridDim.x;
    const double *x = C.x + j * C.ld, *z = C.z ? C.z + j * C.ld : nullptr;
    for (long c = c0; c < c1; c++) {
        const long row = c * SPMV_THREADS + threadIdx.x;
        if (row >= n) continue;
        const double zq = z ? z[row] : 0.0;
        const double acc = pat_row<W, false, false>(P, t, P.code[row], x, (int)row);
        C.y[j * C.ld + row] = finish_col(A, x, row, acc, z, zq, C.a[j]);
    }
}

size_t table_lds(const RowCode &rc) {
    return (size_t)rc.npat * rc.width * sizeof(RowEntry) + sizeof(int) * (size_t)rc.npat;
}

PatArgs pat_args(const RowCode &rc, bool f32) {
    return {rc.code, f32 ? rc.ent32 : rc.ent, rc.len, rc.npat, rc.width, nullptr, nullptr};
}

template <int EPI, int NV>
void launch_pat(const DevMatrix &K, const RowCode &rc, bool f32, const SpmvArgs<double, double> &A, EpiArgs<double> E,
                const int *info, hipStream_t st) {
    // the epilogue's partials keep the row slabs (and so the sums) of the
    // other kernels; without one a block takes at least four chunks, over
    // which it reads the table once
    int grid = spmv_grid(K);
    if (EPI == EPI_NONE)
        grid = std::min(grid, std::max(NUM_XCD * 256, ceil_div(K.nrows, 4 * SPMV_THREADS) / NUM_XCD * NUM_XCD));
    E.nparts = grid;
    PatArgs P = pat_args(rc, f32);
    const dim3 gd(grid), bd(SPMV_THREADS);
    if (!rc.values) {
        P.sval = A.val;
        P.sptr = A.sl_ptr;
    }
    // widths of the 1-, 2- and 3-D stencils, or any
#define PAT_KER(W, OWN, KEEP) \
    hipLaunchKernelGGL((k_spmv_pat<EPI, NV, W, OWN, KEEP>), gd, bd, table_lds(rc), st, A, P, E, info)
#define PAT_GO(W)                        \
    do {                                 \
        if (rc.values) {                 \
            if (A.keep) PAT_KER(W, false, true);  \
            else PAT_KER(W, false, false);        \
        } else {                         \
            if (A.keep) PAT_KER(W, true, true);   \
            else PAT_KER(W, true, false);         \
        }                                \
    } while (0)
    switch (rc.width) {
    case 3: PAT_GO(3); break;
    case 5: PAT_GO(5); break;
    case 7: PAT_GO(7); break;
    default: PAT_GO(0); break;
    }
#undef PAT_GO
#undef PAT_KER
    LAUNCH_CHECK();
}

}  // namespace

RowCode::~RowCode() { pool_free(mem, bytes); }

// Zeroing, the sample, all rows, the table and the codes are enqueued at once
// and waited for once; the first that finds too many distinct rows ends the
// rest at their start.  Buffers come from the pool: a program that builds a
// matrix per solve pays no allocation for it.
std::shared_ptr<RowCode> make_rowcode(const Operator &op, bool values, hipStream_t st) {
    const DevMatrix &K = *op.K;
    if (K.kind == ValKind::Complex || (values && op.values_complex())) return nullptr;
    if (!values && K.fmt != DevFmt::CRS) return nullptr;
    if (K.part || K.nrows != K.ncols || K.nrows < ROWCODE_MIN_ROWS) return nullptr;
    RowSrc S{};
    S.nrows = K.nrows;
    S.ncols = K.ncols;
    S.ud = INT_MAX;
    S.val = values ? (const double *)op.values() : nullptr;
    int width;
    if (K.fmt == DevFmt::CRS) {
        width = K.max_row;
        S.rp = K.row_ptr;
        S.col = K.col;
    } else {
        width = K.ndiag;
        S.ndiag = K.ndiag;
        S.offsets = K.offsets;
        if (op.sval && op.unit_diag >= 0) S.ud = op.unit_diag;
    }
    if (width < 1 || width > ROWCODE_WIDTH) return nullptr;
    auto rc = std::make_shared<RowCode>();
    const size_t ent_bytes = sizeof(RowEntry) * ROWCODE_ENTRIES, len_bytes = sizeof(int) * ROWCODE_MAX;
    rc->bytes = 2 * ent_bytes + len_bytes + sizeof(Work) + (size_t)K.nrows;
    rc->mem = pool_try_alloc(rc->bytes);
    if (!rc->mem) return nullptr;   // optional: without memory for it the products stay uncoded
    char *p = (char *)rc->mem;
    rc->ent = (RowEntry *)p;
    rc->ent32 = (RowEntry *)(p += ent_bytes);
    Work *w = (Work *)(p += ent_bytes);
    rc->len = (int *)(p += sizeof(Work));
    rc->code = (unsigned char *)(p + len_bytes);
    rc->values = values;
    rc->width = width;
    const int g = vec_grid(K.nrows);
    hipLaunchKernelGGL(k_zero_work, dim3(1), dim3(256), 0, st, w);
    LAUNCH_CHECK();
    // a sample of 4096 rows turns away most matrices that do not repeat
    const long rows = K.nrows, step = std::max<long>(1, rows / 4096);
    hipLaunchKernelGGL(k_find_rows, dim3(16), dim3(256), 0, st, S, (rows + step - 1) / step, step, w);
    LAUNCH_CHECK();
    hipLaunchKernelGGL(k_find_rows, dim3(g), dim3(256), 0, st, S, rows, 1L, w);
    LAUNCH_CHECK();
    hipLaunchKernelGGL(k_row_table, dim3(1), dim3(256), 0, st, S, w, width, rc->ent, rc->ent32, rc->len);
    LAUNCH_CHECK();
    hipLaunchKernelGGL(k_code_rows, dim3(g), dim3(256), 0, st, S, w, width, rc->ent, rc->len, rc->code);
    LAUNCH_CHECK();
    int found[2];   // count, bad
    HIP_TRY(hipMemcpyAsync(found, &w->count, sizeof found, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    if (found[1]) return nullptr;
    rc->npat = found[0];
    return rc;
}

void rowcode_spmv(const DevMatrix &K, const RowCode &rc, bool f32, const SpmvArgs<double, double> &A,
                  const EpiArgs<double> &E, int epi, const int *info, hipStream_t st) {
    switch (epi) {
    case EPI_NONE: launch_pat<EPI_NONE, 1>(K, rc, f32, A, E, info, st); break;
    case EPI_NORM: launch_pat<EPI_NORM, 1>(K, rc, f32, A, E, info, st); break;
    case EPI_OMEGA: launch_pat<EPI_OMEGA, 3>(K, rc, f32, A, E, info, st); break;
    case EPI_PDOT:
        if (E.prow < 1 || E.prow > 16 || !E.P) throw std::invalid_argument("P^T y epilogue needs 1..16 rows of P");
        if (E.prow <= 1) launch_pat<EPI_PDOT, 1>(K, rc, f32, A, E, info, st);
        else if (E.prow <= 2) launch_pat<EPI_PDOT, 2>(K, rc, f32, A, E, info, st);
        else if (E.prow <= 4) launch_pat<EPI_PDOT, 4>(K, rc, f32, A, E, info, st);
        else if (E.prow <= 8) launch_pat<EPI_PDOT, 8>(K, rc, f32, A, E, info, st);
        else launch_pat<EPI_PDOT, 16>(K, rc, f32, A, E, info, st);
        break;
    default: throw std::invalid_argument("bad epilogue");
    }
}

void rowcode_cols(const DevMatrix &K, const RowCode &rc, bool f32, const SpmvArgs<double, double> &A,
                  const ColArgs<double> &C, hipStream_t st) {
    const int grid = std::max(1, std::min(spmv_grid(K), ceil_div(K.nrows, 4 * SPMV_THREADS)));
    const dim3 gd(grid, C.nc), bd(SPMV_THREADS);
    const PatArgs P = pat_args(rc, f32);
    switch (rc.width) {
    case 3: hipLaunchKernelGGL(k_spmv_pat_cols<3>, gd, bd, table_lds(rc), st, A, P, C); break;
    case 5: hipLaunchKernelGGL(k_spmv_pat_cols<5>, gd, bd, table_lds(rc), st, A, P, C); break;
    case 7: hipLaunchKernelGGL(k_spmv_pat_cols<7>, gd, bd, table_lds(rc), st, A, P, C); break;
    default: hipLaunchKernelGGL(k_spmv_pat_cols<0>, gd, bd, table_lds(rc), st, A, P, C); break;
    }
    LAUNCH_CHECK();
}

}  // namespace idrs
