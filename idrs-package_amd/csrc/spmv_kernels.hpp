// The SpMV kernels (CRS lanes per row, DIA, sliced CRS; single, block and
// batched products) and their launches, as templates over the value type VT
// and the vector type T.  Each spmv_<pair>.hip instantiates one pair, so the
// pairs compile in parallel.
#pragma once

#include "matrix.hpp"
#include "spmv_epi.hpp"
#include "spmv_launch.hpp"

#include <algorithm>
#include <climits>
#include <stdexcept>

namespace idrs {

// the launch under the cache policy A.keep
#define SPMV_TARGS(...) __VA_ARGS__
#define SPMV_LAUNCH(KER, TARGS, ...)                                                                \
    do {                                                                                            \
        if (A.keep) hipLaunchKernelGGL((KER<SPMV_TARGS TARGS, true>), gd, bd, 0, st, __VA_ARGS__);  \
        else hipLaunchKernelGGL((KER<SPMV_TARGS TARGS, false>), gd, bd, 0, st, __VA_ARGS__);        \
    } while (0)

// CRS: a group of G lanes per row (G >= the typical row length), so a
// wavefront covers 64/G consecutive rows whose entries are one contiguous,
// coalesced stretch of values and column indices.  The block's row pointers
// are staged in LDS once per chunk of rows, which leaves two dependent
// memory latencies per row (column index, then x).  Each group keeps U rows
// in flight: all their first-pass loads, and the P components of the P^T y
// epilogue, are issued before any is used; rows longer than G finish in a
// strided remainder loop.  The group's partial sums are combined
// by a butterfly inside the group, so every lane of the group holds y(row);
// for P^T y lane g takes the P components g, g+G, ... of its rows.
constexpr int CRS_CHUNK = 2048;   // rows whose row pointers sit in LDS at once

template <class VT, class T, int EPI, int NV, int G, bool KEEP>
__global__ __launch_bounds__(SPMV_THREADS) void k_spmv_crs(SpmvArgs<VT, T> A, EpiArgs<T> E, const int *info) {
    if (info && *info >= 0) return;
    constexpr int GPB = SPMV_THREADS / G;
    constexpr int U = 4;
    // epilogue operands per row and lane: P components (PDOT), r (OMEGA)
    constexpr int PC = EPI == EPI_PDOT ? (NV + G - 1) / G : 1;
    __shared__ int s_rp[CRS_CHUNK + 1];
    __shared__ T s_red[NV * (SPMV_THREADS / WAVE)];
    T e[EPI == EPI_PDOT ? PC : NV];
#pragma unroll
    for (int i = 0; i < (EPI == EPI_PDOT ? PC : NV); i++) e[i] = T(0);
    const int g = threadIdx.x % G, grp = threadIdx.x / G;
    const int lb = xcd_block(blockIdx.x, gridDim.x);
    const long n = A.nrows;
    const long r0 = n * lb / gridDim.x, r1 = n * (lb + 1) / gridDim.x;
    const T *__restrict__ x = A.x;
    const VT *__restrict__ val = A.val;
    const int *__restrict__ col = A.col;
    for (long c0 = r0; c0 < r1; c0 += CRS_CHUNK) {
        const long c1 = min(c0 + (long)CRS_CHUNK, r1);
        __syncthreads();
        for (long q = c0 + threadIdx.x; q <= c1; q += SPMV_THREADS) s_rp[q - c0] = A.rp[q];
        __syncthreads();
        for (long base = c0; base < c1; base += (long)GPB * U) {
            long row[U], rq[U];
            int a[U], b[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                row[u] = base + grp + (long)u * GPB;
                const bool in = row[u] < c1;
                rq[u] = in ? row[u] : c0;
                a[u] = in ? s_rp[row[u] - c0] : 0;
                b[u] = in ? s_rp[row[u] - c0 + 1] : 0;
            }
            VT vv[U];
            int cc[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int j = a[u] + g;
                const bool ok = j < b[u];
                vv[u] = ok ? ldp<KEEP>(&val[j]) : VT(0);
                cc[u] = ok ? ldp<KEEP>(&col[j]) : -1;
            }
            // P components of the rows (P^T y) are issued with the matrix
            // loads; z and r are loaded at the finish, where the register
            // budget of the U rows in flight is lower
            T pe[U][PC];
            if constexpr (EPI == EPI_PDOT) {
#pragma unroll
                for (int u = 0; u < U; u++) epi_load<T, EPI, PC, KEEP>(pe[u], E, rq[u], g, G);
            }
            T acc[U];
#pragma unroll
            for (int u = 0; u < U; u++) acc[u] = cc[u] >= 0 ? mulv(vv[u], x[cc[u]]) : T(0);
#pragma unroll
            for (int u = 0; u < U; u++)
                for (int j = a[u] + g + G; j < b[u]; j += G) acc[u] = fmav(ldp<KEEP>(&val[j]), x[ldp<KEEP>(&col[j])], acc[u]);
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int m = G / 2; m >= 1; m >>= 1) acc[u] = acc[u] + shfl_xor(acc[u], m);
#pragma unroll
            for (int u = 0; u < U; u++)
                if (row[u] < c1) {
                    const T zq = A.z ? A.z[row[u]] : T(0);
                    const T yv = finish_value(A, row[u], acc[u], zq);
                    if (g == 0) A.y[row[u]] = yv;
                    if constexpr (EPI == EPI_PDOT) {
                        epi_accum<T, EPI, PC, PC>(e, pe[u], E, yv, g, G);
                    } else if (g == 0) {
                        epi_load<T, EPI, PC, KEEP>(pe[u], E, row[u], 0, 1);
                        epi_accum<T, EPI, NV, PC>(e, pe[u], E, yv, 0, 1);
                    }
                }
        }
    }
    if constexpr (EPI == EPI_PDOT) epi_store_group<T, NV, G, PC>(e, E, s_red);
    else epi_store<T, EPI, NV>(e, E, s_red);
}

// DIA: one thread per row over a contiguous row range; every diagonal is a
// coalesced stream.  ND > 0 unrolls a known diagonal count.
template <class VT, class T, int EPI, int NV, int ND, bool KEEP>
__global__ __launch_bounds__(SPMV_THREADS) void k_spmv_dia(SpmvArgs<VT, T> A, EpiArgs<T> E, const int *info) {
    if (info && *info >= 0) return;
    constexpr int PC = EPI == EPI_PDOT ? NV : 1;
    static_assert(ND <= 8, "known diagonal counts take their offsets by value");
    __shared__ int s_off[ND > 0 ? 1 : MAX_DIAG];
    __shared__ T s_red[NV * (SPMV_THREADS / WAVE)];
    const int ndiag = ND > 0 ? ND : A.ndiag;
    if constexpr (ND == 0) {
        for (int d = threadIdx.x; d < ndiag; d += SPMV_THREADS) s_off[d] = A.offsets[d];
        __syncthreads();
    }
    T e[NV];
#pragma unroll
    for (int i = 0; i < NV; i++) e[i] = T(0);
    const int lb = xcd_block(blockIdx.x, gridDim.x);
    const long n = A.nrows, ncols = A.ncols;
    const long nchunk = (n + SPMV_THREADS - 1) / SPMV_THREADS;
    const long c0 = nchunk * lb / gridDim.x, c1 = nchunk * (lb + 1) / gridDim.x;
    const T *__restrict__ x = A.x;
    const VT *__restrict__ val = A.val;
    const int ud = A.ud;
    const T *zp = A.z;   // Horner vector; products without one read nothing here
    // diagonal d is stored at d - (d > ud); the implicit unit diagonal
    // (d == ud) enters as fmav(1, x, acc), the same operation as a stored
    // 1.0.  With a known diagonal count the offsets and value streams are
    // wave-uniform (scalar registers), rows index them in 32 bits.
    int offr[ND > 0 ? ND : 1];
    const VT *vb[ND > 0 ? ND : 1];
    if constexpr (ND > 0) {
#pragma unroll
        for (int d = 0; d < ND; d++) {
            offr[d] = A.off8[d];
            vb[d] = val + (size_t)(d - (d > ud ? 1 : 0)) * (size_t)n;
        }
    }
    for (long c = c0; c < c1; c++) {
        const long row = c * SPMV_THREADS + threadIdx.x;
        if (row >= n) continue;
        T acc = T(0);
        T zq;
        T pe[PC];
        if constexpr (ND > 0) {
            // 32-bit byte offsets from the wave-uniform bases (one offset
            // register for every stream of the row instead of a 64-bit
            // address each); the launcher takes this path only while the
            // offsets fit: n * 8 * max(1, prow) < 2^32
            const unsigned bo = (unsigned)row * (unsigned)sizeof(T);
            const unsigned vbo = (unsigned)row * (unsigned)sizeof(VT);
            zq = zp ? *(const T *)((const char *)zp + bo) : T(0);
            if constexpr (EPI == EPI_PDOT) {
                const T *p = (const T *)((const char *)E.P + (unsigned)row * (unsigned)(E.prow * sizeof(T)));
                epi_load_row<T, PC, KEEP>(pe, E, p);
            }
            VT vv[ND];
            T xx[ND];
#pragma unroll
            for (int d = 0; d < ND; d++) {
                // every load in bounds without a branch: the stored value
                // of row `row` exists on each diagonal, and a column outside
                // the matrix reads x(row) instead (the launcher takes this
                // path only for nrows <= ncols); both enter as zero
                const long cc = row + offr[d];
                const bool ok = cc >= 0 && cc < ncols;
                if constexpr (std::is_same<VT, T>::value) {
                    const unsigned xo = (unsigned)(ok ? cc : row) * (unsigned)sizeof(T);
                    const VT v = d == ud ? VT(1) : ldp<KEEP>((const VT *)((const char *)vb[d] + vbo));
                    const T xv = *(const T *)((const char *)x + xo);
                    vv[d] = ok ? v : VT(0);
                    xx[d] = ok ? xv : T(0);
                } else {
                    // values of another type: loads under the column test, so
                    // that the conversion is not placed next to each load
                    // (which would wait for it before the next is issued)
                    vv[d] = !ok ? VT(0) : (d == ud ? VT(1) : ldp<KEEP>((const VT *)((const char *)vb[d] + vbo)));
                    xx[d] = ok ? *(const T *)((const char *)x + (unsigned)cc * (unsigned)sizeof(T)) : T(0);
                }
            }
#pragma unroll
            for (int d = 0; d < ND; d++) acc = fmav(vv[d], xx[d], acc);
            const T yv = finish_value(A, row, acc, zq);
            *(T *)((char *)A.y + bo) = yv;
            if constexpr (EPI != EPI_PDOT) epi_load<T, EPI, PC, KEEP>(pe, E, row, 0, 1);
            epi_accum<T, EPI, NV, PC>(e, pe, E, yv, 0, 1);
            continue;
        } else {
            zq = zp ? zp[row] : T(0);
            if constexpr (EPI == EPI_PDOT) epi_load<T, EPI, PC, KEEP>(pe, E, row, 0, 1);
            for (int d = 0; d < ndiag; d++) {
                const long cc = row + s_off[d];
                const long sd = d - (d > ud ? 1 : 0);
                if (cc >= 0 && cc < ncols) acc = fmav(d == ud ? VT(1) : ldp<KEEP>(&val[sd * n + row]), x[cc], acc);
            }
        }
        const T yv = finish_value(A, row, acc, zq);
        A.y[row] = yv;
        if constexpr (EPI != EPI_PDOT) epi_load<T, EPI, PC, KEEP>(pe, E, row, 0, 1);
        epi_accum<T, EPI, NV, PC>(e, pe, E, yv, 0, 1);
    }
    epi_store<T, EPI, NV>(e, E, s_red);
}

// Sliced copy of a CRS matrix (group 1): one thread per row.  Entry k of the
// row is at p0 + SELL_C k, so each load instruction of a wavefront reads
// SELL_C consecutive values (or column indices).  Entries go in chunks of 8:
// all value and index loads of a chunk, then all its x gathers; the row sum
// runs over k in CRS order (the reference's sequential row sum).
template <bool KEEP, class VT, class T>
__device__ inline T sell_row(const SpmvArgs<VT, T> &A, long row, long p0, int w) {
    const VT *__restrict__ val = A.val;
    const int *__restrict__ scol = A.sl_col;
    const T *__restrict__ x = A.x;
    const int len = A.rp[row + 1] - A.rp[row];
    T acc = T(0);
    if constexpr (std::is_same<VT, float>::value) {
        // FP32 copy: one 8-byte load brings an entry's value and column
        // (4-byte loads of each would double the load instructions, which
        // bound this product); the same chunks and sum order as below
        if (A.pair32) {
            const unsigned long long *pr = (const unsigned long long *)val;
            for (int k0 = 0; k0 < w; k0 += 8) {
                float vv[8];
                int cc[8];
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    const bool ok = k0 + k < len;
                    const unsigned long long e = ok ? ldp<KEEP>(&pr[p0 + (long)SELL_C * (k0 + k)]) : 0ull;
                    vv[k] = __uint_as_float((unsigned)(e & 0xffffffffull));
                    cc[k] = (int)(e >> 32);
                }
                T xx[8];
#pragma unroll
                for (int k = 0; k < 8; k++) xx[k] = k0 + k < len ? x[cc[k]] : T(0);
#pragma unroll
                for (int k = 0; k < 8; k++)
                    if (k0 + k < len) acc = fmav(vv[k], xx[k], acc);
            }
            return acc;
        }
    }
    // chunks of 8 entries (w, the slice width, is wave-uniform): all value
    // and index loads of a chunk, then its x gathers, then the in-order sum
    for (int k0 = 0; k0 < w; k0 += 8) {
        VT vv[8];
        int cc[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const bool ok = k0 + k < len;
            vv[k] = ok ? ldp<KEEP>(&val[p0 + (long)SELL_C * (k0 + k)]) : VT(0);
            cc[k] = ok ? ldp<KEEP>(&scol[p0 + (long)SELL_C * (k0 + k)]) : 0;
        }
        T xx[8];
#pragma unroll
        for (int k = 0; k < 8; k++) xx[k] = k0 + k < len ? x[cc[k]] : T(0);
#pragma unroll
        for (int k = 0; k < 8; k++)
            if (k0 + k < len) acc = fmav(vv[k], xx[k], acc);
    }
    return acc;
}

template <class VT, class T, int EPI, int NV, bool KEEP>
__global__ __launch_bounds__(SPMV_THREADS) void k_spmv_sell(SpmvArgs<VT, T> A, EpiArgs<T> E, const int *info) {
    static_assert(SPMV_THREADS % SELL_C == 0 && SELL_C == WAVE, "one slice per wavefront");
    if (info && *info >= 0) return;
    constexpr int PC = EPI == EPI_PDOT ? NV : 1;
    __shared__ T s_red[NV * (SPMV_THREADS / WAVE)];
    T e[NV];
#pragma unroll
    for (int i = 0; i < NV; i++) e[i] = T(0);
    const int lb = xcd_block(blockIdx.x, gridDim.x);
    const long n = A.nrows;
    const long nchunk = (n + SPMV_THREADS - 1) / SPMV_THREADS;
    const long c0 = nchunk * lb / gridDim.x, c1 = nchunk * (lb + 1) / gridDim.x;
    const T *zp = A.z;   // Horner vector; products without one read nothing here
    const int wv = threadIdx.x / WAVE;
    for (long c = c0; c < c1; c++) {
        // the wavefront's slice (uniform: chunks start at multiples of SELL_C)
        const int slice = __builtin_amdgcn_readfirstlane((int)(c * (SPMV_THREADS / SELL_C) + wv));
        const long row = c * SPMV_THREADS + threadIdx.x;
        if (row >= n) continue;
        const long sp = A.sl_ptr[slice];
        const int w = (int)((A.sl_ptr[slice + 1] - sp) / SELL_C);
        const T zq = zp ? zp[row] : T(0);
        T pe[PC];
        if constexpr (EPI == EPI_PDOT) epi_load<T, EPI, PC, KEEP>(pe, E, row, 0, 1);
        const T acc = sell_row<KEEP>(A, row, sp + (row % SELL_C), w);
        const T yv = finish_value(A, row, acc, zq);
        A.y[row] = yv;
        if constexpr (EPI != EPI_PDOT) epi_load<T, EPI, PC, KEEP>(pe, E, row, 0, 1);
        epi_accum<T, EPI, NV, PC>(e, pe, E, yv, 0, 1);
    }
    epi_store<T, EPI, NV>(e, E, s_red);
}

template <class VT, class T, int EPI, int NV>
static void launch_spmv(const DevMatrix &K, const SpmvArgs<VT, T> &A, EpiArgs<T> E, const int *info,
                        hipStream_t st) {
    const int grid = spmv_grid(K);
    E.nparts = grid;
    dim3 gd(grid), bd(SPMV_THREADS);
    if (K.fmt == DevFmt::CRS && A.sl_ptr) {
        SPMV_LAUNCH(k_spmv_sell, (VT, T, EPI, NV), A, E, info);
    } else if (K.fmt == DevFmt::CRS) {
        // group 1 without sliced values (e.g. the FP32 copy): 2 lanes per row
        switch (K.group) {
        case 1:
        case 2: SPMV_LAUNCH(k_spmv_crs, (VT, T, EPI, NV, 2), A, E, info); break;
        case 4: SPMV_LAUNCH(k_spmv_crs, (VT, T, EPI, NV, 4), A, E, info); break;
        case 8: SPMV_LAUNCH(k_spmv_crs, (VT, T, EPI, NV, 8), A, E, info); break;
        case 16: SPMV_LAUNCH(k_spmv_crs, (VT, T, EPI, NV, 16), A, E, info); break;
        case 32: SPMV_LAUNCH(k_spmv_crs, (VT, T, EPI, NV, 32), A, E, info); break;
        default: SPMV_LAUNCH(k_spmv_crs, (VT, T, EPI, NV, 64), A, E, info); break;
        }
    } else {
        // the unrolled kernels address rows by 32-bit byte offsets
        const unsigned long long rowb = sizeof(T) * (EPI == EPI_PDOT ? (unsigned long long)std::max(1, E.prow) : 1ull);
        const int nd =
            K.nrows <= K.ncols && (unsigned long long)K.ncols * rowb < (1ull << 32) ? K.ndiag : 0;
        switch (nd) {
        case 3: SPMV_LAUNCH(k_spmv_dia, (VT, T, EPI, NV, 3), A, E, info); break;
        case 5: SPMV_LAUNCH(k_spmv_dia, (VT, T, EPI, NV, 5), A, E, info); break;
        case 7: SPMV_LAUNCH(k_spmv_dia, (VT, T, EPI, NV, 7), A, E, info); break;
        default: SPMV_LAUNCH(k_spmv_dia, (VT, T, EPI, NV, 0), A, E, info); break;
        }
    }
    LAUNCH_CHECK();
}

template <class VT, class T>
void dispatch_epi(const DevMatrix &K, const SpmvArgs<VT, T> &A, const EpiArgs<T> &E, int epi,
                         const int *info, hipStream_t st) {
    switch (epi) {
    case EPI_NONE: launch_spmv<VT, T, EPI_NONE, 1>(K, A, E, info, st); break;
    case EPI_NORM: launch_spmv<VT, T, EPI_NORM, 1>(K, A, E, info, st); break;
    case EPI_OMEGA: launch_spmv<VT, T, EPI_OMEGA, 3>(K, A, E, info, st); break;
    case EPI_PDOT:
        if (E.prow < 1 || E.prow > 16 || !E.P) throw std::invalid_argument("P^T y epilogue needs 1..16 rows of P");
        if (E.prow <= 1) launch_spmv<VT, T, EPI_PDOT, 1>(K, A, E, info, st);
        else if (E.prow <= 2) launch_spmv<VT, T, EPI_PDOT, 2>(K, A, E, info, st);
        else if (E.prow <= 4) launch_spmv<VT, T, EPI_PDOT, 4>(K, A, E, info, st);
        else if (E.prow <= 8) launch_spmv<VT, T, EPI_PDOT, 8>(K, A, E, info, st);
        else launch_spmv<VT, T, EPI_PDOT, 16>(K, A, E, info, st);
        break;
    default: throw std::invalid_argument("bad epilogue");
    }
}

// ---------------------------------------------------------------------------
// block products y_j = xs (K' x_j - seed x_j / sdiag) + a_j z_j over the
// columns of a block (the multishift solvers' per-shift products and
// scale-backs).  A row's entries are loaded once for all columns of the
// launch; each column's row sum and finish are those of k_spmv_dia /
// k_spmv_sell, so column j equals the one-column product of x_j bit for bit.
// ---------------------------------------------------------------------------
template <class VT, class T, int ND, bool KEEP>
__global__ __launch_bounds__(SPMV_THREADS) void k_spmv_dia_cols(SpmvArgs<VT, T> A, ColArgs<T> C) {
    static_assert(ND > 0 && ND <= 8, "known diagonal counts only");
    const int lb = xcd_block(blockIdx.x, gridDim.x);
    const long n = A.nrows, ncols = A.ncols;
    const long nchunk = (n + SPMV_THREADS - 1) / SPMV_THREADS;
    const long c0 = nchunk * lb / gridDim.x, c1 = nchunk * (lb + 1) / gridDim.x;
    const int ud = A.ud;
    for (long c = c0; c < c1; c++) {
        const long row = c * SPMV_THREADS + threadIdx.x;
        if (row >= n) continue;
        VT vv[ND];
        bool ok[ND];
#pragma unroll
        for (int d = 0; d < ND; d++) {
            const long cc = row + A.off8[d];
            ok[d] = cc >= 0 && cc < ncols;
            const long sd = d - (d > ud ? 1 : 0);
            vv[d] = !ok[d] ? VT(0) : (d == ud ? VT(1) : ldp<KEEP>(A.val + sd * n + row));
        }
#pragma unroll
        for (int j = 0; j < SPMV_COLS; j++) {
            if (j < C.nc) {
                const T *xj = C.x + j * C.ld;
                T xx[ND];
#pragma unroll
                for (int d = 0; d < ND; d++) xx[d] = ok[d] ? xj[row + A.off8[d]] : T(0);
                T acc = T(0);
#pragma unroll
                for (int d = 0; d < ND; d++) acc = fmav(vv[d], xx[d], acc);
                const T *zj = C.z ? C.z + j * C.ld : nullptr;
                const T zq = zj ? zj[row] : T(0);
                C.y[j * C.ld + row] = finish_col(A, xj, row, acc, zj, zq, C.a[j]);
            }
        }
    }
}

template <class VT, class T, bool KEEP>
__global__ __launch_bounds__(SPMV_THREADS) void k_spmv_sell_cols(SpmvArgs<VT, T> A, ColArgs<T> C) {
    const int lb = xcd_block(blockIdx.x, gridDim.x);
    const long n = A.nrows;
    const long nchunk = (n + SPMV_THREADS - 1) / SPMV_THREADS;
    const long c0 = nchunk * lb / gridDim.x, c1 = nchunk * (lb + 1) / gridDim.x;
    const int wv = threadIdx.x / WAVE;
    const VT *__restrict__ val = A.val;
    const int *__restrict__ scol = A.sl_col;
    for (long c = c0; c < c1; c++) {
        const int slice = __builtin_amdgcn_readfirstlane((int)(c * (SPMV_THREADS / SELL_C) + wv));
        const long row = c * SPMV_THREADS + threadIdx.x;
        if (row >= n) continue;
        const long sp = A.sl_ptr[slice];
        const int w = (int)((A.sl_ptr[slice + 1] - sp) / SELL_C);
        const long p0 = sp + (row % SELL_C);
        const int len = A.rp[row + 1] - A.rp[row];
        T acc[SPMV_COLS];
#pragma unroll
        for (int j = 0; j < SPMV_COLS; j++) acc[j] = T(0);
        // the chunks of sell_row, each used for every column
        for (int k0 = 0; k0 < w; k0 += 8) {
            VT vv[8];
            int cc[8];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const bool ok = k0 + k < len;
                vv[k] = ok ? ldp<KEEP>(&val[p0 + (long)SELL_C * (k0 + k)]) : VT(0);
                cc[k] = ok ? ldp<KEEP>(&scol[p0 + (long)SELL_C * (k0 + k)]) : 0;
            }
#pragma unroll
            for (int j = 0; j < SPMV_COLS; j++) {
                if (j < C.nc) {
                    const T *xj = C.x + j * C.ld;
                    T xx[8];
#pragma unroll
                    for (int k = 0; k < 8; k++) xx[k] = k0 + k < len ? xj[cc[k]] : T(0);
#pragma unroll
                    for (int k = 0; k < 8; k++)
                        if (k0 + k < len) acc[j] = fmav(vv[k], xx[k], acc[j]);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < SPMV_COLS; j++) {
            if (j < C.nc) {
                const T *zj = C.z ? C.z + j * C.ld : nullptr;
                const T zq = zj ? zj[row] : T(0);
                C.y[j * C.ld + row] = finish_col(A, C.x + j * C.ld, row, acc[j], zj, zq, C.a[j]);
            }
        }
    }
}

// one block product of at most SPMV_COLS columns; false when K's layout has
// no block kernel (generic DIA, CRS with lanes per row)
template <class VT, class T>
bool launch_cols(const DevMatrix &K, const SpmvArgs<VT, T> &A, const ColArgs<T> &C, hipStream_t st) {
    dim3 gd(spmv_grid(K)), bd(SPMV_THREADS);
    if (K.fmt == DevFmt::CRS) {
        if (!A.sl_ptr || A.pair32) return false;
        SPMV_LAUNCH(k_spmv_sell_cols, (VT, T), A, C);
    } else {
        switch (K.ndiag) {
        case 3: SPMV_LAUNCH(k_spmv_dia_cols, (VT, T, 3), A, C); break;
        case 5: SPMV_LAUNCH(k_spmv_dia_cols, (VT, T, 5), A, C); break;
        case 7: SPMV_LAUNCH(k_spmv_dia_cols, (VT, T, 7), A, C); break;
        default: return false;
        }
    }
    LAUNCH_CHECK();
    return true;
}

// ---------------------------------------------------------------------------
// batched (tile) SpMV: one workgroup per tile of the block-diagonal matrix's
// partition.  Same per-row arithmetic and group layout as k_spmv_crs; the
// epilogue partials are per tile, and a tile whose system has finished
// returns at once.
// ---------------------------------------------------------------------------
struct TileArgs {
    const int *tile_sys;
    const long *tile_r0, *tile_r1;
    const int *info;
    int stride;
};

template <class VT, class T, int EPI, int NV, int G, bool KEEP>
__global__ __launch_bounds__(SPMV_THREADS) void k_bspmv_crs(SpmvArgs<VT, T> A, EpiArgs<T> E, TileArgs ta) {
    const int tile = blockIdx.x;
    if (ta.info && ta.info[(long)ta.tile_sys[tile] * ta.stride] >= 0) return;
    constexpr int GPB = SPMV_THREADS / G;
    constexpr int U = 4;
    constexpr int PC = EPI == EPI_PDOT ? (NV + G - 1) / G : 1;
    __shared__ int s_rp[BATCH_TILE + 1];
    __shared__ T s_red[NV * (SPMV_THREADS / WAVE)];
    T e[EPI == EPI_PDOT ? PC : NV];
#pragma unroll
    for (int i = 0; i < (EPI == EPI_PDOT ? PC : NV); i++) e[i] = T(0);
    const int g = threadIdx.x % G, grp = threadIdx.x / G;
    const long c0 = ta.tile_r0[tile], c1 = ta.tile_r1[tile];
    const T *__restrict__ x = A.x;
    const VT *__restrict__ val = A.val;
    const int *__restrict__ col = A.col;
    for (long q = c0 + threadIdx.x; q <= c1; q += SPMV_THREADS) s_rp[q - c0] = A.rp[q];
    __syncthreads();
    for (long base = c0; base < c1; base += (long)GPB * U) {
        long row[U], rq[U];
        int a[U], b[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            row[u] = base + grp + (long)u * GPB;
            const bool in = row[u] < c1;
            rq[u] = in ? row[u] : c0;
            a[u] = in ? s_rp[row[u] - c0] : 0;
            b[u] = in ? s_rp[row[u] - c0 + 1] : 0;
        }
        VT vv[U];
        int cc[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int j = a[u] + g;
            const bool ok = j < b[u];
            vv[u] = ok ? ldp<KEEP>(&val[j]) : VT(0);
            cc[u] = ok ? ldp<KEEP>(&col[j]) : -1;
        }
        T pe[U][PC];
        if constexpr (EPI == EPI_PDOT) {
#pragma unroll
            for (int u = 0; u < U; u++) epi_load<T, EPI, PC, KEEP>(pe[u], E, rq[u], g, G);
        }
        T acc[U];
#pragma unroll
        for (int u = 0; u < U; u++) acc[u] = cc[u] >= 0 ? mulv(vv[u], x[cc[u]]) : T(0);
#pragma unroll
        for (int u = 0; u < U; u++)
            for (int j = a[u] + g + G; j < b[u]; j += G) acc[u] = fmav(ldp<KEEP>(&val[j]), x[ldp<KEEP>(&col[j])], acc[u]);
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int m = G / 2; m >= 1; m >>= 1) acc[u] = acc[u] + shfl_xor(acc[u], m);
#pragma unroll
        for (int u = 0; u < U; u++)
            if (row[u] < c1) {
                const T zq = A.z ? A.z[row[u]] : T(0);
                const T yv = finish_value(A, row[u], acc[u], zq);
                if (g == 0) A.y[row[u]] = yv;
                if constexpr (EPI == EPI_PDOT) {
                    epi_accum<T, EPI, PC, PC>(e, pe[u], E, yv, g, G);
                } else if (g == 0) {
                    epi_load<T, EPI, PC, KEEP>(pe[u], E, row[u], 0, 1);
                    epi_accum<T, EPI, NV, PC>(e, pe[u], E, yv, 0, 1);
                }
            }
    }
    if constexpr (EPI == EPI_PDOT) epi_store_group<T, NV, G, PC>(e, E, s_red);
    else epi_store<T, EPI, NV>(e, E, s_red);
}

// tile form of k_spmv_sell: a tile starts at any row; each wavefront walks
// whole slices and masks the rows outside the tile
template <class VT, class T, int EPI, int NV, bool KEEP>
__global__ __launch_bounds__(SPMV_THREADS) void k_bspmv_sell(SpmvArgs<VT, T> A, EpiArgs<T> E, TileArgs ta) {
    const int tile = blockIdx.x;
    if (ta.info && ta.info[(long)ta.tile_sys[tile] * ta.stride] >= 0) return;
    constexpr int PC = EPI == EPI_PDOT ? NV : 1;
    __shared__ T s_red[NV * (SPMV_THREADS / WAVE)];
    T e[NV];
#pragma unroll
    for (int i = 0; i < NV; i++) e[i] = T(0);
    const long c0 = ta.tile_r0[tile], c1 = ta.tile_r1[tile];
    const T *zp = A.z;
    // wavefront w takes the slices q0 + w, q0 + w + 4, ... that overlap the
    // tile (one slice per wavefront: uniform start and width); lanes whose
    // row lies outside the tile idle
    const int lane = threadIdx.x % WAVE;
    const long q0 = c0 / SELL_C, q1 = (c1 + SELL_C - 1) / SELL_C;
    for (long q = q0 + threadIdx.x / WAVE; q < q1; q += SPMV_THREADS / WAVE) {
        const int slice = __builtin_amdgcn_readfirstlane((int)q);
        const long row = (long)slice * SELL_C + lane;
        if (row < c0 || row >= c1) continue;
        const long sp = A.sl_ptr[slice];
        const int w = (int)((A.sl_ptr[slice + 1] - sp) / SELL_C);
        const T zq = zp ? zp[row] : T(0);
        T pe[PC];
        if constexpr (EPI == EPI_PDOT) epi_load<T, EPI, PC, KEEP>(pe, E, row, 0, 1);
        const T acc = sell_row<KEEP>(A, row, sp + (row % SELL_C), w);
        const T yv = finish_value(A, row, acc, zq);
        A.y[row] = yv;
        if constexpr (EPI != EPI_PDOT) epi_load<T, EPI, PC, KEEP>(pe, E, row, 0, 1);
        epi_accum<T, EPI, NV, PC>(e, pe, E, yv, 0, 1);
    }
    epi_store<T, EPI, NV>(e, E, s_red);
}

template <class VT, class T, int EPI, int NV>
static void launch_bspmv(const DevMatrix &K, const SpmvArgs<VT, T> &A, EpiArgs<T> E, const TileCtx &tc,
                         hipStream_t st) {
    if (K.fmt != DevFmt::CRS) throw std::invalid_argument("batched systems must be stored as CRS");
    const Partition &P = *tc.part;
    TileArgs ta = tc.tile_sys ? TileArgs{tc.tile_sys, tc.tile_r0, tc.tile_r1, tc.info, tc.stride}
                              : TileArgs{P.tile_sys, P.tile_r0, P.tile_r0 + 1, tc.info, tc.stride};
    const int nt = tc.tile_sys ? tc.ntiles : P.ntiles;
    if (nt < 1) return;
    E.nparts = nt;
    dim3 gd(nt), bd(SPMV_THREADS);
    if (A.sl_ptr) {
        SPMV_LAUNCH(k_bspmv_sell, (VT, T, EPI, NV), A, E, ta);
        LAUNCH_CHECK();
        return;
    }
    switch (K.group) {
    case 1:
    case 2: SPMV_LAUNCH(k_bspmv_crs, (VT, T, EPI, NV, 2), A, E, ta); break;
    case 4: SPMV_LAUNCH(k_bspmv_crs, (VT, T, EPI, NV, 4), A, E, ta); break;
    case 8: SPMV_LAUNCH(k_bspmv_crs, (VT, T, EPI, NV, 8), A, E, ta); break;
    case 16: SPMV_LAUNCH(k_bspmv_crs, (VT, T, EPI, NV, 16), A, E, ta); break;
    case 32: SPMV_LAUNCH(k_bspmv_crs, (VT, T, EPI, NV, 32), A, E, ta); break;
    default: SPMV_LAUNCH(k_bspmv_crs, (VT, T, EPI, NV, 64), A, E, ta); break;
    }
    LAUNCH_CHECK();
}

template <class VT, class T>
void dispatch_epi_tiles(const DevMatrix &K, const SpmvArgs<VT, T> &A, const EpiArgs<T> &E, int epi,
                               const TileCtx &tc, hipStream_t st) {
    if (!tc.part || K.part.get() != tc.part) throw std::invalid_argument("tile launch without the matrix's partition");
    switch (epi) {
    case EPI_NONE: launch_bspmv<VT, T, EPI_NONE, 1>(K, A, E, tc, st); break;
    case EPI_NORM: launch_bspmv<VT, T, EPI_NORM, 1>(K, A, E, tc, st); break;
    case EPI_OMEGA: launch_bspmv<VT, T, EPI_OMEGA, 3>(K, A, E, tc, st); break;
    case EPI_PDOT:
        if (E.prow < 1 || E.prow > 16 || !E.P) throw std::invalid_argument("P^T y epilogue needs 1..16 rows of P");
        if (E.prow <= 1) launch_bspmv<VT, T, EPI_PDOT, 1>(K, A, E, tc, st);
        else if (E.prow <= 2) launch_bspmv<VT, T, EPI_PDOT, 2>(K, A, E, tc, st);
        else if (E.prow <= 4) launch_bspmv<VT, T, EPI_PDOT, 4>(K, A, E, tc, st);
        else if (E.prow <= 8) launch_bspmv<VT, T, EPI_PDOT, 8>(K, A, E, tc, st);
        else launch_bspmv<VT, T, EPI_PDOT, 16>(K, A, E, tc, st);
        break;
    default: throw std::invalid_argument("bad epilogue");
    }
}

#define IDRS_SPMV_PAIR(VT, T)                                                                                  \
    template void dispatch_epi<VT, T>(const DevMatrix &, const SpmvArgs<VT, T> &, const EpiArgs<T> &, int,      \
                                      const int *, hipStream_t);                                               \
    template void dispatch_epi_tiles<VT, T>(const DevMatrix &, const SpmvArgs<VT, T> &, const EpiArgs<T> &, int, \
                                            const TileCtx &, hipStream_t);                                     \
    template bool launch_cols<VT, T>(const DevMatrix &, const SpmvArgs<VT, T> &, const ColArgs<T> &, hipStream_t);

}  // namespace idrs
