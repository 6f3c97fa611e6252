// A whole IDR(s) solve (MODULES/IDRS/idrs.inc:1-311 with MAKE_P, P_DOT,
// COMP_OM of idrs_module.f90) inside one workgroup: one launch per solve, one
// workgroup per system of a batch.
//
// What bounds it: with a launch per statement group a small solve waits for
// about four dependent launches per inner step (25 us at 12^3, of which the
// memory traffic is under 1 us).  Here a step's reductions are workgroup
// barriers: the product's input vector (and the Horner vectors) lie in LDS,
// where the gathers are cheap, r, x, the product, the matrix, G, U and P are
// read and written by the thread that owns the row, out of the caches, and the
// s x s logic runs on a State in LDS (r, x and the product in registers:
// spills, 21.7 us a step at 1728 rows against 9.5).  The systems of a batch need not wait
// for each other, so a batch costs its work, not its slowest system's steps.
#include "block.hpp"

#include "idrs_state.hpp"
#include "spmv_epi.hpp"

#include <algorithm>
#include <climits>

namespace idrs {
namespace {

constexpr int BLK_THREADS = 1024;
constexpr int BLK_NMAX = 4096;                     // rows of a system of a batch
constexpr int BLK_SINGLE = 2560;                   // rows of a single system, or with a wide s
constexpr int BLK_S = PDOT_MAX;                    // largest s
constexpr int BLK_DIAG = 32;                       // most stored diagonals
constexpr int BLK_WIDTH = 32;                      // entries of the longest CRS row
constexpr int BLK_DEG = 32;                        // largest polynomial degree
constexpr size_t BLK_LDS = 144 << 10;              // vectors in LDS (of 160 KB)

template <class VT, class T>
struct BlkArgs {
    const long *row0;
    long n;
    // matrix: DIA values [diagonal][n], or CRS, from which the kernel makes
    // an entry-major copy (ev, ec), local column indices in 16 bits
    int ndiag, ud;
    int off[BLK_DIAG];
    const int *rp, *col;
    const VT *val;
    int width;
    VT *ev;
    unsigned short *ec;
    // operator
    int degree;
    T alpha[BLK_DEG + 1];
    // solve
    int s, method, prow, conjP, has_maxit, maxit, user_omega, n_omega, inispace, rv_cap, nritz;
    long max_cycles;
    double kappa, tol;
    unsigned long long p_seed;
    const T *b, *x0, *U0, *PT_raw, *m1, *omega;
    T *x, *G, *U, *P, *r, *y, *H;
    double *resvec;
    BlockResult *out;
};

// Sums of v[0..cnt) (cnt <= 4) over the workgroup into red[0..cnt) (LDS), in a
// fixed order, then f() by wavefront 0; red and what f wrote are valid for
// every thread after the call.  scr: 4 * 16 values of LDS.
template <class T, class F>
__device__ inline void blk_sum(T (&v)[4], int cnt, T *scr, T *red, F &&f) {
    constexpr int NW = BLK_THREADS / WAVE;
    const int lane = threadIdx.x % WAVE, wid = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
#pragma unroll
    for (int q = 0; q < 4; q++)
        if (q < cnt) v[q] = wave_sum(v[q]);
    if (lane == 0)
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (q < cnt) scr[q * NW + wid] = v[q];
    __syncthreads();
    if (wid == 0) {
        // lane 16 q + w holds wavefront w's part of value q
        static_assert(NW == 16, "one row of 16 lanes per value");
        T t = lane / NW < cnt && lane % NW < nw ? scr[lane] : T(0);
        t = row_sum(t);
        if (lane % NW == 0 && lane / NW < cnt) red[lane / NW] = t;
        wave_fence();
        f();
    }
    __syncthreads();
}
template <class T>
__device__ inline void blk_sum(T (&v)[4], int cnt, T *scr, T *red) {
    blk_sum(v, cnt, scr, red, [] {});
}

// a thread's rows
#define BLK_ROWS(q) for (int q = threadIdx.x; q < n; q += blockDim.x)

template <class VT, class T>
struct Blk {
    const BlkArgs<VT, T> &a;
    long r0;
    int n;
    const VT *ev;
    const unsigned short *ec;
    const unsigned char *len;   // LDS: entries of every row

    // (K' X)(q), X in LDS; the entries of a row in stored order
    __device__ inline T product(const T *X, int q) const {
        T acc = T(0);
        if (a.ndiag > 0) {
            for (int d = 0; d < a.ndiag; d++) {
                const int c = q + a.off[d];
                if (c >= 0 && c < n)
                    acc = fmav(d == a.ud ? VT(1) : a.val[(long)(d - (d > a.ud ? 1 : 0)) * n + q], X[c], acc);
            }
            return acc;
        }
        const int m = len[q];
        const VT *v0 = ev + q;
        const unsigned short *c0 = ec + q;
        for (int k0 = 0; k0 < a.width; k0 += 8) {
            VT v[8];
            int c[8];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const bool ok = k0 + k < m;
                v[k] = ok ? v0[(k0 + k) * n] : VT(0);
                c[k] = ok ? c0[(k0 + k) * n] : 0;
            }
#pragma unroll
            for (int k = 0; k < 8; k++)
                if (k0 + k < m) acc = fmav(v[k], X[c[k]], acc);
        }
        return acc;
    }

    // the Horner part of A V (op_apply): returns the vector whose product is
    // A V; V, W1, W2 in LDS, V complete on entry, the result complete on return
    __device__ inline const T *horner(const T *V, T *W1, T *W2) const {
        const T *cur = V;
        T *nxt = W1, *other = W2;
        for (int i = a.degree - 1; i >= 0; i--) {
            const T xs = i == a.degree - 1 ? a.alpha[a.degree] : T(1);
            BLK_ROWS(q) nxt[q] = Tr<T>::fma(a.alpha[i], V[q], xs * product(cur, q));
            __syncthreads();
            cur = nxt;
            T *t = nxt;
            nxt = other;
            other = t;
        }
        return cur;
    }
};

// MAKE_P (idrs_module.f90:839-937): every thread orthonormalises its rows'
// components, the dots and norms over the workgroup
template <class VT, class T>
__device__ inline void blk_make_p(const BlkArgs<VT, T> &a, long r0, int n, T *P, const T *r, T *scr, T *red) {
    const int prow = a.prow;
    if (a.method == 2) {
        BLK_ROWS(q) P[q] = Tr<T>::conj(r[q]);
        return;
    }
    const long cnt = (long)prow * n;
    BLK_ROWS(q) {
        for (int i = 0; i < prow; i++) {
            const long e = (long)q * prow + i;
            if (a.PT_raw) P[e] = a.PT_raw[(long)prow * r0 + e];
            else if constexpr (Tr<T>::is_complex)
                P[e] = T(uniform01(a.p_seed, (uint64_t)e), uniform01(a.p_seed, (uint64_t)(cnt + e)));
            else P[e] = uniform01(a.p_seed, (uint64_t)e);
        }
    }
    for (int k = 0; k < prow; k++) {
        for (int i0 = 0; i0 < k; i0 += 4) {
            T e[4] = {T(0), T(0), T(0), T(0)};
            BLK_ROWS(q) {
                const T pk = P[(long)q * prow + k];
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (i0 + i < k) e[i] = fmaT(Tr<T>::conj(P[(long)q * prow + i0 + i]), pk, e[i]);
            }
            blk_sum(e, min(4, k - i0), scr, red + i0);
        }
        T e[4] = {T(0), T(0), T(0), T(0)};
        BLK_ROWS(q) {
            T p = P[(long)q * prow + k];
            for (int i = 0; i < k; i++) p = fmaT(-red[i], P[(long)q * prow + i], p);
            P[(long)q * prow + k] = p;
            e[0] = e[0] + T(Tr<T>::abs2(p));
        }
        blk_sum(e, 1, scr, red);
        const double rho = sqrt(sre(red[0]));
        BLK_ROWS(q) {
            const T p = P[(long)q * prow + k];
            if constexpr (Tr<T>::is_complex) P[(long)q * prow + k] = T(p.re / rho, p.im / rho);
            else P[(long)q * prow + k] = p / rho;
        }
    }
}

// One solve.  The products are the passes of one loop: phase -1 the initial
// residual (with x0), 0..s-1 the inner steps, s the omega step, s+1 the final
// true residual.  V holds the vector the next product takes.
template <class VT, class T>
__global__ __launch_bounds__(BLK_THREADS) void k_block_solve(BlkArgs<VT, T> a) {
    extern __shared__ __align__(16) unsigned char dyn[];
    __shared__ State<T, BLK_S> st;
    __shared__ T scr[4 * (BLK_THREADS / WAVE)], red[BLK_S + 4];
    __shared__ unsigned char len[BLK_NMAX];
    const int sys = blockIdx.x, lane = threadIdx.x;
    const long r0 = a.row0 ? a.row0[sys] : 0;
    const int n = (int)((a.row0 ? a.row0[sys + 1] : a.n) - r0);
    T *V = (T *)dyn, *W1 = V + n, *W2 = W1 + (a.degree > 1 ? n : 0);
    const int s = a.s, prow = a.prow;
    // no two of a solve's vectors overlap
    T *G = a.G + (long)s * r0, *U = a.U + (long)s * r0;
    T *P = a.P + (long)prow * r0;
    T *r = a.r + r0, *y = a.y + r0;
    const T *m1 = a.m1 ? a.m1 + r0 : nullptr;
    const T *b = a.b + r0;
    T *x = a.x + r0;
    // the entry-major copy of a CRS matrix (every thread reads its own rows')
    VT *ev = a.ndiag ? nullptr : a.ev + (long)a.width * r0;
    unsigned short *ec = a.ndiag ? nullptr : a.ec + (long)a.width * r0;
    if (a.ndiag == 0)
        BLK_ROWS(q) {
            const int p0 = a.rp[r0 + q], m = a.rp[r0 + q + 1] - p0;
            len[q] = (unsigned char)m;
            for (int p = 0; p < m; p++) {
                ev[p * n + q] = a.val[p0 + p];
                ec[p * n + q] = (unsigned short)(a.col[p0 + p] - r0);
            }
        }
    const Blk<VT, T> B{a, r0, n, ev, ec, len};
    if (threadIdx.x == 0) {
        const int mx = a.has_maxit ? a.maxit : (int)min(2L * n, 1000L);    // idrs.inc:37-38
        scalar_init(&st, s, a.method, prow, a.conjP, mx, a.kappa, a.tol, a.user_omega, a.n_omega, a.inispace,
                    a.rv_cap);
        st.H = a.H;
        st.nritz = a.nritz;
    }
    // x = 0 or x0, U = U0 (idrs.inc:52-65); normb, tolb (idrs.inc:93-95)
    {
        T e[4] = {T(0), T(0), T(0), T(0)};
        BLK_ROWS(q) {
            const T bq = b[q], xq = a.x0 ? a.x0[r0 + q] : T(0);
            x[q] = xq;
            V[q] = xq;
            r[q] = bq;
            e[0] = e[0] + T(Tr<T>::abs2(bq));
            if (a.inispace)
                for (int i = 0; i < s; i++) U[i * n + q] = a.U0[(long)i * n + q];
        }
        blk_sum(e, 1, scr, red, [&] {
            if (lane == 0) {
                st.normb = sqrt(sre(red[0]));
                st.tolb = st.tol * st.normb;
            }
        });
    }
    int phase = a.x0 ? -1 : s + 2;
    long cycles = 0;
    while (true) {
        const T *X = V;
        if (phase <= s + 1) X = B.horner(V, W1, W2);
        if (phase < 0 || phase == s + 2) {
            // r = b - A x0; normr (idrs.inc:96-101); P and f = P^T r
            // (idrs.inc:109-126, 147)
            T e[4] = {T(0), T(0), T(0), T(0)};
            BLK_ROWS(q) {
                T rq = r[q];
                if (phase < 0) {
                    rq = rq - B.product(X, q);
                    r[q] = rq;
                }
                e[0] = e[0] + T(Tr<T>::abs2(rq));
            }
            blk_sum(e, 1, scr, red, [&] {
                if (lane == 0) {
                    const double nr = sqrt(sre(red[0]));
                    st.normr = nr;
                    if (a.resvec) a.resvec[0] = nr;                        // idrs.inc:97
                    if (nr <= st.tolb) st.info = 0;                        // idrs.inc:101
                }
            });
            blk_make_p<VT, T>(a, r0, n, P, r, scr, red);
            for (int i0 = 0; i0 < prow; i0 += 4) {
                T f[4] = {T(0), T(0), T(0), T(0)};
                BLK_ROWS(q) {
                    const T rq = r[q];
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (i0 + i < prow) {
                            T p = P[q * prow + i0 + i];
                            if (a.conjP) p = Tr<T>::conj(p);
                            f[i] = fmaT(p, rq, f[i]);
                        }
                }
                blk_sum(f, min(4, prow - i0), scr, red + i0);
            }
            if (threadIdx.x < s) st.f[threadIdx.x] = threadIdx.x < prow ? red[threadIdx.x] : T(0);
            phase = s + 1;   // to the next cycle, or the end
        } else if (phase < s) {
            // G(:,k) = A U(:,k), mu = P^T G(:,k) -> alpha, beta, gamma
            // (idrs.inc:194-229)
            const int k = phase;
            for (int i0 = 0; i0 < prow; i0 += 4) {
                T e[4] = {T(0), T(0), T(0), T(0)};
                BLK_ROWS(q) {
                    T yq;
                    if (i0 == 0) {
                        yq = B.product(X, q);
                        y[q] = yq;
                    } else {
                        yq = y[q];
                    }
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (i0 + i < prow) {
                            T p = P[q * prow + i0 + i];
                            if (a.conjP) p = Tr<T>::conj(p);
                            e[i] = fmaT(p, yq, e[i]);
                        }
                }
                blk_sum(e, min(4, prow - i0), scr, red + i0, [&] {
                    if (i0 + 4 >= prow) wave_mu(&st, st.M, BLK_S, k, red, lane);
                });
            }
            if (st.info < 0) {
                // bi-orthogonalise G(:,k), U(:,k); r, x; U(:,k+1)
                // (idrs.inc:199-224, 155-190)
                const T beta = st.beta[k], om = st.om;
                const int jj = st.jj;
                T e[4] = {T(0), T(0), T(0), T(0)};
                BLK_ROWS(q) {
                    T gk = y[q], uk = V[q];
                    const T rq0 = r[q], xq0 = x[q];
                    for (int i = 0; i < k; i++) {
                        const T al = st.alpha[i];
                        gk = fmaT(-al, G[i * n + q], gk);
                        uk = fmaT(-al, U[i * n + q], uk);
                    }
                    G[k * n + q] = gk;
                    U[k * n + q] = uk;
                    const T rq = fmaT(-beta, gk, rq0);
                    r[q] = rq;
                    x[q] = fmaT(beta, uk, xq0);
                    e[0] = e[0] + T(Tr<T>::abs2(rq));
                    T t = rq;   // the omega step's vector after the last inner step
                    if (k + 1 < s) {
                        if (jj > 0) {
                            T v = rq;
                            for (int i = k + 1; i < s; i++) v = fmaT(-st.gamma[i], G[i * n + q], v);
                            t = om * (m1 ? sdiv(v, m1[q]) : v);
                            for (int i = k + 1; i < s; i++) t = fmaT(st.gamma[i], U[i * n + q], t);
                        } else {
                            t = a.inispace ? U[(k + 1) * n + q] : m1 ? sdiv(rq, m1[q]) : rq;
                        }
                    } else if (m1) {
                        t = sdiv(rq, m1[q]);
                    }
                    V[q] = t;
                }
                blk_sum(e, 1, scr, red, [&] {
                    if (lane == 0) scalar_norm(&st, sqrt(sre(red[0])), a.resvec);
                });
            }
            phase = k + 1;
        } else if (phase == s) {
            // omega step (idrs.inc:260-299)
            {
                T e[4] = {T(0), T(0), T(0), T(0)};
                BLK_ROWS(q) {
                    const T yq = B.product(X, q), rq = r[q];
                    y[q] = yq;
                    e[0] = fmaT(Tr<T>::conj(rq), rq, e[0]);
                    e[1] = fmaT(Tr<T>::conj(yq), yq, e[1]);
                    e[2] = fmaT(Tr<T>::conj(yq), rq, e[2]);
                }
                blk_sum(e, 3, scr, red, [&] {
                    if (lane == 0) scalar_om(&st, red, a.omega);
                });
            }
            if (st.info < 0) {
                const T om = st.om;
                for (int i0 = -1; i0 < prow; i0 += 4) {
                    // values ||r||^2 and P^T r, four at a time
                    T e[4] = {T(0), T(0), T(0), T(0)};
                    BLK_ROWS(q) {
                        T rq = r[q];
                        if (i0 < 0) {
                            rq = fmaT(-om, y[q], rq);
                            r[q] = rq;
                            x[q] = fmaT(om, V[q], x[q]);
                            e[0] = T(Tr<T>::abs2(rq)) + e[0];
                        }
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            if (i0 + i >= 0 && i0 + i < prow) {
                                T p = P[q * prow + i0 + i];
                                if (a.conjP) p = Tr<T>::conj(p);
                                e[i] = fmaT(p, rq, e[i]);
                            }
                    }
                    blk_sum(e, min(4, prow - i0), scr, red + i0 + 1, [&] {
                        if (i0 + 4 >= prow) wave_cycle(&st, st.M, BLK_S, red, a.resvec, lane);
                    });
                }
            }
            phase = s + 1;
        } else {
            // the true residual (idrs.inc:304-310)
            T e[4] = {T(0), T(0), T(0), T(0)};
            BLK_ROWS(q) {
                const T rq = b[q] - B.product(X, q);
                e[0] = e[0] + T(Tr<T>::abs2(rq));
            }
            blk_sum(e, 1, scr, red);
            if (threadIdx.x == 0) {
                const double nr = sqrt(sre(red[0]));
                a.out[sys] = BlockResult{st.info == 0 && nr > st.tolb ? 2 : st.info, st.iter, nr, st.normb};
            }
            return;
        }
        // the next product's vector
        __syncthreads();
        const bool end = st.info >= 0 || (phase == s + 1 && cycles++ == a.max_cycles);
        if (end) {
            BLK_ROWS(q) V[q] = x[q];
            phase = s + 1;
            __syncthreads();
        } else if (phase == s + 1) {
            // U(:,0) of the next cycle (idrs.inc:155-190)
            const T om = st.om;
            const int jj = st.jj;
            BLK_ROWS(q) {
                T t = r[q];
                if (jj > 0) {
                    for (int i = 0; i < s; i++) t = fmaT(-st.gamma[i], G[i * n + q], t);
                    t = om * (m1 ? sdiv(t, m1[q]) : t);
                    for (int i = 0; i < s; i++) t = fmaT(st.gamma[i], U[i * n + q], t);
                } else if (a.inispace) {
                    t = U[q];
                } else if (m1) {
                    t = sdiv(t, m1[q]);
                }
                V[q] = t;
            }
            phase = 0;
            __syncthreads();
        }
    }
}

template <class T>
size_t lds_bytes(const Operator &A, long n) {
    return sizeof(T) * (size_t)n * (1 + (A.degree > 0 ? 1 : 0) + (A.degree > 1 ? 1 : 0));
}

size_t up(size_t b) { return (b + 255) & ~(size_t)255; }

template <class T> T alpha_T(std::complex<double> c);
template <> double alpha_T<double>(std::complex<double> c) { return c.real(); }
template <> c128 alpha_T<c128>(std::complex<double> c) { return c128(c.real(), c.imag()); }

template <class VT, class T>
void launch(const Operator &A, BlkArgs<VT, T> &a, long nmax, int nsys, hipStream_t st) {
    const int threads = (int)std::min<long>(BLK_THREADS, (nmax + WAVE - 1) / WAVE * WAVE);
    HIP_TRY(hipFuncSetAttribute((const void *)(k_block_solve<VT, T>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)BLK_LDS));
    hipLaunchKernelGGL((k_block_solve<VT, T>), dim3(nsys), dim3(threads), lds_bytes<T>(A, nmax), st, a);
    LAUNCH_CHECK();
}

}  // namespace

// One workgroup's time of a step of a single system against that of its
// launches, both in us without what they have in common: rows times the
// entries of the step's products and the columns of G, U and P, against a
// latency per launch (lanes per row, DIA, sliced).  Fitted to 60 steps of 256
// to 2560 rows with 3 to 32 entries, degree 0 to 32, s = 1 to 16, real and
// complex: the choice is within 12 % of the faster one but for one case of 570
// (16 %).  One workgroup / launches, us a step: 7 entries CRS, IDR(4), 1728
// rows 9.5 / 19, 2560 rows 12 / 19, with degree 8 39 / 60; DIA with degree 32
// 153 / 114; 32 entries with degree 4 78 / 38; IDR(16), 7 entries, 1024 rows
// 22 / 29, 2560 rows 46 / 30.
static bool block_is_faster(const DevMatrix &K, long n, int s, int degree) {
    const bool dia = K.fmt == DevFmt::DIA;
    const double w = dia ? K.ndiag : K.max_row, products = (degree + 1) * (s + 1.0) / s;
    const double launch = dia ? 2.8 + 0.026 * w : K.group == 1 ? 1.2 + 0.12 * w : 3.1;
    return 1e-3 * n * ((dia ? 0.19 : 0.1) * w * products + 0.45 * s + 0.009 * s * s) <
           7.4 + 0.36 * s + launch * products;
}

// The systems of a batch, up to 4096 rows each, do not wait for each other and
// the tile launches cost more, so they take the kernel with any degree and row
// length (256 systems of 24^2 to 64^2 rows, IDR(2): 13.8 -> 4.4 ms; one of 4096
// rows with 32 entries and degree 32: tiles 2262 us a step, here 716); above
// 2560 rows a wide shadow space, or a wider one over long complex rows, stays
// on the tiles (one system of 4096 rows, sliced: IDR(16) 52 / 74, IDR(8) with
// 32 complex entries 61 / 77).  A single system takes it up to 2560 rows, where
// it is the faster one.  The vectors have to fit LDS, and the form has to be
// one the kernel has.
template <class T>
bool block_fits(const Operator &A, long n, int s, const SolveOpts<T> &o, bool batch) {
    if constexpr (!std::is_same<T, double>::value && !std::is_same<T, c128>::value) return false;
    const DevMatrix &K = *A.K;
    if (A.general() || A.values32 || s > BLK_S || A.degree > BLK_DEG) return false;
    if (K.nrows != K.ncols) return false;
    if (K.fmt == DevFmt::DIA ? K.ndiag > BLK_DIAG : K.max_row > BLK_WIDTH) return false;
    if (batch) {
        const bool wide = s > 8 || (Tr<T>::is_complex && s > 4 && K.max_row > 16);
        if (n > (wide ? BLK_SINGLE : BLK_NMAX)) return false;
    } else if (n > BLK_SINGLE || !block_is_faster(K, n, s, A.degree)) {
        return false;
    }
    if (!Tr<T>::is_complex && A.values_complex()) return false;   // refused further on
    // the kernel has no seed shift; the inner solve of a flexible Krylov method
    // stays on the launches, as its outer count follows the inner rounding
    if (A.seed != std::complex<double>(0.0, 0.0) || o.inner) return false;
    return lds_bytes<T>(A, n) <= BLK_LDS;
}

template <class T>
size_t block_scratch(const Operator &A, long ntot, int s, const SolveOpts<T> &o) {
    const DevMatrix &K = *A.K;
    const int prow = o.variant == 1 ? s : 1;
    size_t b = up(sizeof(T) * (size_t)ntot * s) * 2 + up(sizeof(T) * (size_t)ntot * prow) +
               up(sizeof(T) * (size_t)ntot) * 2;
    if (K.fmt == DevFmt::CRS) {
        const size_t vsz = A.values_complex() ? sizeof(c128) : sizeof(double);
        b += up(vsz * (size_t)ntot * K.max_row) + up(sizeof(unsigned short) * (size_t)ntot * K.max_row);
    }
    return b;
}

template <class T>
void block_solve(const Operator &A, int nsys, const long *row0, long ntot, int s, const T *b, T *x,
                 const SolveOpts<T> &o, const T *m1, const T *omega, double *resvec, int rv_cap, T *H,
                 long max_cycles, void *scratch, BlockResult *out, hipStream_t st) {
    const DevMatrix &K = *A.K;
    // without row0 the rows are one system, also those of a batch's matrix
    long nmax = ntot;
    if (row0) {
        nmax = 0;
        for (int k = 0; k < nsys; k++) nmax = std::max(nmax, K.part->h_row0[k + 1] - K.part->h_row0[k]);
    }
    auto go = [&](auto tag) {
        using VT = decltype(tag);
        BlkArgs<VT, T> a{};
        a.row0 = row0;
        a.n = ntot;
        a.ud = INT_MAX;
        a.val = (const VT *)A.values();
        if (K.fmt == DevFmt::DIA) {
            a.ndiag = K.ndiag;
            for (int d = 0; d < K.ndiag; d++) a.off[d] = K.h_offsets[d];
            if (A.sval && A.unit_diag >= 0) a.ud = A.unit_diag;
        }
        a.rp = K.row_ptr;
        a.col = K.col;
        a.width = K.max_row;
        a.degree = A.degree;
        for (int i = 0; i <= A.degree && A.degree > 0; i++) a.alpha[i] = alpha_T<T>(A.alpha[i]);
        a.s = s;
        a.method = o.variant;
        a.prow = o.variant == 1 ? s : 1;
        a.conjP = (o.variant >= 3 && Tr<T>::is_complex) ? 1 : 0;
        a.has_maxit = o.has_maxit;
        a.maxit = o.maxit;
        a.user_omega = omega ? 1 : 0;
        a.n_omega = omega ? o.n_omega : 0;
        a.inispace = o.U0 ? 1 : 0;
        a.rv_cap = rv_cap;
        a.nritz = o.nritz;
        a.max_cycles = max_cycles;
        a.kappa = (o.variant == 1 || o.variant == 3) ? (double)0.7f : 0.0;   // idrs.inc:112-124
        a.tol = o.tol;
        a.p_seed = o.p_seed;
        a.b = b;
        a.x0 = o.x0;
        a.U0 = o.U0;
        a.PT_raw = o.PT_raw;
        a.m1 = m1;
        a.omega = omega;
        a.x = x;
        a.H = H;
        a.resvec = resvec;
        a.out = out;
        char *p = (char *)scratch;
        auto take = [&](size_t bytes) {
            void *q = p;
            p += up(bytes);
            return q;
        };
        a.G = (T *)take(sizeof(T) * (size_t)ntot * s);
        a.U = (T *)take(sizeof(T) * (size_t)ntot * s);
        a.P = (T *)take(sizeof(T) * (size_t)ntot * a.prow);
        a.r = (T *)take(sizeof(T) * (size_t)ntot);
        a.y = (T *)take(sizeof(T) * (size_t)ntot);
        if (K.fmt == DevFmt::CRS) {
            a.ev = (VT *)take(sizeof(VT) * (size_t)ntot * K.max_row);
            a.ec = (unsigned short *)take(sizeof(unsigned short) * (size_t)ntot * K.max_row);
        }
        launch<VT, T>(A, a, nmax, nsys, st);
    };
    if (A.values_complex()) {
        if constexpr (Tr<T>::is_complex) go(c128{});
    } else {
        go(double{});
    }
}

#define IDRS_BLOCK(T)                                                                                            \
    template bool block_fits<T>(const Operator &, long, int, const SolveOpts<T> &, bool);                        \
    template size_t block_scratch<T>(const Operator &, long, int, const SolveOpts<T> &);                         \
    template void block_solve<T>(const Operator &, int, const long *, long, int, const T *, T *,                 \
                                 const SolveOpts<T> &, const T *, const T *, double *, int, T *, long, void *,   \
                                 BlockResult *, hipStream_t);
IDRS_BLOCK(double)
IDRS_BLOCK(c128)

}  // namespace idrs
