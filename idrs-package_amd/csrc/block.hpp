// A whole IDR(s) solve inside one workgroup, for systems small enough that
// the launches, not the work, would set the time.
#pragma once

#include "idrs.hpp"

#include <vector>

namespace idrs {

// true when the solve of A as one system of n rows, or (batch) of every system
// of its partition, the largest of n rows, fits the one-workgroup kernel
template <class T>
bool block_fits(const Operator &A, long n, int s, const SolveOpts<T> &o, bool batch);

// The scratch memory of such a solve, in bytes, for ntot rows in all
template <class T>
size_t block_scratch(const Operator &A, long ntot, int s, const SolveOpts<T> &o);

// What one system's solve ends with
struct BlockResult {
    int info, iter;
    double normr, normb;
};

// Enqueues the solves: nsys systems, rows [row0[k], row0[k+1]) each (device
// array of A's partition; nullptr: one system of ntot rows).  Pointers are device pointers;
// m1 the diagonal of M1 or nullptr, omega the user omegas, resvec of rv_cap
// entries or nullptr, H as State::H.  max_cycles bounds every solve's cycles.
template <class T>
void block_solve(const Operator &A, int nsys, const long *row0, long ntot, int s, const T *b, T *x,
                 const SolveOpts<T> &o, const T *m1, const T *omega, double *resvec, int rv_cap, T *H,
                 long max_cycles, void *scratch, BlockResult *out, hipStream_t st);

}  // namespace idrs
