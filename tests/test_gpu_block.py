"""Small systems solved whole in one workgroup, against the oracle at the
sizes where that kernel's shape changes: one row, a wavefront and a workgroup
of rows and one more, the largest single system and the first above it, every
stored form, and a batch up to its largest system.

The fixed-count solutions agree to 1e-10 relative, the bar of the other GPU
solves against the oracle; both sides take the same steps, so their rounding
is all that differs.
"""
import numpy as np
import pytest

import idrs_amd
import orc
from helpers import rel, rounding_spread
from idrs_amd import problems as P

pytestmark = pytest.mark.gpu


def _system(n, seed, cplx=False):
    """A banded nonsymmetric diagonally dominant matrix as CRS arrays and as
    diagonals (offsets -7, -1, 0, 2)."""
    rng = np.random.default_rng(seed)
    offs = [o for o in (-7, -1, 0, 2) if abs(o) < n]
    i = np.arange(n)
    vals = rng.uniform(-1, 1, (n, len(offs))) + (1j * rng.uniform(-1, 1, (n, len(offs))) if cplx else 0)
    vals[:, offs.index(0)] = 4.0 + rng.uniform(0, 1, n)
    ok = np.stack([(i + o >= 0) & (i + o < n) for o in offs], axis=1)
    vals = np.where(ok, vals, 0)
    rp = np.concatenate([[1], 1 + np.cumsum(ok.sum(1))]).astype(np.int32)
    col = (i[:, None] + np.array(offs) + 1)[ok].astype(np.int32)
    return P.Crs(n, rp, col, np.ascontiguousarray(vals[ok])), (np.array(offs, dtype=np.int32), vals)


def _box(dims):
    """A 7-point stencil as CRS arrays and diagonals."""
    n = dims[0] * dims[1] * dims[2]
    i = np.arange(n)
    xyz, st = (i % dims[0], (i // dims[0]) % dims[1], i // (dims[0] * dims[1])), (1, dims[0], dims[0] * dims[1])
    cols = {0: np.full(n, 7.0)}
    for d in range(3):
        cols[-st[d]] = np.where(xyz[d] > 0, -1.0 - 0.05 * d, 0.0)
        cols[st[d]] = np.where(xyz[d] < dims[d] - 1, -0.9 + 0.05 * d, 0.0)
    offs = np.array(sorted(cols), dtype=np.int32)
    vals = np.stack([cols[o] for o in offs], axis=1)
    keep = vals != 0
    rp = np.concatenate([[1], 1 + np.cumsum(keep.sum(1))]).astype(np.int32)
    return P.Crs(n, rp, (i[:, None] + offs + 1)[keep].astype(np.int32), vals[keep]), offs, vals


@pytest.mark.parametrize("n,s,form", [
    (1, 1, "crs"), (2, 1, "crs"), (63, 2, "dia"), (64, 4, "crs"), (65, 5, "crs"), (1023, 4, "dia"), (1024, 3, "crs"),
    (1025, 16, "crs"), (2047, 4, "complex"), (2049, 8, "dia"), (2560, 4, "crs"), (2561, 4, "crs"),
    (1500, 4, "poly"), (1500, 4, "m1"), (700, 2, "x0"), (700, 1, "variant2"), (700, 1, "variant4"),
    (700, 4, "variant3"), (700, 4, "variant4")])
def test_small_solves_match_oracle(gpu, n, s, form):
    cplx = form == "complex"
    crs, (offs, vals) = _system(n, 3 + n, cplx)
    rng = np.random.default_rng(n)
    b = rng.uniform(-1, 1, n) + (1j * rng.uniform(-1, 1, n) if cplx else 0)
    PT = P.gaussian_shadow(n, s, seed=1, complex=cplx)
    kw, okw, mk = {}, {}, dict(which_precon=0)
    if form == "dia":
        K = idrs_amd.dia_format(n, n, offs, rvals=vals)
    else:
        K = idrs_amd.crs_format(n, n, crs.row_ptr, crs.col_ind, **{"cval" if cplx else "rval": crs.val})
    if form == "poly":
        mk = dict(which_precon=1, degree=3, alpha=orc.chebyshev(3, np.array([0.3, 1.7])))
    A = idrs_amd.Matrix(K, which_precon=mk["which_precon"])
    if form == "poly":
        idrs_amd.real_preconditioner(A, 2, 3, foci=[0.3, 1.7])
    Ao = orc.OracleMatrix(orc.CRS, n, crs=crs, complex_vectors=cplx, **mk)
    if form == "m1":
        kw["M1"], okw["M1"] = idrs_amd.Matrix(K, which_precon=1), orc.OracleMatrix(orc.CRS, n, crs=crs, which_precon=1)
    if form == "x0":
        kw["x0"] = okw["x0"] = rng.standard_normal(n)
    if form.startswith("variant"):
        kw["variant"] = okw["variant"] = int(form[-1])
    k = min(10, n)
    g = idrs_amd.idrs(A, b, s, tolerance=0.0, maximum_iterations=k, PT_raw=PT, resvec=True, **kw)
    o = orc.idrs(Ao, b, s, tolerance=0.0, maximum_iterations=k, PT_raw=PT, **okw)
    assert idrs_amd.last_solve_path() == ("workgroup" if n <= 2560 else "folded")
    assert g.iterations == o[3]
    if n > 2:   # one or two unknowns end in a breakdown on both sides
        assert g.flag == o[1] and rel(g.x, o[0]) < 1e-10
    c = idrs_amd.idrs(A, b, s, tolerance=1e-9, maximum_iterations=500, PT_raw=PT, **kw)
    co = orc.idrs(Ao, b, s, tolerance=1e-9, maximum_iterations=500, PT_raw=PT, **okw)
    assert c.flag == co[1] and abs(c.iterations - co[3]) <= 2


@pytest.mark.parametrize("sizes,s", [([1, 64, 65, 900], 2), ([4096, 3, 1025, 2048, 4095], 4), ([4097, 30], 2)])
def test_small_batches_match_oracle(gpu, sizes, s):
    systems = [_system(n, 11 + n)[0] for n in sizes]
    K = idrs_amd.batch_format([idrs_amd.crs_format(c.n, c.n, c.row_ptr, c.col_ind, rval=c.val) for c in systems])
    b = np.random.default_rng(5).uniform(-1, 1, sum(sizes))
    r = idrs_amd.idrs_batched(idrs_amd.Matrix(K), b, s, tolerance=1e-9, maximum_iterations=300)
    assert idrs_amd.last_solve_path() == ("workgroup" if max(sizes) <= 4096 else "tiles")
    at = 0
    for k, c in enumerate(systems):
        bk = b[at:at + c.n]
        o = orc.idrs(orc.OracleMatrix(orc.CRS, c.n, crs=c), bk, s, tolerance=1e-9, maximum_iterations=300)
        assert abs(int(r.iterations[k]) - o[3]) <= 2
        if c.n > s:   # a system of at most s unknowns ends in a breakdown
            assert r.flag[k] == o[1] == 0
            assert np.linalg.norm(c.matvec(r.x[at:at + c.n]) - bk) <= 1.01e-9 * np.linalg.norm(bk)
        at += c.n


# One solve of a batch's whole matrix, each system of another size: the rows in
# all, not a system's, decide the kernel (964 and 2560 rows: one workgroup).
@pytest.mark.parametrize("sizes", [[64, 900], [900, 64], [60, 1500, 1000], [60, 1500, 1001], [1, 4000]])
@pytest.mark.parametrize("entry", ["host", "ritz"])
def test_single_solve_on_a_batch_matrix(gpu, sizes, entry):
    systems = [_system(n, 11 + n)[0] for n in sizes]
    KB = idrs_amd.batch_format([idrs_amd.crs_format(c.n, c.n, c.row_ptr, c.col_ind, rval=c.val) for c in systems])
    at = np.concatenate([[0], np.cumsum(sizes)])
    nz = np.concatenate([[0], np.cumsum([c.nnz for c in systems])])
    whole = P.Crs(int(at[-1]), np.concatenate([[1]] + [c.row_ptr[1:] + nz[k] for k, c in enumerate(systems)]).astype(np.int32),
                  np.concatenate([c.col_ind + at[k] for k, c in enumerate(systems)]).astype(np.int32),
                  np.concatenate([c.val for c in systems]))
    n, s = whole.n, 4
    b = np.random.default_rng(7).uniform(-1, 1, n)
    PT = P.gaussian_shadow(n, s, seed=2)
    solve = idrs_amd.idrs if entry == "host" else idrs_amd.idrs_ritz
    g = solve(idrs_amd.Matrix(KB), b, s, tolerance=0.0, maximum_iterations=10, PT_raw=PT)
    assert idrs_amd.last_solve_path() == ("workgroup" if n <= 2560 else "folded")
    o = orc.idrs(orc.OracleMatrix(orc.CRS, n, crs=whole), b, s, tolerance=0.0, maximum_iterations=10, PT_raw=PT)
    assert (g.flag, g.iterations) == (o[1], o[3]) and rel(g.x, o[0]) < 1e-10


# Which solves the kernel takes: on both sides of the lines by the work of a
# step against its launches, each against the oracle (degree 32 in powers of A,
# coefficients up to 7e10, amplifies rounding: there the bar is what 1e-16
# perturbations of b do to the oracle itself).
@pytest.mark.parametrize("dims,form,s,degree,path", [
    ((12, 12, 12), "crs", 4, 0, "workgroup"), ((16, 16, 10), "crs", 4, 8, "workgroup"),
    ((16, 8, 8), "crs", 16, 0, "workgroup"), ((16, 16, 10), "crs", 16, 0, "folded"),
    ((8, 8, 8), "dia", 4, 32, "workgroup"), ((16, 16, 10), "dia", 4, 32, "folded"),
    (512, "dense rows", 4, 8, "workgroup"), (2560, "dense rows", 4, 4, "folded")])
def test_choice_of_the_one_workgroup_solve(gpu, dims, form, s, degree, path):
    if form == "dense rows":
        crs = P.random_dominant(dims, k=31, seed=1)
        K = idrs_amd.crs_format(crs.n, crs.n, crs.row_ptr, crs.col_ind, rval=crs.val)
    else:
        crs, offs, vals = _box(dims)
        if form == "dia":
            K = idrs_amd.dia_format(crs.n, crs.n, offs, rvals=vals)
        else:
            K = idrs_amd.crs_format(crs.n, crs.n, crs.row_ptr, crs.col_ind, rval=crs.val)
    A = idrs_amd.Matrix(K, which_precon=1 if degree else 0)
    mk = {}
    if degree:
        idrs_amd.real_preconditioner(A, 2, degree, foci=[0.3, 1.7])
        mk = dict(which_precon=1, degree=degree, alpha=orc.chebyshev(degree, np.array([0.3, 1.7])))
    b = np.random.default_rng(3).uniform(-1, 1, crs.n)
    PT = P.gaussian_shadow(crs.n, s, seed=4)
    g = idrs_amd.idrs(A, b, s, tolerance=0.0, maximum_iterations=6, PT_raw=PT)
    assert idrs_amd.last_solve_path() == path
    Ao = orc.OracleMatrix(orc.CRS, crs.n, crs=crs, **mk)

    def run(bp):
        o = orc.idrs(Ao, bp, s, tolerance=0.0, maximum_iterations=6, PT_raw=PT)
        return o[0], o[3]

    xo, its = run(b)
    bar = max(1e-10, 100 * rounding_spread(run, b)[0]) if degree == 32 else 1e-10
    assert (g.flag, g.iterations) == (1, its) and rel(g.x, xo) < bar


@pytest.mark.parametrize("n,s,cplx,k,path", [
    (4096, 8, False, 4, "workgroup"), (4096, 9, False, 4, "tiles"), (2560, 16, False, 4, "workgroup"),
    (4096, 4, True, 31, "workgroup"), (4096, 8, True, 31, "tiles"), (4096, 8, True, 4, "workgroup")])
def test_choice_of_the_one_workgroup_batch(gpu, n, s, cplx, k, path):
    crs = [P.random_dominant(m, k=k, seed=m) for m in (n, 70)]
    if cplx:
        for c in crs:
            c.val = c.val * (1 + 0.1j)
    K = idrs_amd.batch_format([idrs_amd.crs_format(c.n, c.n, c.row_ptr, c.col_ind,
                                                   **{"cval" if cplx else "rval": c.val}) for c in crs])
    b = np.random.default_rng(6).uniform(-1, 1, n + 70) + (0j if cplx else 0)
    r = idrs_amd.idrs_batched(idrs_amd.Matrix(K), b, s, tolerance=0.0, maximum_iterations=7)
    assert idrs_amd.last_solve_path() == path
    for c, sl in ((crs[0], slice(0, n)), (crs[1], slice(n, n + 70))):
        o = orc.idrs(orc.OracleMatrix(orc.CRS, c.n, crs=c, complex_vectors=cplx), b[sl], s, tolerance=0.0,
                     maximum_iterations=7)
        assert rel(r.x[sl], o[0]) < 1e-10
