"""Row-coded products (a byte per row and a table of the distinct rows)
against the uncoded products of the same matrices, bit for bit: the same
operations on the same values in the same order.  A solve looks for the code,
a product alone does not, so that an operator's products before its first
solve, and the allocation-free solve, which builds nothing, are the uncoded
ones (many products look too).
"""
import ctypes

import numpy as np
import pytest

import idrs_amd
from idrs_amd import _lib
from test_gpu_fold import _b, _solve

pytestmark = pytest.mark.gpu


def _box(dims, rows):
    """7-point stencil on a box with 'rows' kinds of interior rows."""
    nx, ny, nz = dims
    n = nx * ny * nz
    i = np.arange(n)
    xyz, ext, st = (i % nx, (i // nx) % ny, i // (nx * ny)), dims, (1, nx, nx * ny)
    kind = 1.0 + (i * 2654435761 % rows) / 7.0
    cols = {0: 6.5 * kind}
    for d in range(3):
        cols[-st[d]] = np.where(xyz[d] > 0, -1.0 - 0.1 * d, 0.0) * kind
        cols[st[d]] = np.where(xyz[d] < ext[d] - 1, -0.9 + 0.1 * d, 0.0) * kind
    offs = np.array(sorted(cols), dtype=np.int32)
    return n, offs, np.stack([cols[o] for o in offs], axis=1)


# 32^3 is the fewest rows coded; 1 kind has 27 distinct rows, 9 kinds 243, 10
# kinds more than a byte holds (DIA stays uncoded and sliced CRS codes its
# column offsets alone: still the same bits), 1000 as with variable coefficients
@pytest.mark.parametrize("dims,kinds", [((32, 32, 32), 1), ((33, 31, 37), 2), ((41, 29, 35), 9), ((41, 29, 35), 10),
                                        ((35, 33, 31), 1000)])
@pytest.mark.parametrize("fmt", ["dia", "crs"])
@pytest.mark.parametrize("scaled", [False, True])
def test_coded_products_are_the_same_bits(gpu, dims, kinds, fmt, scaled):
    n, offs, vals = _box(dims, kinds)
    rng = np.random.default_rng(1)
    if fmt == "dia":
        K = idrs_amd.dia_format(n, n, offs, rvals=vals)
    else:
        keep = vals != 0
        col = np.arange(n)[:, None] + offs + 1
        rp = np.concatenate([[1], 1 + np.cumsum(keep.sum(1))]).astype(np.int32)
        K = idrs_amd.crs_format(n, n, rp, col[keep].astype(np.int32), rval=vals[keep])
        K.set_group(1)
    A = idrs_amd.Matrix(K, which_precon=1 if scaled else 0)
    V = rng.uniform(-1, 1, (n, 11))
    V[0, 0], V[n // 2, 1], V[n - 1, 2] = np.inf, np.nan, -0.0
    assert A.rowcode()[0] is None
    # the reference's values: K, or K D^-1 scaled on the host (the same
    # divisions), as a matrix of its own that is never coded
    ref = vals / vals[:, 3][np.clip(np.arange(n)[:, None] + offs, 0, n - 1)] if scaled else vals
    if fmt == "dia":
        R = idrs_amd.dia_format(n, n, offs, rvals=ref)
    else:
        R = idrs_amd.crs_format(n, n, rp, col[keep].astype(np.int32), rval=ref[keep])
        R.set_group(1)
    want = [R * V[:, j] for j in range(11)]
    W = A * V
    for j in range(11):
        assert np.array_equal(W[:, j], want[j], equal_nan=True)
    idrs_amd.idrs(A, rng.uniform(-1, 1, n), 4, maximum_iterations=1)
    # the code is built where at most 256 rows are distinct
    i = np.arange(n)[:, None]
    there = keep if fmt == "crs" else (i + offs >= 0) & (i + offs < n)
    distinct = len(np.unique(np.concatenate([there, np.where(there, ref, 0.0)], axis=1), axis=0))
    if distinct <= 256:
        assert A.rowcode() == ("values", distinct)
    else:
        assert A.rowcode() == (("offsets", 27) if fmt == "crs" else (None, 0))
    assert distinct <= 256 or kinds > 9 or scaled
    W = A * V
    for j in range(11):
        assert np.array_equal(A * V[:, j], want[j], equal_nan=True)
        assert np.array_equal(W[:, j], want[j], equal_nan=True)
    # the epilogues (P^T y, the omega dots) through a solve, and the true
    # residual it reports
    b = rng.uniform(-1, 1, n)
    r = idrs_amd.idrs(A, b, 4, tolerance=1e-9, maximum_iterations=400)
    true = np.linalg.norm(b - R * r.x) / np.linalg.norm(b)
    assert r.flag == 0 and abs(true - r.relres) <= 1e-12


def _stencil(shape, reach):
    """Offsets and values (zero outside the box) of a stencil in 1, 2 or 3
    dimensions; reach "star" or "box" (all neighbours)."""
    n, stride, pos, st = int(np.prod(shape)), [], [], 1
    i = np.arange(n)
    for m in shape:
        stride.append(st)
        pos.append((i // st) % m)
        st *= m
    cols = {}
    for d in np.ndindex(*[3] * len(shape)):
        d = np.array(d) - 1
        if reach == "star" and np.abs(d).sum() > 1:
            continue
        inside = np.ones(n, dtype=bool)
        for k, m in enumerate(shape):
            inside &= (pos[k] + d[k] >= 0) & (pos[k] + d[k] < m)
        o = int(sum(dk * sk for dk, sk in zip(d, stride)))
        cols[o] = np.where(inside, 3.0 * len(shape) + 6.0 if o == 0 else -1.0 + 0.01 * o / stride[-1], 0.0)
    offs = np.array(sorted(cols), dtype=np.int32)
    return n, offs, np.stack([cols[o] for o in offs], axis=1)


def _matrix(n, offs, vals, fmt):
    if fmt == "dia":
        return idrs_amd.dia_format(n, n, offs, rvals=vals)
    keep = vals != 0
    col = np.arange(n)[:, None] + offs + 1
    rp = np.concatenate([[1], 1 + np.cumsum(keep.sum(1))]).astype(np.int32)
    K = idrs_amd.crs_format(n, n, rp, col[keep].astype(np.int32), rval=vals[keep])
    K.set_group(1)
    return K


# every width the kernels are compiled for (3, 5, 7 and any: 9, 27), every
# shadow width of the P^T y epilogue, with and without a seed shift (s = 8:
# scaled values, whose shift is divided by the diagonal)
@pytest.mark.parametrize("shape,reach", [((40000,), "star"), ((211, 190), "star"), ((34, 33, 32), "star"),
                                         ((211, 190), "box"), ((34, 33, 32), "box")])
@pytest.mark.parametrize("fmt", ["dia", "crs"])
@pytest.mark.parametrize("s,variant,seed", [(1, 1, 0.0), (2, 1, 0.0), (4, 1, 0.3), (8, 1, 0.0), (8, 1, 0.3),
                                            (16, 1, 0.0), (1, 2, 0.0)])
def test_coded_solves_are_the_same_bits(gpu, shape, reach, fmt, s, variant, seed):
    n, offs, vals = _stencil(shape, reach)
    A = idrs_amd.Matrix(_matrix(n, offs, vals, fmt), which_precon=1 if s == 8 else 0)
    if seed:
        A.set_seed(seed)
    b, v = _b(n, 3), np.random.default_rng(2).uniform(-1, 1, n)
    lib = _lib.load()
    w = _solve(lib.idrs_idrs_f64_noalloc, A, b, s, 0.0, 2 * s + 5, variant=variant)
    Av = A * v
    assert A.rowcode()[0] is None
    g = _solve(lib.idrs_idrs_f64, A, b, s, 0.0, 2 * s + 5, variant=variant)
    kind, distinct = A.rowcode()   # a stored diagonal that leaves the matrix makes a row of its own
    assert kind == "values" and (fmt == "dia" or distinct == 3 ** len(shape))
    assert g[1:4] == w[1:4] and np.array_equal(g[0], w[0]) and np.array_equal(g[4], w[4])
    assert np.array_equal(A * v, Av)
    w = _solve(lib.idrs_idrs_f64_noalloc, A, b, s, 0.0, 2 * s + 5, variant=variant)   # now coded
    assert np.array_equal(g[0], w[0]) and np.array_equal(g[4], w[4])


def _set_values(K, val):
    val = np.ascontiguousarray(val)
    idrs_amd._lib.check(_lib.load().idrs_user_matrix_set_values_f64(K.handle, ctypes.c_void_p(val.ctypes.data), 0))


@pytest.mark.parametrize("scaled", [False, True])
def test_new_values_drop_the_code(gpu, scaled):
    n, offs, vals = _stencil((34, 33, 32), "star")
    K = _matrix(n, offs, vals, "crs")
    A = idrs_amd.Matrix(K, which_precon=1 if scaled else 0)
    b, v = _b(n, 3), np.random.default_rng(2).uniform(-1, 1, n)
    idrs_amd.idrs(A, b, 4, tolerance=0.0, maximum_iterations=5)
    assert A.rowcode() == ("values", 27)
    _set_values(K, 2.0 * vals[vals != 0])
    assert np.array_equal(K * v, _matrix(n, offs, 2.0 * vals, "crs") * v)
    if scaled:
        A.set_precon(1)
    x = idrs_amd.idrs(A, b, 4, tolerance=0.0, maximum_iterations=5).x
    # a scaled operator looks again while it finds a code
    assert A.rowcode() == ("values" if scaled else "offsets", 27)
    R = idrs_amd.Matrix(_matrix(n, offs, 2.0 * vals, "crs"), which_precon=1 if scaled else 0)
    assert np.array_equal(idrs_amd.idrs(R, b, 4, tolerance=0.0, maximum_iterations=5).x.cpu(), x.cpu())
    assert R.rowcode() == ("values", 27) and np.array_equal(A * v, R * v)
    # values that do not repeat, and then constant ones again: no more searches
    varied = vals * np.random.default_rng(5).uniform(1, 2, n)[:, None]
    for new in (varied, vals):
        _set_values(K, new[vals != 0])
        if scaled:
            A.set_precon(1)
        x = idrs_amd.idrs(A, b, 4, tolerance=0.0, maximum_iterations=5).x
        assert A.rowcode() == ("offsets", 27)
        R = idrs_amd.Matrix(_matrix(n, offs, new, "crs"), which_precon=1 if scaled else 0)
        assert np.array_equal(idrs_amd.idrs(R, b, 4, tolerance=0.0, maximum_iterations=5).x.cpu(), x.cpu())


@pytest.mark.parametrize("scaled", [False, True])
def test_coded_single_precision_values(gpu, scaled):
    """The mixed solve's FP32-value products: coded, against a matrix that
    holds the same values after others in which no code was found (its
    offsets, coded, serve FP64 values only)."""
    n, offs, vals = _stencil((34, 33, 32), "star")
    vals = vals / 3.0
    K, K1 = _matrix(n, offs, vals, "crs"), _matrix(n, offs, vals, "crs")
    b = np.random.default_rng(4).uniform(-1, 1, n)
    A, A1 = (idrs_amd.Matrix(k, which_precon=1 if scaled else 0) for k in (K, K1))
    for new in (vals * np.random.default_rng(5).uniform(1, 2, n)[:, None], vals):
        _set_values(K1, new[vals != 0])
        if scaled:
            A1.set_precon(1)
        idrs_amd.idrs(A1, b, 4, maximum_iterations=1)
    x, x1 = (idrs_amd.idrs_mixed(a, b, 4, tolerance=1e-9) for a in (A, A1))
    assert A.rowcode() == ("values", 27) and A1.rowcode() == ("offsets", 27)
    assert x.flag == 0 and (x.iterations, x.outer) == (x1.iterations, x1.outer) and np.array_equal(x.x, x1.x)


def test_many_products_look_for_a_code(gpu):
    n, offs, vals = _stencil((34, 33, 32), "star")
    A = idrs_amd.Matrix(_matrix(n, offs, vals, "dia"))
    V = np.random.default_rng(2).uniform(-1, 1, (n, 21))
    before = A * V
    for _ in range(2):
        assert np.array_equal(A * V, before) and A.rowcode()[0] is None      # 42, 63 products
    assert np.array_equal(A * V[:, 0], before[:, 0]) and A.rowcode() == ("values", 27)
    assert np.array_equal(A * V, before)


def test_complex_vectors_look_for_no_code(gpu):
    n, offs, vals = _stencil((34, 33, 32), "star")
    A = idrs_amd.Matrix(_matrix(n, offs, vals, "dia"))
    idrs_amd.idrs(A, _b(n, 3) + 0j, 4, maximum_iterations=3)
    assert A.rowcode()[0] is None


def test_lanes_per_row_keep_no_code(gpu):
    """A layout whose products cannot use the codes gives their memory back,
    and going back to the sliced copy finds them again."""
    n, offs, vals = _stencil((64, 33, 32), "star")
    K = _matrix(n, offs, vals, "crs")
    A = idrs_amd.Matrix(K)
    b = _b(n, 3)
    idrs_amd.idrs(A, b, 2, maximum_iterations=3)
    assert A.rowcode() == ("values", 27)
    idrs_amd.release_pool()
    K.set_group(4)
    assert A.rowcode() == (None, 0) and idrs_amd.release_pool() >= n     # a byte a row
    K.set_group(1)
    idrs_amd.idrs(A, b, 2, maximum_iterations=3)
    assert A.rowcode() == ("values", 27)
