"""Row-coded products (a byte per row and a table of the distinct rows)
against the uncoded products of the same matrices, bit for bit: the same
operations on the same values in the same order.  A user matrix's own product
does not look for the code, an operator's does.
"""
import numpy as np
import pytest

import idrs_amd
from idrs_amd import problems as P

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
        assert np.array_equal(A * V[:, j], want[j], equal_nan=True)
        assert np.array_equal(W[:, j], want[j], equal_nan=True)
    # the epilogues (P^T y, the omega dots) through a solve, and the true
    # residual it reports
    b = rng.uniform(-1, 1, n)
    r = idrs_amd.idrs(A, b, 4, tolerance=1e-9, maximum_iterations=400)
    true = np.linalg.norm(b - R * r.x) / np.linalg.norm(b)
    assert r.flag == 0 and abs(true - r.relres) <= 1e-12
