"""The folded IDR(s) cycle (reductions and scalar steps inside the streaming
kernels, up to 3 * 2^16 rows) against the allocation-free entry, which always runs
them as kernels of their own: the same sums in the same order, so x, the flag,
the count, relres and the residual history are the same bits -- for shadow
spaces on both sides of the kernel's 4-column form, stops at every step of a
cycle, the omega step's user values, M1, and the largest folded system.
"""
import ctypes

import numpy as np
import pytest

import idrs_amd
import orc
from helpers import gpu_crs, oracle_crs, rel
from idrs_amd import _lib
from idrs_amd import problems as P

pytestmark = pytest.mark.gpu


def _solve(f, A, b, s, tol, maxit, variant=1, M1=None, omega=None):
    import torch

    x = torch.full_like(b, np.nan)
    rv = np.zeros(maxit + 1)
    o = _lib.idrs_opts_t()
    o.has_tolerance, o.tolerance = 1, tol
    o.has_maximum_iterations, o.maximum_iterations = 1, maxit
    o.has_variant, o.variant = 1, variant
    o.device_pointers = 1
    o.resvec, o.resvec_len = rv.ctypes.data, len(rv)
    if M1 is not None:
        o.has_M1, o.M1 = 1, M1.handle
    if omega is not None:
        o.omega, o.n_omega = omega.ctypes.data, len(omega)
    st = _lib.idrs_stats_t()
    torch.cuda.synchronize()
    rc = f(A.handle, int(b.shape[0]), ctypes.c_void_p(b.data_ptr()), s, ctypes.byref(o), ctypes.c_void_p(x.data_ptr()),
           ctypes.byref(st))
    assert rc == 0, _lib.load().idrs_last_error().decode()
    return x.cpu().numpy(), st.flag, st.iterations, st.relres, rv[: st.iterations + 1]


def _same(A, b, s, tol, maxit, path="folded", **kw):
    lib = _lib.load()
    g = _solve(lib.idrs_idrs_f64, A, b, s, tol, maxit, **kw)
    assert idrs_amd.last_solve_path() == path
    w = _solve(lib.idrs_idrs_f64_noalloc, A, b, s, tol, maxit, **kw)
    assert idrs_amd.last_solve_path() == "launches"
    assert g[1:4] == w[1:4]
    assert np.array_equal(g[0], w[0]) and np.array_equal(g[4], w[4])
    return g


def _b(n, seed=1):
    import torch

    return torch.tensor(np.random.default_rng(seed).uniform(-1, 1, n), device="cuda:0")


@pytest.mark.parametrize("s", [1, 2, 3, 4, 5, 8, 16])
def test_folded_cycle_is_the_same_bits(gpu, s):
    crs, _ = P.convection_diffusion_3d(14, 8.0, reaction=1.0)     # 2744 rows
    A = idrs_amd.Matrix(idrs_amd.crs_format(crs.n, crs.n, crs.row_ptr, crs.col_ind, rval=crs.val))
    b = _b(crs.n)
    assert _same(A, b, s, 1e-9, 800)[1] == 0
    for maxit in range(1, s + 4):        # a stop at every step of the first cycles
        assert _same(A, b, s, 0.0, maxit)[1:3] == (1, maxit)


def test_folded_cycle_options(gpu):
    crs, dia = P.convection_diffusion_3d(20, 12.0, reaction=1.0)
    K = idrs_amd.dia_format(crs.n, crs.n, dia.offsets, rvals=dia.vals)
    A, b = idrs_amd.Matrix(K), _b(crs.n, 2)
    _same(A, b, 4, 1e-9, 800, M1=idrs_amd.Matrix(K, which_precon=1))
    _same(A, b, 1, 1e-9, 900, variant=2)
    _same(A, b, 4, 0.0, 37, omega=np.array([0.9, 1.1, 0.7]))
    P8 = idrs_amd.Matrix(K, which_precon=1)
    idrs_amd.real_preconditioner(P8, 2, 8, foci=(0.15, 1.85))
    _same(P8, b, 6, 1e-10, 300)


@pytest.mark.parametrize("n", [3 << 16, (3 << 16) + 1, 1 << 18, (1 << 18) + 1])
def test_largest_folded_system(gpu, n):
    crs, _, _ = P.toeplitz_1d(n)
    K = idrs_amd.crs_format(n, n, crs.row_ptr, crs.col_ind, rval=crs.val)
    K.set_group(1)          # one thread per row: a partial per 256 rows
    _same(idrs_amd.Matrix(K), _b(n, 3), 2, 0.0, 8, path="folded" if n <= 3 << 16 else "launches")


@pytest.mark.parametrize("n", [163840, 163841 + 1024])
def test_largest_folded_product_grid(gpu, n):
    """Eight lanes per row: 128 rows a partial, 1280 partials the most folded."""
    crs, _, _ = P.toeplitz_1d(n)
    K = idrs_amd.crs_format(n, n, crs.row_ptr, crs.col_ind, rval=crs.val)
    K.set_group(8)
    _same(idrs_amd.Matrix(K), _b(n, 4), 3, 0.0, 9, path="folded" if n <= 163840 else "launches")


# complex vectors in each form of the solve, every shadow space and option,
# against the oracle at a fixed count (1e-10, the bar of the other solves; the
# Hessenberg matrix 1e-9 of its largest entry)
@pytest.mark.parametrize("m,path", [(10, "workgroup"), (16, "folded"), (60, "launches")])
@pytest.mark.parametrize("s,variant,extra", [(4, 1, "x0 U0"), (8, 1, "H"), (4, 1, "M1 omega"), (1, 2, "M1"), (1, 3, ""),
                                             (1, 4, "x0"), (16, 1, "")])
def test_complex_solves_match_oracle(gpu, m, path, s, variant, extra):
    crs, _ = P.convection_diffusion_3d(m, 10.0, reaction=1.0)
    crs.val = crs.val * (1.0 + 0.2j)
    n, rng = crs.n, np.random.default_rng(s)
    rand = lambda *shape: rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    A, Ao, b = gpu_crs(crs), oracle_crs(crs), rand(n)
    kw = dict(tolerance=0.0, maximum_iterations=14, variant=variant)
    okw = dict(kw)
    if "x0" in extra:
        kw["x0"] = okw["x0"] = rand(n)
    if "U0" in extra:
        kw["U0"] = okw["U0"] = rand(n, s)
    if "omega" in extra:
        kw["omega"] = okw["omega"] = np.array([0.9 + 0.1j, 1.1 - 0.2j])
    if "M1" in extra:
        kw["M1"], okw["M1"] = gpu_crs(crs, diag_precon=True), oracle_crs(crs, diag_precon=True)
    if "H" in extra:
        kw["H"] = okw["H_nritz"] = 13
    g = idrs_amd.idrs(A, b, s, **kw)
    assert idrs_amd.last_solve_path() == path
    o = orc.idrs(Ao, b, s, **okw)
    assert (g.flag, g.iterations) == (o[1], o[3]) and rel(g.x, o[0]) < 1e-10
    if "H" in extra:
        assert np.abs(g.H - o[5]).max() <= 1e-9 * np.abs(o[5]).max()


@pytest.mark.parametrize("k", [1, 5, 6, 23, 24, 70])
def test_pattern_gradient_lanes(gpu, k):
    """-lambda_i x_j on the pattern for row lengths on both sides of the
    lanes-per-row lines, exactly."""
    import torch

    crs = P.random_dominant(1003, k=k, seed=k)
    system = idrs_amd.SparseSystem(crs.n, crs.row_ptr, crs.col_ind, crs.val)
    lam, x = _b(crs.n, 4), _b(crs.n, 5)
    out = torch.full((crs.nnz,), np.nan, dtype=torch.float64, device="cuda:0")
    system.pattern_grad(lam, x, out)
    rows = np.repeat(np.arange(crs.n), np.diff(crs.row_ptr))
    assert np.array_equal(out.cpu().numpy(), -(lam.cpu().numpy()[rows] * x.cpu().numpy()[crs.col_ind - 1]))
