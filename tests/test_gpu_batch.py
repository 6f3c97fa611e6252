"""GPU parity of the batched IDR(s) solve (idrs_idrs_batched_*): every system
of a batch must behave as its own IDRS solve (MODULES/IDRS/idrs.inc) on the
oracle, with the same default shadow-space stream per system.

Bar (FP64): at the convergence tolerance each system's flag equals the
oracle's and its iteration count is within +-2; at an equal, fixed
iteration count each system's solution agrees within 1e-10 relative.
Systems that finish early stay frozen while the others continue.
"""
import numpy as np
import pytest

import idrs_amd
import orc
from idrs_amd import problems as P

from helpers import oracle_crs, rel, rounding_spread

pytestmark = pytest.mark.gpu


def _systems(specs, seed=0):
    """2-D 5-point convection-diffusion systems (m, Pe, angle) and random b."""
    rng = np.random.default_rng(seed)
    out = []
    for m, pe, ang in specs:
        crs, _ = P.convection_diffusion_2d(m, pe, angle=ang)
        out.append((crs, rng.uniform(-1.0, 1.0, crs.n)))
    return out


def _batch(systems, diag_precon=False, poly=None):
    Ks = [idrs_amd.crs_format(c.n, c.n, c.row_ptr, c.col_ind, rval=c.val) for c, _ in systems]
    KB = idrs_amd.batch_format(Ks)
    A = idrs_amd.Matrix(KB)
    if diag_precon:
        A.set_precon(1)
    if poly is not None:
        kind, degree, foci = poly
        idrs_amd.real_preconditioner(A, kind, degree, foci=foci)
    b = np.concatenate([bb for _, bb in systems])
    return A, b


# Batches whose systems all have at most 4096 rows run each in one workgroup;
# with one larger system every system runs on the tile kernels.
LARGER = [(65, 20.0, 0.9)]
PATHS = pytest.mark.parametrize("path", ["workgroup", "tiles"])


def _more(specs, path):
    return specs + (LARGER if path == "tiles" else [])


SPECS = [(5, 1.0, 0.3), (9, 30.0, 1.1), (17, 5.0, 2.0), (33, 80.0, 4.0), (40, 12.0, 5.5), (12, 60.0, 0.7)]


def test_batch_partition(gpu):
    systems = _systems(SPECS)
    A, b = _batch(systems)
    nsys, row0 = idrs_amd.batch_info(A.K)
    assert nsys == len(SPECS)
    assert list(np.diff(row0)) == [c.n for c, _ in systems]
    # the block-diagonal product is every system's own product
    v = np.random.default_rng(1).standard_normal(row0[-1])
    w = A.K * v
    for k, (c, _) in enumerate(systems):
        assert np.allclose(w[row0[k]:row0[k + 1]], c.matvec(v[row0[k]:row0[k + 1]]), rtol=1e-13, atol=1e-10)


@PATHS
@pytest.mark.parametrize("s,variant", [(2, 1), (4, 1), (1, 2)])
def test_batch_matches_single_solves(gpu, s, variant, path):
    systems = _systems(_more(SPECS, path))
    A, b = _batch(systems)
    _, row0 = idrs_amd.batch_info(A.K)
    r = idrs_amd.idrs_batched(A, b, s, tolerance=1e-8, maximum_iterations=3000, variant=variant)
    assert idrs_amd.last_solve_path() == path
    for k, (c, bb) in enumerate(systems):
        Ao = oracle_crs(c)
        xo, fo, ro, io, _ = orc.idrs(Ao, bb, s, tolerance=1e-8, maximum_iterations=3000, variant=variant)
        xk = r.x[row0[k]:row0[k + 1]]
        print(f"sys {k} n={c.n}: batch it={r.iterations[k]} flag={r.flag[k]}  oracle it={io} flag={fo}")
        slack = 2
        if abs(r.iterations[k] - io) > 2:
            # BiCGSTAB's count can move by more than 2 under rounding alone:
            # allow what the oracle itself shows under 1e-16 perturbations of b
            _, dit = rounding_spread(lambda bp: (lambda o: (o[0], o[3]))(
                orc.idrs(Ao, bp, s, tolerance=1e-8, maximum_iterations=3000, variant=variant)), bb)
            slack = max(2, dit)
        assert r.flag[k] == fo == 0 and abs(r.iterations[k] - io) <= slack
        assert r.relres[k] <= 1e-8
        assert np.linalg.norm(bb - c.matvec(xk)) <= 1.01e-8 * np.linalg.norm(bb)
    # equal fixed iteration count: every system's iterate
    g = idrs_amd.idrs_batched(A, b, s, tolerance=0.0, maximum_iterations=14, variant=variant)
    assert np.all(g.iterations == 14) and np.all(g.flag == 1)
    for k, (c, bb) in enumerate(systems):
        Ao = oracle_crs(c)

        def run(bp):
            o = orc.idrs(Ao, bp, s, tolerance=0.0, maximum_iterations=14, variant=variant)
            return o[0], o[3]

        d = rel(g.x[row0[k]:row0[k + 1]], run(bb)[0])
        if d >= 1e-10:
            dx, _ = rounding_spread(run, bb)
            assert d < max(1e-10, 100 * dx), (k, d, dx)


@PATHS
def test_batch_chebyshev_and_scaling(gpu, path):
    """Diagonal scaling and a Chebyshev polynomial on every system (the
    pp_idrs operator), against the oracle's per-system operator."""
    systems = _systems(_more(SPECS[:4], path), seed=3)
    poly = (2, 4, (0.15, 1.85))
    A, b = _batch(systems, diag_precon=True, poly=poly)
    _, row0 = idrs_amd.batch_info(A.K)
    g = idrs_amd.idrs_batched(A, b, 4, tolerance=0.0, maximum_iterations=10)
    assert idrs_amd.last_solve_path() == path
    for k, (c, bb) in enumerate(systems):
        Ao = oracle_crs(c, diag_precon=True, poly=poly)

        def run(bp):
            o = orc.idrs(Ao, bp, 4, tolerance=0.0, maximum_iterations=10)
            return o[0], o[3]

        xo = run(bb)[0]
        d = rel(g.x[row0[k]:row0[k + 1]], xo)
        if d >= 1e-10:
            # this operator amplifies rounding (one system moves by ~4e-9
            # under a 1e-16 perturbation of b on the oracle alone)
            dx, _ = rounding_spread(run, bb)
            assert d < max(1e-10, 100 * dx), (k, d, dx)


@PATHS
def test_batch_x0_pt_raw_and_device(gpu, path):
    import torch

    systems = _systems(_more(SPECS[:3], path), seed=5)
    A, b = _batch(systems)
    _, row0 = idrs_amd.batch_info(A.K)
    rng = np.random.default_rng(6)
    x0 = rng.standard_normal(row0[-1])
    PT = rng.standard_normal((row0[-1], 2))
    h = idrs_amd.idrs_batched(A, b, 2, tolerance=0.0, maximum_iterations=9, x0=x0, PT_raw=PT)
    assert idrs_amd.last_solve_path() == path
    for k, (c, bb) in enumerate(systems):
        sl = slice(row0[k], row0[k + 1])
        xo = orc.idrs(oracle_crs(c), bb, 2, tolerance=0.0, maximum_iterations=9, x0=x0[sl], PT_raw=PT[sl])[0]
        assert rel(h.x[sl], xo) < 1e-10
    dev = torch.device("cuda:0")
    d = idrs_amd.idrs_batched(A, torch.from_numpy(b).to(dev), 2, tolerance=0.0, maximum_iterations=9,
                              x0=torch.from_numpy(x0).to(dev), PT_raw=torch.from_numpy(PT).to(dev))
    assert rel(d.x.cpu().numpy(), h.x) < 1e-14


@PATHS
def test_batch_frozen_systems(gpu, path):
    """One easy and one hard system: the easy one stops at its own count and
    its solution stays what its own solve returns."""
    systems = _systems([(6, 0.0, 0.0), (48 if path == "workgroup" else 66, 90.0, 0.4)], seed=8)
    A, b = _batch(systems)
    _, row0 = idrs_amd.batch_info(A.K)
    r = idrs_amd.idrs_batched(A, b, 2, tolerance=1e-10, maximum_iterations=4000)
    assert idrs_amd.last_solve_path() == path
    its = []
    for k, (c, bb) in enumerate(systems):
        xo, fo, ro, io, _ = orc.idrs(oracle_crs(c), bb, 2, tolerance=1e-10, maximum_iterations=4000)
        its.append(io)
        assert r.flag[k] == fo == 0 and abs(r.iterations[k] - io) <= 2
        assert rel(r.x[row0[k]:row0[k + 1]], xo) < 1e-8
    assert its[0] < its[1]


@pytest.mark.parametrize("poly", [None, (2, 4, [0.2, 1.8])])
def test_batch_graph_replay_is_bit_identical(gpu, poly):
    """Graph replay (recaptured after each drop of finished systems' tiles)
    against eager launches: 40 systems that finish at different counts, so
    the tile lists shrink several times; every output is bit-identical."""
    rng = np.random.default_rng(11)
    specs = [(int(m), float(pe), float(a)) for m, pe, a in
             zip(rng.integers(4, 70, 40), rng.uniform(0.0, 90.0, 40), rng.uniform(0, 6.28, 40))]
    systems = _systems(specs, seed=5)
    A, b = _batch(systems, diag_precon=poly is not None, poly=poly)
    kw = dict(tolerance=1e-9, maximum_iterations=3000)
    e = idrs_amd.idrs_batched(A, b, 2, graph=False, **kw)
    g = idrs_amd.idrs_batched(A, b, 2, graph=True, **kw)
    assert idrs_amd.last_solve_path() == "tiles"
    print("iterations", sorted(set(e.iterations.tolist())))
    assert len(set(e.iterations.tolist())) >= 8
    assert np.array_equal(e.iterations, g.iterations) and np.array_equal(e.flag, g.flag)
    # systems that break down (flag 2 on two of the Chebyshev systems) are
    # compared too; equal_nan covers a breakdown's NaN
    assert np.array_equal(e.relres, g.relres, equal_nan=True)
    assert np.array_equal(e.x, g.x, equal_nan=True)


@PATHS
def test_batch_sliced_copy(gpu, path):
    """The batch's tile product on the sliced-ELL copy (group 1; tiles start
    mid-slice at system boundaries) against each system's oracle solve."""
    systems = _systems(_more(SPECS, path))
    A, b = _batch(systems)
    A.K.set_group(1)
    _, row0 = idrs_amd.batch_info(A.K)
    r = idrs_amd.idrs_batched(A, b, 2, tolerance=1e-8, maximum_iterations=3000)
    assert idrs_amd.last_solve_path() == path
    for k, (c, bb) in enumerate(systems):
        xo, fo, ro, io, _ = orc.idrs(oracle_crs(c), bb, 2, tolerance=1e-8, maximum_iterations=3000)
        assert r.flag[k] == fo == 0 and abs(r.iterations[k] - io) <= 2, (k, r.iterations[k], io)
        assert np.linalg.norm(bb - c.matvec(r.x[row0[k]:row0[k + 1]])) <= 1.01e-8 * np.linalg.norm(bb)
    g = idrs_amd.idrs_batched(A, b, 2, tolerance=0.0, maximum_iterations=14)
    for k, (c, bb) in enumerate(systems):
        xo = orc.idrs(oracle_crs(c), bb, 2, tolerance=0.0, maximum_iterations=14)[0]
        assert rel(g.x[row0[k]:row0[k + 1]], xo) < 1e-10, k


def test_batch_rejects(gpu):
    crs, _ = P.convection_diffusion_2d(6, 1.0)
    K = idrs_amd.crs_format(crs.n, crs.n, crs.row_ptr, crs.col_ind, rval=crs.val)
    with pytest.raises(ValueError):
        idrs_amd.idrs_batched(idrs_amd.Matrix(K), np.ones(crs.n), 2)
    A, b = _batch(_systems(SPECS[:2]))
    with pytest.raises(idrs_amd.IdrsError):
        idrs_amd.idrs_batched(A, b, 0)


@pytest.mark.parametrize("layout", ["lanes", "sliced"])
def test_batch_mixed_precision(gpu, layout):
    """Batched mixed precision (idrs_idrs_batched_mixed_f64), plain and with
    diagonal scaling on the sliced copy: every system
    meets the FP64 tolerance on its own true residual, recomputed here in
    FP64 from the returned x by the oracle's operator; the solutions agree with the oracle's FP64
    solves to the accuracy the tolerance allows; a zero right-hand side
    finishes at once with x = 0."""
    systems = _systems(SPECS, seed=7)
    systems[2] = (systems[2][0], np.zeros(systems[2][0].n))
    scaled = layout == "sliced"
    A, b = _batch(systems, diag_precon=scaled)
    if layout == "sliced":
        A.K.set_group(1)
    tol = 1e-8
    r = idrs_amd.idrs_batched_mixed(A, b, 4, tolerance=tol, inner_tolerance=1e-5)
    _, row0 = idrs_amd.batch_info(A.K)
    assert list(r.flag) == [0] * len(SPECS)
    for k, (c, bk) in enumerate(systems):
        xk = r.x[row0[k]:row0[k + 1]]
        if not bk.any():
            assert not xk.any() and r.outer[k] == 0
            continue
        # the operator's residual (with scaling, A = K D^-1)
        Ao = oracle_crs(c, diag_precon=scaled)
        res = np.linalg.norm(bk - Ao.matvec(xk)) / np.linalg.norm(bk)
        assert res <= tol * (1 + 1e-6), (k, res)
        assert abs(res - r.relres[k]) <= 1e-12 + 1e-6 * res
        assert r.outer[k] >= 1 and r.iterations[k] > 0
        xo = orc.idrs(Ao, bk, 4, tolerance=1e-12, maximum_iterations=5000)[0]
        assert rel(xk, xo) < 1e-4, k
    # device vectors give the same result
    import torch

    bd = torch.from_numpy(b).to("cuda:0")
    rd = idrs_amd.idrs_batched_mixed(A, bd, 4, tolerance=tol, inner_tolerance=1e-5)
    assert np.array_equal(rd.x.cpu().numpy(), r.x)
    # options the scheme does not offer
    with pytest.raises(idrs_amd.IdrsError):
        idrs_amd.idrs_batched_mixed(A, b, 4, tolerance=tol, inner_tolerance=2.0)
