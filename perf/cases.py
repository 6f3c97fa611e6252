"""Performance cases of the IDR(s) library: the solves its users run, through
the public Python entry points, from the smallest systems (latency) to the
200^3 headline workload (HBM bandwidth).

Every case builds a sparse system from seeded random data, picks a known
solution x (1 + uniform noise), forms b = K x in float64 and solves for x to a
residual tight enough that the solution itself is good to 1e-9 (the largest
boxes, where rounding bounds the solution first, run a fixed number of
iterations instead).  A pass is a whole solve (with the scale-back of the polynomial preconditioner where one
is used) on device-resident vectors; the matrix handle, its layout and its
preconditioner are what a program keeps between solves.

Kinds:
  solve     IDR(s) on 3-D 7-point convection-diffusion boxes: CRS or offset-list
            diagonal storage, plain or with diagonal scaling and a Chebyshev
            polynomial, constant or variable coefficients, real or complex.
  mixed     the same systems by FP32 inner solves with FP64 residuals.
  shifts    16 shifted Laplacian systems by MSQMRIDR(s) / MSIDRS(s) with the
            per-shift scale-back.
  batch     many independent 2-D systems of uneven size at once.
  adjoint   a differentiable solve through torch autograd: forward, adjoint
            and the gradient on the sparsity pattern (random sparse systems).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "idrs-package_amd"))

import idrs_amd  # noqa: E402

FOCI = (0.15, 1.85)          # spectrum of the diagonally scaled operators
SHIFT_FOCI = (0.05, 11.95)   # spectrum of the h^2-scaled Laplacian


def listed():
    return [
        # the smallest solve: a 12^3 box, one call's latency
        _solve("solve-12cube-crs", 12, 12, 12, "crs", s=4, degree=0, pe=10.0),
        # the reference's own CPU-sized example: plain IDR(4) on 32^3
        _solve("solve-32cube-crs", 32, 32, 32, "crs", s=4, degree=0, pe=10.0),
        # an odd-sized box in diagonal storage with variable diffusion and
        # the Chebyshev preconditioner
        _solve("solve-61x47x53-dia-var", 61, 47, 53, "dia", s=4, degree=8, pe=20.0, variable=True),
        # complex values and vectors (a damped wave operator), CRS
        _solve("solve-41x37x43-complex", 41, 37, 43, "crs", s=4, degree=0, pe=0.0, cplx=True),
        # a million rows with variable diffusion, CRS with a tuned layout, s = 8
        _solve("solve-101x97x103-crs-var", 101, 97, 103, "crs", s=8, degree=8, pe=40.0, variable=True, tune=True),
        # two million rows, constant coefficients, CRS with a tuned layout
        _solve("solve-128cube-crs", 128, 128, 128, "crs", s=4, degree=8, pe=50.0, tune=True),
        # the headline workload: 200^3 in diagonal storage, IDR(4) + Chebyshev(8)
        _solve("solve-200cube-dia", 200, 200, 200, "dia", s=4, degree=8, pe=50.0),
        # single-precision inner solves, FP64 residuals
        dict(_solve("mixed-120x128x111-dia", 120, 128, 111, "dia", s=4, degree=8, pe=50.0), kind="mixed", budget=0),
        # 16 shifts sharing one Krylov space
        dict(name="shifts-64x60x62-msqmridr", kind="shifts", nx=64, ny=60, nz=62, s=8, solver="msqmridr", nshift=16,
             degree=8, tol=1e-11),
        # a batch of small uneven systems (24^2 to 64^2 rows)
        dict(name="batch-256-small", kind="batch", nsys=256, lo=24, hi=64, s=2, tol=1e-12),
        # a batch of larger uneven systems (64^2 to 180^2 rows)
        dict(name="batch-96-large", kind="batch", nsys=96, lo=64, hi=180, s=2, tol=1e-12),
        # the differentiable solve: forward, adjoint and pattern gradient
        dict(name="adjoint-1e6", kind="adjoint", n=1_000_000, k=16, s=4, tol=1e-11),
    ]


def _solve(name, nx, ny, nz, storage, s, degree, pe, variable=False, cplx=False, tune=False):
    # budget: above a side of 110 the pass is 25 iterations (a time step's
    # budget), below it a solve to the tolerance
    return dict(name=name, kind="solve", nx=nx, ny=ny, nz=nz, storage=storage, s=s, degree=degree, pe=pe,
                variable=variable, cplx=cplx, tune=tune, tol=1e-12, budget=25 if max(nx, ny, nz) > 110 else 0)


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "solve", "mixed", "shifts", "batch", "batch", "adjoint"])
    if kind in ("solve", "mixed"):
        cheb = kind == "mixed" or rng.random() < 0.6
        side = math.exp(rng.uniform(math.log(16), math.log(180))) if cheb else math.exp(
            rng.uniform(math.log(8), math.log(44)))
        if kind == "mixed":
            side = max(40.0, min(side, 140.0))
        cplx = kind == "solve" and not cheb and rng.random() < 0.25
        dims = [max(6, int(side * rng.uniform(0.85, 1.1))) for _ in range(3)]
        variable = cheb and kind == "solve" and rng.random() < 0.4
        # the polynomial's real ellipse wants a grid Peclet number well below 1
        pe = rng.uniform(1.0, min(50.0, (0.25 if variable else 0.5) * side)) if cheb else rng.uniform(1.0, 20.0)
        c = _solve("", *dims, rng.choice(["crs", "dia"]), s=rng.choice([2, 4, 4, 8]), degree=8 if cheb else 0,
                   pe=0.0 if cplx else round(pe, 2), variable=variable, cplx=cplx, tune=cheb and rng.random() < 0.5)
        c["kind"] = kind
        if kind == "mixed":
            c["budget"] = 0
        del c["name"]
        return c
    if kind == "shifts":
        side = math.exp(rng.uniform(math.log(16), math.log(100)))
        dims = [max(8, int(side * rng.uniform(0.85, 1.1))) for _ in range(3)]
        solver = rng.choice(["msqmridr", "msidrs"])
        return dict(kind="shifts", nx=dims[0], ny=dims[1], nz=dims[2], s=8 if solver == "msqmridr" else 4,
                    solver=solver, nshift=rng.choice([5, 11, 16]), degree=8, tol=1e-11)
    if kind == "batch":
        lo = rng.choice([16, 24, 33, 64])
        hi = int(lo * rng.uniform(1.3, 3.0))
        rows = (hi * hi - lo * lo) / (2 * math.log(hi / lo))
        nsys = max(3, min(512, int(math.exp(rng.uniform(math.log(1e5), math.log(1.5e6))) / rows)))
        return dict(kind="batch", nsys=nsys, lo=lo, hi=hi, s=rng.choice([2, 2, 4]), tol=1e-12)
    n = int(math.exp(rng.uniform(math.log(2e4), math.log(1e6))))
    return dict(kind="adjoint", n=n, k=rng.choice([6, 11, 16]), s=4, tol=1e-11)


# --------------------------------------------------------------------------
# systems
# --------------------------------------------------------------------------
def _gen(seed, what):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + what)


def _uniform(n, g, lo=0.0, hi=1.0):
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * (hi - lo) + lo


def _solution(n, seed, cplx=False):
    x = 1.0 + _uniform(n, _gen(seed, 1), -1.0, 1.0)
    return torch.complex(x, _uniform(n, _gen(seed, 2), -1.0, 1.0)) if cplx else x


def _box(c, seed):
    """Offsets (ascending) and (n, ndiag) values, zero outside the box, of a
    7-point convection-diffusion-reaction operator (h = 1/(side + 1)); with
    'variable' the diffusion coefficient varies smoothly and by layers, its
    phase drawn from the seed; with 'cplx' a damped wave operator
    (Laplacian - k^2 (1 - 0.5 i) h^2-scaled)."""
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    n = nx * ny * nz
    i = torch.arange(n, device="cuda")
    xyz = (i % nx, (i // nx) % ny, i // (nx * ny))
    dims, strides = (nx, ny, nz), (1, nx, nx * ny)
    # the Peclet number drawn near the case's: another seed, another matrix
    r = float(torch.rand(1, generator=_gen(seed, 3), device="cuda"))
    dt = torch.complex128 if c["cplx"] else torch.float64
    cols = {0: torch.zeros(n, device="cuda", dtype=dt)}
    if c["cplx"]:
        kh2 = (2 * math.pi / 24.0) ** 2 * (0.9 + 0.2 * r)
        cols[0] += complex(6.0 - kh2, 0.5 * kh2)
        for d in range(3):
            cols[-strides[d]] = -(xyz[d] > 0).to(dt)
            cols[strides[d]] = -(xyz[d] < dims[d] - 1).to(dt)
    else:
        h = 1.0 / (max(dims) + 1)
        pe = c["pe"] * (0.9 + 0.2 * r)
        if c["variable"]:
            u = [(q.double() + 1) / (m + 1) for q, m in zip(xyz, dims)]

            def eps(a, b, e):
                return ((1.0 + 0.5 * torch.sin(2 * math.pi * (a + r)) * torch.sin(2 * math.pi * b))
                        * torch.where(torch.sin(6 * math.pi * (e + r)) > 0, 1.0, 3.0))
        for d in range(3):
            for sgn in (-1, 1):
                inside = (xyz[d] > 0) if sgn < 0 else (xyz[d] < dims[d] - 1)
                if c["variable"]:
                    f = [q + (sgn * 0.5 / (m + 1) if k == d else 0.0) for k, (q, m) in enumerate(zip(u, dims))]
                    e = eps(*f) / h ** 2
                else:
                    e = torch.full((n,), 1.0 / h ** 2, device="cuda", dtype=torch.float64)
                cols[sgn * strides[d]] = (-e + sgn * pe / (2 * h)) * inside
                cols[0] += e
        cols[0] += 1.0
    offs = sorted(cols)
    return offs, torch.stack([cols[o] for o in offs], dim=1)


def _dia_matvec(offs, vals, x):
    n = x.shape[0]
    y = torch.zeros_like(x)
    for d, o in enumerate(offs):
        a, e = max(0, -o), min(n, n - o)
        y[a:e] += vals[a:e, d] * x[a + o:e + o]
    return y


def _user_matrix(c, offs, vals):
    n = vals.shape[0]
    key = "cvals" if c["cplx"] else "rvals"
    if c["storage"] == "dia":
        host = np.asfortranarray(vals.t().contiguous().cpu().numpy().T)
        return idrs_amd.dia_format(n, n, offs, **{key: host})
    keep = vals != 0
    col = torch.arange(n, device="cuda")[:, None] + torch.tensor(offs, device="cuda") + 1
    rp = torch.ones(n + 1, dtype=torch.int64, device="cuda")
    rp[1:] += keep.sum(1).cumsum(0)
    val = vals[keep].cpu().numpy()
    return idrs_amd.crs_format(n, n, rp.int().cpu().numpy(), col[keep].int().cpu().numpy(),
                               **{"cval" if c["cplx"] else "rval": val})


def _prepare_solve(c, seed):
    offs, vals = _box(c, seed)
    n = vals.shape[0]
    b = _dia_matvec(offs, vals, _solution(n, seed, c["cplx"]))
    K = _user_matrix(c, offs, vals)
    del vals
    if c["tune"] and c["kind"] == "solve":
        K.autotune()
    A = idrs_amd.Matrix(K)
    alpha = None
    if c["degree"]:
        A.set_precon(1)
        idrs_amd.real_preconditioner(A, 2, c["degree"], foci=FOCI)
        alpha = A.alpha.reshape(-1, 1)
    return dict(case=c, A=A, b=b, alpha=alpha)


def _run_solve(st):
    c, A, b = st["case"], st["A"], st["b"]
    if c["kind"] == "mixed":
        r = idrs_amd.idrs_mixed(A, b, c["s"], tolerance=c["tol"], maximum_iterations=5000, inner_tolerance=1e-7)
    elif c["budget"]:
        r = idrs_amd.idrs(A, b, c["s"], tolerance=0.0, maximum_iterations=c["budget"])
    else:
        r = idrs_amd.idrs(A, b, c["s"], tolerance=c["tol"], maximum_iterations=5000)
    if st["alpha"] is None:
        return r.x
    return idrs_amd.ms_scaleback(A, st["alpha"], r.x.reshape(-1, 1))[:, 0]


# --------------------------------------------------------------------------
# shifted systems (K - sigma_k I) x_k = b, K the h^2-scaled Laplacian
# --------------------------------------------------------------------------
def _shift_rhs(c, seed):
    return _uniform(c["nx"] * c["ny"] * c["nz"], _gen(seed, 4), -1.0, 1.0)


def _shifts(c, seed):
    step = 0.009 + 0.002 * float(torch.rand(1, generator=_gen(seed, 5), device="cuda"))
    return -step * np.arange(c["nshift"])


def _prepare_shifts(c, seed):
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    n = nx * ny * nz
    i = torch.arange(n, device="cuda")
    xyz, dims, strides = (i % nx, (i // nx) % ny, i // (nx * ny)), (nx, ny, nz), (1, nx, nx * ny)
    cols = {0: torch.full((n,), 6.0, device="cuda", dtype=torch.float64)}
    for d in range(3):
        cols[-strides[d]] = -(xyz[d] > 0).double()
        cols[strides[d]] = -(xyz[d] < dims[d] - 1).double()
    offs = sorted(cols)
    K = _user_matrix(dict(storage="crs", cplx=False), offs, torch.stack([cols[o] for o in offs], dim=1))
    K.autotune()
    A = idrs_amd.Matrix(K)
    idrs_amd.real_preconditioner(A, 2, c["degree"], foci=SHIFT_FOCI)
    sigma, alpha = idrs_amd.ms_parameters(A, _shifts(c, seed))
    return dict(case=c, A=A, b=_shift_rhs(c, seed), sigma=sigma, alpha=alpha)


def _run_shifts(st):
    c = st["case"]
    solver = idrs_amd.msqmridr if c["solver"] == "msqmridr" else idrs_amd.msidrs
    r = solver(st["A"], st["b"], st["sigma"], c["s"], tolerance=c["tol"], maximum_iterations=2000)
    return idrs_amd.ms_scaleback(st["A"], st["alpha"], r.x)


def _exact_shifts(c, seed):
    # sine-transform diagonalisation of the Dirichlet Laplacian
    dims = (c["nz"], c["ny"], c["nx"])
    S, lam = [], []
    for m in dims:
        k = torch.arange(1, m + 1, device="cuda", dtype=torch.float64)
        S.append(math.sqrt(2.0 / (m + 1)) * torch.sin(math.pi * torch.outer(k, k) / (m + 1)))
        lam.append(2.0 - 2.0 * torch.cos(math.pi * k / (m + 1)))

    def transform(v):
        v = (S[0] @ v.reshape(dims[0], -1)).reshape(dims)
        v = torch.stack([S[1] @ p for p in v])
        return (v.reshape(-1, dims[2]) @ S[2]).reshape(dims)
    bh = transform(_shift_rhs(c, seed).reshape(dims))
    eig = lam[0][:, None, None] + lam[1][None, :, None] + lam[2][None, None, :]
    return torch.stack([transform(bh / (eig - float(sk))).reshape(-1) for sk in _shifts(c, seed)], dim=1)


# --------------------------------------------------------------------------
# batches of 2-D 5-point convection-diffusion systems
# --------------------------------------------------------------------------
def _batch_sides(c, seed):
    # sizes fixed by the case (every seed solves the same shapes), log-uniform
    rng = np.random.default_rng(c["nsys"] * 1000 + c["lo"])
    return np.floor(c["lo"] * (c["hi"] / c["lo"]) ** rng.uniform(0.0, 1.0, c["nsys"])).astype(int)


def _prepare_batch(c, seed):
    sides = _batch_sides(c, seed)
    rng = np.random.default_rng(seed)
    Ks, bs = [], []
    xs = _solution(int((sides ** 2).sum()), seed)
    r0 = 0
    for m in sides:
        m = int(m)
        n = m * m
        pe, ang = rng.uniform(1.0, 100.0), rng.uniform(0.0, 2 * np.pi)
        e2, bx, by = (m + 1.0) ** 2, pe * np.cos(ang) * (m + 1) / 2, pe * np.sin(ang) * (m + 1) / 2
        i = np.arange(n)
        x, y = i % m, i // m
        mask = np.stack([y > 0, x > 0, x >= 0, x < m - 1, y < m - 1], axis=1)
        col = i[:, None] + np.array([-m, -1, 0, 1, m]) + 1
        val = np.broadcast_to(np.array([-e2 - by, -e2 - bx, 4 * e2, -e2 + bx, -e2 + by]), (n, 5))
        rp = np.ones(n + 1, dtype=np.int32)
        rp[1:] += mask.sum(1).cumsum().astype(np.int32)
        Ks.append(idrs_amd.crs_format(n, n, rp, col[mask].astype(np.int32), rval=val[mask]))
        vals = torch.from_numpy(np.where(mask, val, 0.0)).cuda()
        bs.append(_dia_matvec([-m, -1, 0, 1, m], vals, xs[r0:r0 + n]))
        r0 += n
    KB = idrs_amd.batch_format(Ks)
    KB.autotune()
    return dict(case=c, A=idrs_amd.Matrix(KB), b=torch.cat(bs))


def _run_batch(st):
    c = st["case"]
    return idrs_amd.idrs_batched(st["A"], st["b"], c["s"], tolerance=c["tol"], maximum_iterations=4000).x


# --------------------------------------------------------------------------
# differentiable solves on random sparse, diagonally dominant systems
# --------------------------------------------------------------------------
def _random_system(c, seed):
    """Columns (ascending, 0-based) and values (n, k+1): k off-diagonals at
    random columns, the diagonal 1.2 x the row's absolute sum."""
    n, k = c["n"], c["k"]
    g = _gen(seed, 6)
    row = torch.arange(n, device="cuda")[:, None]
    col = torch.randint(0, n - 1, (n, k), generator=g, device="cuda")
    col = col + (col >= row)
    val = torch.randn((n, k), generator=g, device="cuda", dtype=torch.float64)
    col = torch.cat([col, row], dim=1)
    val = torch.cat([val, 1.2 * val.abs().sum(1, keepdim=True)], dim=1)
    col, order = col.sort(dim=1)
    return col, val.gather(1, order)


def _prepare_adjoint(c, seed):
    n = c["n"]
    col, val = _random_system(c, seed)
    rp = (1 + np.arange(n + 1, dtype=np.int64) * (c["k"] + 1)).astype(np.int32)
    system = idrs_amd.SparseSystem(n, rp, (col.reshape(-1) + 1).int().cpu().numpy(), val.reshape(-1).cpu().numpy())
    system.K.autotune()
    system.KT.autotune()
    x, lam = _solution(n, seed), _uniform(n, _gen(seed, 7), -1.0, 1.0)
    b = (val * x[col]).sum(1)
    gx = torch.zeros(n, device="cuda", dtype=torch.float64)
    # A^T lam, one entry of every row at a time in a fixed order
    for j in range(col.shape[1]):
        order = col[:, j].argsort(stable=True)
        cs = col[order, j]
        run = torch.cat([torch.zeros(1, device="cuda", dtype=torch.float64), (val[:, j] * lam)[order].cumsum(0)])
        ends = torch.searchsorted(cs, torch.arange(n, device="cuda"), right=True)
        begs = torch.searchsorted(cs, torch.arange(n, device="cuda"), right=False)
        gx += run[ends] - run[begs]
    return dict(case=c, system=system, vals=val.reshape(-1).contiguous(), b=b, gx=gx)


def _run_adjoint(st):
    c = st["case"]
    v = st["vals"].detach().clone().requires_grad_(True)
    b = st["b"].detach().clone().requires_grad_(True)
    x = idrs_amd.idrs_solve(st["system"], v, b, s=c["s"], tolerance=c["tol"])
    gv, gb = torch.autograd.grad(x, (v, b), grad_outputs=st["gx"])
    return dict(x=x.detach(), grad_values=gv, grad_b=gb)


def _exact_adjoint(c, seed):
    col, _ = _random_system(c, seed)
    x, lam = _solution(c["n"], seed), _uniform(c["n"], _gen(seed, 7), -1.0, 1.0)
    return dict(x=x, grad_values=(-lam[:, None] * x[col]).reshape(-1), grad_b=lam)


# --------------------------------------------------------------------------
def prepare(case, seed):
    if case["kind"] in ("solve", "mixed"):
        return _prepare_solve(case, seed)
    return {"shifts": _prepare_shifts, "batch": _prepare_batch, "adjoint": _prepare_adjoint}[case["kind"]](case, seed)


def run(state):
    kind = state["case"]["kind"]
    if kind in ("solve", "mixed"):
        return _run_solve(state)
    return {"shifts": _run_shifts, "batch": _run_batch, "adjoint": _run_adjoint}[kind](state)


def exact(case, seed):
    """The solution the right-hand side was made from (a fixed number of
    iterations has none)."""
    kind = case["kind"]
    if kind == "solve" and case["budget"]:
        return None
    if kind in ("solve", "mixed"):
        return _solution(case["nx"] * case["ny"] * case["nz"], seed, case["cplx"])
    if kind == "shifts":
        return _exact_shifts(case, seed)
    if kind == "batch":
        return _solution(int((_batch_sides(case, seed) ** 2).sum()), seed)
    return _exact_adjoint(case, seed)


def _iteration_work(n, nnz, s, degree, vec, index):
    """Bytes and flops of one IDR(s) iteration, every operand read once:
    degree + 1 products (values, indices, x, y and the Horner vector) and
    the vector updates 8N (3s^2 + 11s + 3)/(s + 1)."""
    prod = (vec + index) * nnz + 2 * vec * n
    upd = (3 * s * s + 11 * s + 3) / (s + 1)
    return dict(bytes=(degree + 1) * prod + degree * vec * n + vec * n * upd,
                flops=(vec / 8) ** 2 * ((degree + 1) * 2 * nnz + 2 * degree * n + 2 * n * upd))


def work(case):
    """A pass counted over a nominal number of iterations of its kind and
    size (grid solves grow with the side, the random systems do not)."""
    kind = case["kind"]
    if kind in ("solve", "mixed", "shifts"):
        n = case["nx"] * case["ny"] * case["nz"]
        side = max(case["nx"], case["ny"], case["nz"])
    if kind in ("solve", "mixed"):
        its = case["budget"] or ((1.0 * side + 10) if case["degree"] else 5.0 * side + 10)
        w = _iteration_work(n, 7 * n, case["s"], case["degree"], 16 if case["cplx"] else 8,
                            4 if case["storage"] == "crs" else 0)
        return {k: v * its for k, v in w.items()}
    if kind == "shifts":
        its = 0.6 * side + 10
        w = _iteration_work(n, 7 * n, case["s"], case["degree"], 8, 4)
        per = case["nshift"] * n * (case["s"] + 4)      # every shift's window and solution
        return dict(bytes=(w["bytes"] + 8 * per) * its, flops=(w["flops"] + 2 * per) * its)
    if kind == "batch":
        sides = _batch_sides(case, 0)
        tot = dict(bytes=0.0, flops=0.0)
        for m in sides:
            w = _iteration_work(m * m, 5 * m * m, case["s"], 0, 8, 4)
            for k in tot:
                tot[k] += w[k] * 5.0 * m
        return {k: float(v) for k, v in tot.items()}
    n, nnz = case["n"], case["n"] * (case["k"] + 1)
    w = _iteration_work(n, nnz, case["s"], 0, 8, 4)
    return dict(bytes=w["bytes"] * 70 + 20.0 * nnz, flops=w["flops"] * 70 + nnz)
