"""Performance cases of the Krylov library: what a program that uses it has it do.

Each case is one call sequence through the public entry points (`XSolver`,
`XBatch`, `autograd.sparse_solve`).  The sizes are those of the benchmark's
workloads and of the tests, with small and odd ones between them:

* ``cg``       CG + Jacobi on the 2D 5-point Poisson matrix, rtol 1e-8
* ``spmv``     y = A x on a 3D 7- or 27-point stencil, or on rows of very
               uneven length
* ``spmm``     Y = A X for k interleaved columns, 3D 7-point stencil
* ``apply``    y = M^-1 x, exact triangular solves with the ILU(0) factors of
               the 3D convection-diffusion matrix
* ``bicgstab`` set-up + solve of the 3D convection-diffusion system, BiCGSTAB +
               ParILU(0), rtol 1e-10, FP64 or mixed precision
* ``gmres``    set-up + solve of the 27-point lognormal system, GMRES(30) +
               ParILUT, rtol 1e-10, FP64 or mixed precision
* ``batch``    many independent 2D variable-coefficient diffusion systems,
               CG + Jacobi, rtol 1e-8, FP64 or FP32 with FP64 updates
* ``block``    k right-hand sides of the convection-diffusion system at once
* ``adjoint``  forward solve, adjoint solve and gradients by autograd on a 2D
               variable-coefficient diffusion system, CG + ParILU(0)

Right-hand sides are manufactured (b = A x*, x* uniform in [-1, 1]), so x* is
the 64-bit result of every solve.  All inputs are made on the GPU from the
seed.
"""
import math

import numpy as np
import torch

from xsolver_amd import XBatch, XSolver
from xsolver_amd.autograd import make_solver, sparse_solve

DEV = "cuda"


def listed():
    return [
        # the smallest solve: a coarse grid, launch latency and host work only
        {"name": "cg_poisson2d_33", "kind": "cg", "nx": 33, "ny": 33},
        # the 256^2 Poisson benchmark: hundreds of short iterations
        {"name": "cg_poisson2d_256", "kind": "cg", "nx": 256, "ny": 256},
        # a matrix-vector product inside a user's own loop, wide stencil
        {"name": "spmv_27pt_100", "kind": "spmv", "matrix": "27pt", "N": 100},
        # the same on an unstructured matrix: a few long rows, odd size
        {"name": "spmv_irregular", "kind": "spmv", "matrix": "irregular", "N": 262147},
        # a few columns at once, odd in number, odd grid
        {"name": "spmm_7pt_75_k5", "kind": "spmm", "N": 75, "k": 5},
        # the default preconditioner application of a user's own Krylov loop
        {"name": "ilu0_exact_apply_128", "kind": "apply", "N": 128},
        # the benchmark's headline solve: ILU applied by 5 / 2 Jacobi sweeps
        {"name": "bicgstab_ilu0_128", "kind": "bicgstab", "N": 128, "precision": 0, "storage": 0,
         "lsweeps": 5, "usweeps": 2},
        # its mixed-precision form, factors stored in BF16
        {"name": "bicgstab_mixed_128", "kind": "bicgstab", "N": 128, "precision": 1, "storage": 1,
         "lsweeps": 5, "usweeps": 3},
        # the 27-point system with its ParILUT set-up
        {"name": "gmres_parilut_100", "kind": "gmres", "N": 100, "precision": 0, "storage": 0},
        # a time step over many uneven subdomains
        {"name": "batch_512", "kind": "batch", "count": 512, "smin": 32, "smax": 160,
         "precision": 0},
        # many loads on one structure
        {"name": "block_32rhs_128", "kind": "block", "N": 128, "k": 32},
        # a differentiable solve inside a training loop
        {"name": "adjoint_512", "kind": "adjoint", "N": 512},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cg", "spmv", "spmm", "apply", "bicgstab", "gmres", "batch", "block",
                       "adjoint"])
    if kind == "cg":
        return {"kind": kind, "nx": _log_int(rng, 17, 256), "ny": _log_int(rng, 17, 256)}
    if kind == "spmv":
        m = rng.choice(["7pt", "27pt", "irregular"])
        N = {"7pt": (20, 128), "27pt": (16, 100), "irregular": (4000, 262147)}[m]
        return {"kind": kind, "matrix": m, "N": _log_int(rng, *N)}
    if kind == "spmm":
        return {"kind": kind, "N": rng.randint(24, 96), "k": rng.randint(2, 32)}
    if kind == "apply":
        return {"kind": kind, "N": rng.randint(24, 128)}
    if kind == "bicgstab":
        p, st = rng.choice([(0, 0), (1, 0), (1, 1)])
        ls, us = rng.choice([(5, 2), (5, 3), (-1, -1)])
        return {"kind": kind, "N": rng.randint(24, 128), "precision": p, "storage": st,
                "lsweeps": ls, "usweeps": us}
    if kind == "gmres":
        p, st = rng.choice([(0, 0), (1, 1)])
        return {"kind": kind, "N": rng.randint(20, 100), "precision": p, "storage": st}
    if kind == "batch":
        smin = rng.randint(8, 48)
        return {"kind": kind, "count": _log_int(rng, 24, 512), "smin": smin,
                "smax": rng.randint(smin + 8, 160), "precision": rng.randint(0, 1)}
    if kind == "block":
        return {"kind": kind, "N": rng.randint(24, 96), "k": rng.randint(3, 32)}
    return {"kind": kind, "N": rng.randint(40, 320)}


# ---------------------------------------------------------------------------
# matrices, as device CSR triples (int32, int32, float64)
# ---------------------------------------------------------------------------
def _grid(dims):
    """Coordinates (x fastest) of a lexicographic grid."""
    i = torch.arange(math.prod(dims), device=DEV)
    out = []
    for d in dims:
        out.append(i % d)
        i = i // d
    return out


def _stencil_csr(dims, offs, values):
    """CSR of a stencil; values(k, off, mask, shift) gives the entries of
    offset k (its neighbour is the row + shift where mask holds)."""
    n = math.prod(dims)
    xs = _grid(dims)
    rows = torch.arange(n, device=DEV)
    cols = torch.empty((n, len(offs)), dtype=torch.int32, device=DEV)
    mask = torch.empty((n, len(offs)), dtype=torch.bool, device=DEV)
    vals = torch.empty((n, len(offs)), dtype=torch.float64, device=DEV)
    for k, off in enumerate(offs):
        shift, stride = 0, 1
        m = torch.ones(n, dtype=torch.bool, device=DEV)
        for x, d, o in zip(xs, dims, off):
            if o:
                m &= (x + o >= 0) & (x + o < d)
            shift += o * stride
            stride *= d
        cols[:, k] = rows + shift
        mask[:, k] = m
        vals[:, k] = values(k, off, m, shift)
    rp = torch.zeros(n + 1, dtype=torch.int32, device=DEV)
    rp[1:] = mask.sum(1).cumsum(0)
    return rp, cols[mask].contiguous(), vals[mask].contiguous()


POINTS5 = [(0, -1), (-1, 0), (0, 0), (1, 0), (0, 1)]
POINTS7 = [(0, 0, -1), (0, -1, 0), (-1, 0, 0), (0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1)]
POINTS27 = [(x, y, z) for z in (-1, 0, 1) for y in (-1, 0, 1) for x in (-1, 0, 1)]
# 7-point convection-diffusion: velocity (1, 0.5, 0.25), cell Peclet number 0.5
PECLET = (0.5, 0.25, 0.125)
CONVDIFF = [-(1 + PECLET[2]), -(1 + PECLET[1]), -(1 + PECLET[0]), 6.0,
            -(1 - PECLET[0]), -(1 - PECLET[1]), -(1 - PECLET[2])]


def _poisson2d(nx, ny):
    return _stencil_csr((nx, ny), POINTS5, lambda k, off, m, s: 4.0 if k == 2 else -1.0)


def _convdiff3d(N):
    return _stencil_csr((N, N, N), POINTS7, lambda k, off, m, s: CONVDIFF[k])


def _lognormal27(N, gen):
    """Symmetric 27-point matrix: -exp(N(0, 1)) per edge, diagonal 1.05 times
    the row's sum of magnitudes."""
    n = N ** 3
    edge = {o: torch.exp(torch.randn(n, dtype=torch.float64, device=DEV, generator=gen))
            for o in POINTS27[14:]}
    total = torch.zeros(n, dtype=torch.float64, device=DEV)

    def values(k, off, m, shift):
        if k == 13:
            return 0.0
        if off in edge:
            w = edge[off]
        else:   # the edge of the neighbour behind
            w = torch.roll(edge[tuple(-o for o in off)], -shift)
        total.add_(torch.where(m, w, 0.0))
        return -w

    rp, ci, v = _stencil_csr((N, N, N), POINTS27, values)
    rows = torch.repeat_interleave(torch.arange(n, device=DEV), (rp[1:] - rp[:-1]).long())
    v[ci == rows] = 1.05 * total
    return rp, ci, v


def _vardiff2d(kappa):
    """5-point diffusion: harmonic means of the cell coefficients on interior
    faces, the cell's own on the boundary."""
    ny, nx = kappa.shape
    kap = kappa.reshape(-1)
    diag = torch.zeros_like(kap)

    def values(k, off, m, shift):
        if k == 2:
            return 0.0
        other = torch.roll(kap, -shift)
        face = torch.where(m, 2.0 * kap * other / (kap + other), kap)
        diag.add_(face)
        return -face

    rp, ci, v = _stencil_csr((nx, ny), POINTS5, values)
    rows = torch.repeat_interleave(torch.arange(nx * ny, device=DEV), (rp[1:] - rp[:-1]).long())
    v[ci == rows] = diag
    return rp, ci, v


def _random_field(N, gen, ell=0.1):
    """exp of a unit-variance Gaussian random field, squared-exponential
    covariance of length ell on the unit square."""
    w = torch.randn(N, N, dtype=torch.float64, device=DEV, generator=gen)
    kx = torch.fft.fftfreq(N, d=1.0 / N, device=DEV, dtype=torch.float64) * 2 * math.pi
    ky = torch.fft.rfftfreq(N, d=1.0 / N, device=DEV, dtype=torch.float64) * 2 * math.pi
    spec = torch.exp(-0.5 * ell * ell * (kx[:, None] ** 2 + ky[None, :] ** 2))
    g = torch.fft.irfft2(torch.fft.rfft2(w) * spec, s=(N, N))
    return torch.exp((g - g.mean()) / g.std())


def _irregular(n, gen):
    """Rows of 4 to 2000 entries (a power law, about 10 on average), half of
    them near the diagonal, the others anywhere."""
    u = torch.rand(n, dtype=torch.float64, device=DEV, generator=gen)
    lens = (3.0 * u.clamp_min(1e-9) ** -0.7).clamp_max(min(2000.0, n / 4)).long()
    rows = torch.repeat_interleave(torch.arange(n, device=DEV), lens)
    m = rows.numel()
    far = torch.randint(0, n, (m,), device=DEV, generator=gen)
    near = rows + torch.randint(-200, 201, (m,), device=DEV, generator=gen)
    pick = torch.rand(m, device=DEV, generator=gen) < 0.5
    cols = torch.where(pick, near.clamp(0, n - 1), far)
    diag = torch.arange(n, device=DEV)
    key = torch.unique(torch.cat([rows * n + cols, diag * n + diag]))
    r, c = key // n, key % n
    v = torch.rand(key.numel(), dtype=torch.float64, device=DEV, generator=gen) * 2 - 1
    rp = torch.zeros(n + 1, dtype=torch.int32, device=DEV)
    rp[1:] = torch.bincount(r, minlength=n).cumsum(0)
    return rp, c.int().contiguous(), v


def _batch_matrix(sizes, gen):
    """Block-diagonal CSR of independent s x s variable-coefficient diffusion
    systems, kappa = exp(0.5 N(0, 1)) per cell."""
    s = torch.tensor(sizes, device=DEV)
    sys_ptr = torch.zeros(len(sizes) + 1, dtype=torch.int64, device=DEV)
    sys_ptr[1:] = (s * s).cumsum(0)
    n = int(sys_ptr[-1])
    width = torch.repeat_interleave(s, s * s)
    local = torch.arange(n, device=DEV) - torch.repeat_interleave(sys_ptr[:-1], s * s)
    x, y = local % width, local // width
    kap = torch.exp(0.5 * torch.randn(n, dtype=torch.float64, device=DEV, generator=gen))
    rows = torch.arange(n, device=DEV)
    cols = torch.empty((n, 5), dtype=torch.int64, device=DEV)
    mask = torch.ones((n, 5), dtype=torch.bool, device=DEV)
    vals = torch.zeros((n, 5), dtype=torch.float64, device=DEV)
    for k, (ox, oy) in enumerate(POINTS5):
        m = (x + ox >= 0) & (x + ox < width) & (y + oy >= 0) & (y + oy < width)
        c = torch.where(m, rows + ox + oy * width, rows)
        cols[:, k], mask[:, k] = c, m
        if k != 2:
            face = torch.where(m, 2.0 * kap * kap[c] / (kap + kap[c]), kap)
            vals[:, k] = -face
            vals[:, 2] += face
    rp = torch.zeros(n + 1, dtype=torch.int32, device=DEV)
    rp[1:] = mask.sum(1).cumsum(0)
    return sys_ptr.int(), (rp, cols[mask].int().contiguous(), vals[mask].contiguous())


def _matvec(A, x):
    """A x in 64 bits; x of shape (n,) or (n, k)."""
    rp, ci, v = A
    rows = torch.repeat_interleave(torch.arange(rp.numel() - 1, device=DEV),
                                   (rp[1:] - rp[:-1]).long())
    y = torch.zeros_like(x)
    ci = ci.long()
    if x.dim() == 1:
        return y.index_add_(0, rows, v * x[ci])
    for j in range(x.shape[1]):   # a column at a time: the products fit beside the states
        y[:, j] = torch.zeros_like(x[:, j]).index_add_(0, rows, v * x[ci, j])
    return y


def _matvec_t(A, x):
    rp, ci, v = A
    rows = torch.repeat_interleave(torch.arange(rp.numel() - 1, device=DEV),
                                   (rp[1:] - rp[:-1]).long())
    return torch.zeros_like(x).index_add_(0, ci.long(), v * x[rows])


def _uniform(shape, gen):
    return torch.rand(shape, dtype=torch.float64, device=DEV, generator=gen) * 2 - 1


def _inputs(case, seed):
    """The matrix, the vectors it is used with and the known solution."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    kind = case["kind"]
    sys_ptr = None
    if kind == "cg":
        A = _poisson2d(case["nx"], case["ny"])
    elif kind == "spmv":
        A = {"7pt": lambda: _convdiff3d(case["N"]),
             "27pt": lambda: _lognormal27(case["N"], gen),
             "irregular": lambda: _irregular(case["N"], gen)}[case["matrix"]]()
    elif kind == "gmres":
        A = _lognormal27(case["N"], gen)
    elif kind == "batch":
        # the subdomains are the case's, their coefficients the seed's
        sizes = np.random.default_rng(3).integers(case["smin"], case["smax"] + 1, case["count"])
        sys_ptr, A = _batch_matrix(sizes.tolist(), gen)
    elif kind == "adjoint":
        A = _vardiff2d(_random_field(case["N"], gen))
    else:
        A = _convdiff3d(case["N"])
    n = A[0].numel() - 1
    x = _uniform((n, case["k"]) if kind in ("spmm", "block") else (n,), gen)
    return A, x, sys_ptr, gen


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    A, x, sys_ptr, gen = _inputs(case, seed)
    kind = case["kind"]
    st = {"kind": kind, "A": A}
    if kind == "batch":
        st["solver"] = XBatch(sys_ptr.cpu().numpy(), *(t.cpu().numpy() for t in A))
        st["b"], st["x"] = _matvec(A, x), torch.empty_like(x)
        st["precision"] = case["precision"]
        del st["A"]
        return st
    if kind == "adjoint":
        rp, ci, v = A
        st["solver"] = make_solver(rp.cpu().numpy(), ci.cpu().numpy(), v.cpu().numpy(), "cg",
                                   "ilu0", tol=1e-10, maxiter=20000)
        st["vals"] = v.clone().requires_grad_(True)
        st["b"] = _matvec(A, x).requires_grad_(True)
        st["g"] = _matvec_t(A, _uniform(x.shape, gen))   # dL/dx whose adjoint is known
        return st
    S = XSolver()
    S.mat_setup_device(*A)
    st["solver"] = S
    if kind in ("spmv", "spmm", "apply"):
        st["x"], st["y"] = x, torch.empty_like(x)
        if kind == "apply":   # ILU(0) itself: deterministic sweeps to the fixed point
            S.pc_settype("ilu0")
            S.set_option("parilu_async", 0)
            S.set_option("parilu_scale", 0)
            S.set_option("parilu_sweeps", 100)
            S.pc_setup()
        return st
    st["b"], st["x"] = _matvec(A, x), torch.empty_like(x)
    if kind == "cg":
        S.ksp_settype("cg")
        S.ksp_setoption(1e-8, 5000)
        S.pc_settype("jacobi")
    elif kind == "gmres":
        S.ksp_settype("gmres")
        S.ksp_setoption(1e-10, 3000, 30)
        S.pc_settype("ilut")
        S.pc_setilut(1e-4, 2)
        S.set_option("precision", case["precision"])
        S.set_option("factor_storage", case["storage"])
        S.set_option("lsolve_sweeps", 10)
        S.set_option("usolve_sweeps", 15)
    else:
        S.ksp_settype("bicgstab")
        S.ksp_setoption(1e-10, 2000)
        S.pc_settype("ilu0")
        S.set_option("precision", case.get("precision", 0))
        S.set_option("factor_storage", case.get("storage", 0))
        S.set_option("lsolve_sweeps", case.get("lsweeps", 5))
        S.set_option("usolve_sweeps", case.get("usweeps", 2))
    return st


def run(st):
    S, kind = st["solver"], st["kind"]
    if kind == "spmv":
        S.spmv(st["x"], st["y"], torch.cuda.current_stream().cuda_stream)
        return st["y"]
    if kind == "spmm":
        S.spmm(st["x"], st["y"], torch.cuda.current_stream().cuda_stream)
        return st["y"]
    if kind == "apply":
        S.pc_apply(st["x"], st["y"], torch.cuda.current_stream().cuda_stream)
        return st["y"]
    if kind == "adjoint":
        x = sparse_solve(st["vals"], st["b"], S)
        dv, db = torch.autograd.grad(x, (st["vals"], st["b"]), st["g"])
        return {"x": x.detach(), "dvals": dv, "db": db}
    x = st["x"]
    x.zero_()
    if kind == "batch":
        status = S.solve_device(st["b"], x, tol=1e-8, maxiter=5000, precision=st["precision"])
    elif kind == "block":
        status = S.solve_multi_device(st["b"], x)
    else:
        if kind != "cg":   # new values of the matrix: the factors are made again
            S.set_option("refactor", 1)
            S.pc_setup()
        status = S.solve_device(st["b"], x)
    if status != 0:
        raise RuntimeError("the solve did not converge: status %d" % status)
    return x


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _nnz(case):
    kind = case["kind"]
    N = case.get("N", 0)
    if kind == "cg":
        nx, ny = case["nx"], case["ny"]
        return nx * ny, 5 * nx * ny - 2 * (nx + ny)
    if kind == "adjoint":
        return N * N, 5 * N * N - 4 * N
    if kind == "batch":
        lo, hi = case["smin"], case["smax"]
        n = int(case["count"] * sum(s * s for s in range(lo, hi + 1)) / (hi - lo + 1))
        return n, 5 * n
    if kind == "gmres" or case.get("matrix") == "27pt":
        return N ** 3, (3 * N - 2) ** 3
    if case.get("matrix") == "irregular":
        return N, int(10.6 * N)
    return N ** 3, 7 * N ** 3 - 6 * N ** 2


def work(case):
    """Matrix (8-byte values, 4-byte columns and row pointers) and vectors, read
    or written once per product; a solve repeats that for the method's usual
    number of iterations, of which a system that fits the chip's caches
    (256 MB) reads its matrix and vectors from memory once."""
    kind = case["kind"]
    n, nnz = _nnz(case)
    mat = 12 * nnz + 4 * (n + 1)
    if kind == "spmv":
        return {"bytes": mat + 16 * n, "flops": 2 * nnz}
    if kind == "spmm":
        k = case["k"]
        return {"bytes": mat + 16 * n * k, "flops": 2 * nnz * k}
    if kind == "apply":   # L and U with 1/u_ii, x in, the middle vector once, y out
        return {"bytes": 12 * (nnz - n) + 8 * (n + 1) + 32 * n, "flops": 2 * nnz}
    if kind == "cg":
        its = 2.2 * max(case["nx"], case["ny"])
        return {"bytes": mat + 24 * n, "flops": its * (2 * nnz + 12 * n)}
    if kind == "adjoint":   # two CG solves with ILU(0), the gradient gather
        its = 2.1 * case["N"]
        return {"bytes": 4 * mat + 64 * n, "flops": its * (4 * nnz + 12 * n)}
    if kind == "batch":   # rows x iterations: a system of s^2 rows takes about 2.5 s of them
        lo, hi = case["smin"], case["smax"]
        its = 2.5 * sum(s ** 3 for s in range(lo, hi + 1)) / sum(s * s for s in range(lo, hi + 1))
        return {"bytes": its * mat, "flops": its * (2 * nnz + 12 * n)}
    if kind == "gmres":   # ParILUT: ten steps over a pattern of twice A's entries; 13 iterations
        f = 2 * nnz
        return {"bytes": 10 * (mat + 24 * f) + 13 * (mat + 12 * f + 64 * n),
                "flops": 10 * 2.0 * f * (f / n) / 4 + 13 * 2 * (nnz + 25 * f / 2)}
    its = 72 * case["N"] / 128 + 2
    k = case.get("k", 1)
    b = 4 if case.get("precision") else 8
    # an iteration: two products, two applies of L and U, 10 vectors
    apply_l, apply_u = max(1, case.get("lsweeps", 5)), max(1, case.get("usweeps", 2))
    return {"bytes": its * (4 * (b + 4) * nnz + 10 * b * n * k),
            "flops": its * k * (4 * nnz + nnz * (apply_l + apply_u) + 20 * n)}


def tolerance(case):
    """About four times the distance from the 64-bit result: rounding for a
    product or an apply; for a solve, what is left of x - x* when the residual
    reaches its tolerance (it grows with the condition number, for the 2D
    matrices with the square of the grid's width)."""
    kind = case["kind"]
    if kind in ("spmv", "spmm", "apply"):
        return {"rel": 2e-15}
    if kind in ("cg", "batch"):
        s = max(case["nx"], case["ny"]) if kind == "cg" else case["smax"]
        return {"rel": max(1e-7, 2e-10 * s * s)}
    if kind == "adjoint":
        return {"rel": max(1e-7, 8e-12 * case["N"] ** 2)}
    if kind == "gmres":
        return {"rel": 1e-9}
    return {"rel": 3e-8}


# ---------------------------------------------------------------------------
# 64-bit results without the library
# ---------------------------------------------------------------------------
def _ilu0_apply(N, b):
    """(L U)^-1 b for the ILU(0) factors of the convection-diffusion matrix,
    plane by plane of the grid's diagonals x + y + z = const."""
    lower, upper = CONVDIFF[:3], [CONVDIFF[6], CONVDIFF[5], CONVDIFF[4]]   # along -z, -y, -x
    g = torch.stack(_grid((N, N, N)), 1)
    level = g.sum(1)
    order = torch.argsort(level, stable=True)
    bounds = [0] + torch.bincount(level).cumsum(0).tolist()
    shifts = [(2, N * N), (1, N), (0, 1)]
    d = torch.empty_like(b)
    y = b.clone()
    for a, e in zip(bounds[:-1], bounds[1:]):
        r = order[a:e]
        dr, yr = torch.full_like(b[r], 6.0), b[r].clone()
        for (axis, s), lo, up in zip(shifts, lower, upper):
            m = g[r, axis] > 0
            q = (r - s).clamp_min(0)
            l = torch.where(m, lo / d[q], 0.0)
            dr -= l * up
            yr -= l * y[q]
        d[r], y[r] = dr, yr
    for a, e in zip(bounds[-2::-1], bounds[:0:-1]):
        r = order[a:e]
        yr = y[r].clone()
        for (axis, s), up in zip(shifts, upper):
            m = g[r, axis] < N - 1
            yr -= torch.where(m, up * y[(r + s).clamp_max(N ** 3 - 1)], 0.0)
        y[r] = yr / d[r]
    return y


def exact(case, seed):
    A, x, _, gen = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("spmv", "spmm"):
        return _matvec(A, x)
    if kind == "apply":
        return _ilu0_apply(case["N"], x)
    if kind == "adjoint":
        lam = _uniform(x.shape, gen)
        rp, ci, _ = A
        rows = torch.repeat_interleave(torch.arange(x.numel(), device=DEV),
                                       (rp[1:] - rp[:-1]).long())
        return {"x": x, "dvals": -lam[rows] * x[ci.long()], "db": lam}
    return x
