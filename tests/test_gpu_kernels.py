"""GPU parity of the kernels through the C-ABI (xs_spmv, xs_bmax, xs_trsv,
ParILU set-up) against the oracle on the same seeded inputs."""
import numpy as np
import pytest

import oracle
from tests.helpers import random_sparse, rel_err, say, split_factors, true_relres
from xsolver_amd import XSolver, gen

pytestmark = pytest.mark.gpu

MATS = {
    "poisson2d_64": lambda: gen.poisson2d(64),
    "convdiff3d_24": lambda: gen.convdiff3d(24),
    "lognormal27_14": lambda: gen.lognormal27(14, seed=2),
    "grf2d_48": lambda: gen.vardiff2d(gen.grf_kappa(48, 0.1, 4)),
    "random_3000": lambda: random_sparse(3000, 6, 21),
    "longrows_2500": lambda: random_sparse(2500, 4, 22, long_rows=[(7, 2400), (1000, 5000 // 3), (2499, 2300)]),
}


def torch_stream():
    import torch
    return torch.cuda.current_stream().cuda_stream


def dev_tensor(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


@pytest.mark.parametrize("fmt", ["csr", "vec", "ell"])
@pytest.mark.parametrize("name", list(MATS))
def test_spmv_and_bmax_parity(dev, name, fmt):
    import torch
    A = MATS[name]()
    n = len(A[0]) - 1
    say(f"[spmv] {name} {fmt} n={n} nnz={len(A[2])}")
    S = XSolver()
    S.mat_setup(*A, advanced_pam=(0, 1 if fmt == "ell" else 0, 1))
    S.set_option("spmv_kernel", 1 if fmt == "vec" else 0)
    rng = np.random.default_rng(3)
    x = rng.uniform(-1, 1, n)
    b = rng.uniform(-1, 1, n)
    xd, bd = dev_tensor(x, dev), dev_tensor(b, dev)
    yd = torch.empty(n, dtype=torch.float64, device=dev)
    S.spmv(xd, yd, torch_stream())
    torch.cuda.synchronize()
    ref = oracle.spmv(A, x)
    scale = np.abs(A[2]).max() * np.abs(x).max() * np.diff(A[0]).max()
    assert np.abs(yd.cpu().numpy() - ref).max() <= 1e-14 * scale
    S.bmax(bd, xd, yd, torch_stream())
    torch.cuda.synchronize()
    assert np.abs(yd.cpu().numpy() - oracle.bmax(A, b, x)).max() <= 1e-14 * scale
    S.close()


def test_spmv_full_size_convdiff128(dev):
    import torch
    A = gen.convdiff3d(128)
    n = len(A[0]) - 1
    say(f"[spmv] convdiff3d_128 n={n} nnz={len(A[2])}")
    x = np.random.default_rng(1).uniform(-1, 1, n)
    ref = gen.spmv(A, x)
    for ell, vec in ((0, 0), (0, 1), (1, 0)):
        S = XSolver()
        S.mat_setup(*A, advanced_pam=(0, ell, 1))
        S.set_option("spmv_kernel", vec)
        yd = torch.empty(n, dtype=torch.float64, device=dev)
        S.spmv(dev_tensor(x, dev), yd, torch_stream())
        torch.cuda.synchronize()
        assert rel_err(yd.cpu().numpy(), ref) < 1e-14
        S.close()


@pytest.mark.parametrize("name", ["convdiff3d_24", "grf2d_48", "random_3000"])
def test_spmv_diagonal_slots(dev, name):
    """A matrix with at most 8 distinct column - row offsets (the 7-point and
    5-point stencils) gets a diagonal-slot copy for the FP64 SpMV: no index
    per entry, the same entries summed in the same column order (zero
    products where a boundary row lacks a diagonal), so y and b - Ax are bit
    for bit those of the ELL kernel; other matrices keep the ELL copy."""
    import torch
    A = gen.convdiff3d(24) if name == "convdiff3d_24" else MATS[name]()
    n = len(A[0]) - 1
    offs = set()
    rp, ci = A[0], A[1]
    for i in range(n):
        offs.update((ci[rp[i]:rp[i + 1]] - i).tolist())
    rng = np.random.default_rng(6)
    x, b = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
    out = []
    for dia in (1, 0):
        S = XSolver()
        S.set_option("spmv_dia", dia)
        S.mat_setup(*A, advanced_pam=(0, 1, 1))
        nd = S.time_ms("spmv:dia")
        say(f"[spmv-dia] {name} dia={dia}: {int(nd)} slots ({len(offs)} offsets)")
        assert nd == (len(offs) if dia and len(offs) <= 8 else 0)
        yd = torch.empty(n, dtype=torch.float64, device=dev)
        S.spmv(dev_tensor(x, dev), yd, torch_stream())
        zd = torch.empty(n, dtype=torch.float64, device=dev)
        S.bmax(dev_tensor(b, dev), dev_tensor(x, dev), zd, torch_stream())
        torch.cuda.synchronize()
        out.append((yd.cpu().numpy(), zd.cpu().numpy()))
        S.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    scale = np.abs(A[2]).max() * np.abs(x).max() * np.diff(A[0]).max()
    assert np.abs(out[0][0] - oracle.spmv(A, x)).max() <= 1e-14 * scale


def test_default_spmv_kernel_choice(dev):
    """Automatic SpMV kernel for CSR input: ELL copy for near-uniform rows
    (7-point stencil), vector CSR for regular rows with a wider spread, LDS
    row blocks when some rows are long; every choice matches the oracle."""
    import torch
    cases = [("convdiff3d_24", gen.convdiff3d(24), 2),
             ("mixedlen_3000", random_sparse(3000, 3, 15, long_rows=[(i, 12) for i in range(0, 3000, 3)]), 1),
             ("longrows_3000", random_sparse(3000, 5, 31, long_rows=[(7, 2500)]), 0)]
    for name, A, want in cases:
        n = len(A[0]) - 1
        S = XSolver()
        S.mat_setup(*A)
        got = S.time_ms("spmv:kernel")
        say(f"[spmv-default] {name}: kernel {got}")
        assert got == want
        x = np.random.default_rng(4).uniform(-1, 1, n)
        yd = torch.empty(n, dtype=torch.float64, device=dev)
        S.spmv(dev_tensor(x, dev), yd, torch_stream())
        torch.cuda.synchronize()
        scale = np.abs(A[2]).max() * np.diff(A[0]).max()
        assert np.abs(yd.cpu().numpy() - oracle.spmv(A, x)).max() <= 1e-14 * scale
        S.set_option("spmv_kernel", 0)            # explicit choice drops the ELL copy
        assert S.time_ms("spmv:kernel") == 0
        S.close()


def test_ell_column_offsets_and_wide_band(dev):
    """The ELL copy stores 16-bit column offsets when every entry lies within
    32767 of its row, and falls back to int32 columns otherwise; both give
    the oracle's SpMV, and a solve over the sweep copies works either way."""
    import torch
    n = 40000
    rows = np.repeat(np.arange(n), 3)
    cols = np.stack([np.arange(n), (np.arange(n) + 1) % n, (np.arange(n) + 35000) % n], 1).ravel()
    order = np.lexsort((cols, rows))
    rows, cols = rows[order], cols[order]
    rp = np.zeros(n + 1, np.int32)
    np.add.at(rp, rows + 1, 1)
    rp = np.cumsum(rp).astype(np.int32)
    v = np.where(rows == cols, 4.0, -1.0)
    wide = (rp, cols.astype(np.int32), v)
    for name, A, want in (("convdiff3d_20", gen.convdiff3d(20), 1), ("wide_40000", wide, 0)):
        nn = len(A[0]) - 1
        S = XSolver()
        S.mat_setup(*A)
        assert S.time_ms("spmv:kernel") == 2 and S.time_ms("spmv:idx16") == want
        x = np.random.default_rng(5).uniform(-1, 1, nn)
        yd = torch.empty(nn, dtype=torch.float64, device=dev)
        S.spmv(dev_tensor(x, dev), yd, torch_stream())
        torch.cuda.synchronize()
        assert rel_err(yd.cpu().numpy(), oracle.spmv(A, x)) < 1e-14
        xs_, b = gen.manufactured(A, 2)
        S.ksp_settype("bicgstab")
        S.ksp_setoption(1e-10, 500)
        S.pc_settype("ilu0")
        S.set_option("lsolve_sweeps", 3)
        S.set_option("usolve_sweeps", 3)
        xg, st = S.solve(b)
        say(f"[ell-offsets] {name}: idx16={want} it={S.iterations}")
        assert st == 0 and true_relres(A, b, xg) < 1e-10
        S.close()


def _tridiag(n):
    rows, cols, vals = [], [], []
    for i in range(n):
        for j, a in ((i - 1, -1.0), (i, 3.0), (i + 1, -1.2)):
            if 0 <= j < n:
                rows.append(i); cols.append(j); vals.append(a)
    rp = np.zeros(n + 1, np.int32)
    np.add.at(rp, np.array(rows) + 1, 1)
    return np.cumsum(rp).astype(np.int32), np.array(cols, np.int32), np.array(vals)


@pytest.mark.parametrize("name", ["diag_100", "tridiag_1", "tridiag_65", "tridiag_1000",
                                  "random_257"])
def test_small_and_ragged_sizes(dev, name):
    """Edge sizes for the ELL copies, 16-bit offsets and sweep apply: a
    diagonal matrix (empty strict parts, width 0), n = 1, n not a multiple of
    64 / 256 / 512; SpMV, the 3/2 sweep apply (FP64 and k-column) and a solve
    against the oracle."""
    import torch
    if name == "diag_100":
        n = 100
        A = (np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), np.linspace(1, 3, n))
    elif name.startswith("tridiag"):
        A = _tridiag(int(name.split("_")[1]))
    else:
        A = random_sparse(257, 4, 17)
    n = len(A[0]) - 1
    S = XSolver()
    S.mat_setup(*A)
    x = np.random.default_rng(3).uniform(-1, 1, n)
    yd = torch.empty(n, dtype=torch.float64, device=dev)
    S.spmv(dev_tensor(x, dev), yd, torch_stream())
    torch.cuda.synchronize()
    assert rel_err(yd.cpu().numpy(), oracle.spmv(A, x)) < 1e-14
    S.ksp_settype("bicgstab")
    S.ksp_setoption(1e-10, 500)
    S.pc_settype("ilu0")
    S.set_option("parilu_async", 0)
    S.set_option("parilu_sweeps", 60)
    S.set_option("lsolve_sweeps", 3)
    S.set_option("usolve_sweeps", 2)
    S.pc_setup()
    rp, ci, lu, dpos = S.factors(n, len(A[2]))
    S.pc_apply(dev_tensor(x, dev), yd, torch_stream())
    torch.cuda.synchronize()
    ref = oracle.ilu_sweeps(rp, ci, lu, dpos, 3, 2, x)
    assert rel_err(yd.cpu().numpy(), ref) < 1e-13
    X = np.random.default_rng(4).uniform(-1, 1, (n, 3))
    Yd = torch.empty((n, 3), dtype=torch.float64, device=dev)
    S.pc_apply_multi(dev_tensor(X, dev), Yd, torch_stream())
    torch.cuda.synchronize()
    for j in range(3):
        assert rel_err(Yd.cpu().numpy()[:, j], oracle.ilu_sweeps(rp, ci, lu, dpos, 3, 2, X[:, j])) < 1e-13
    _, b = gen.manufactured(A, 5)
    xg, st = S.solve(b)
    say(f"[edge] {name}: n={n} it={S.iterations} idx16={S.time_ms('spmv:idx16')} "
        f"pc_idx16={S.time_ms('pc:idx16')}")
    assert st == 0 and true_relres(A, b, xg) < 1e-10
    S.close()


TRSV_MATS = {
    "convdiff3d_20": lambda: gen.convdiff3d(20),     # in-wave chains (scan path)
    "poisson2d_16": lambda: gen.poisson2d(16),       # in-wave deps r-1, r-16 (loop path)
    "lognormal27_12": lambda: gen.lognormal27(12, seed=2),
    "random_4000": lambda: random_sparse(4000, 7, 23),
    "grf2d_40": lambda: gen.vardiff2d(gen.grf_kappa(40, 0.1, 4)),
}


@pytest.mark.parametrize("name", list(TRSV_MATS))
def test_trsv_parity(dev, name):
    import torch
    A = TRSV_MATS[name]()
    n = len(A[0]) - 1
    say(f"[trsv] {name} n={n}")
    S = XSolver()
    S.mat_setup(*A)
    S.ksp_settype("bicgstab")
    S.pc_settype("ilu0")
    S.pc_setup()
    rp, ci, lu, dpos = S.factors(n, len(A[2]))
    L, U, dinv = split_factors(rp, ci, lu, dpos)
    b = np.random.default_rng(5).uniform(-1, 1, n)
    bd = dev_tensor(b, dev)
    xd = torch.empty(n, dtype=torch.float64, device=dev)
    for rep in range(3):  # repeated calls reuse the self-resetting tickets
        S.trsv(0, bd, xd, torch_stream())
        torch.cuda.synchronize()
        ref = oracle.lower_solve(L, b)
        assert rel_err(xd.cpu().numpy(), ref) < 1e-12
        S.trsv(1, bd, xd, torch_stream())
        torch.cuda.synchronize()
        ref = oracle.upper_solve(U, dinv, b)
        assert rel_err(xd.cpu().numpy(), ref) < 1e-12
    yd = torch.empty(n, dtype=torch.float64, device=dev)
    S.pc_apply(bd, yd, torch_stream())
    torch.cuda.synchronize()
    ref = oracle.upper_solve(U, dinv, oracle.lower_solve(L, b))
    assert rel_err(yd.cpu().numpy(), ref) < 1e-12
    S.close()


@pytest.mark.parametrize("name", ["convdiff3d_20", "lognormal27_12", "grf2d_40", "random_4000",
                                  "convdiff3d_64"])
def test_parilu_converges_to_ilu0(dev, name):
    # convdiff3d_64: 1.8 M entries, so the update lists' scan runs over
    # 1,770 block sums (more than one per scan thread, not a multiple of 1024)
    A = gen.convdiff3d(64) if name == "convdiff3d_64" else TRSV_MATS[name]()
    n = len(A[0]) - 1
    say(f"[parilu] {name} n={n}")
    ref_lu, uptr = oracle.ilu0(A)
    for mode, sweeps, tol in (("sync", 60, 1e-11), ("async", 20, 1e-5)):
        S = XSolver()
        S.mat_setup(*A)
        S.ksp_settype("cg")
        S.pc_settype("ilu0")
        S.set_option("parilu_async", mode == "async")
        S.set_option("parilu_sweeps", sweeps)
        S.pc_setup()
        rp, ci, lu, dpos = S.factors(n, len(A[2]))
        assert np.array_equal(dpos, uptr)
        err = rel_err(lu, ref_lu)
        say(f"   {mode} sweeps={sweeps} max rel diff to ILU(0) = {err:.3e}")
        assert err < tol
        S.close()


@pytest.mark.parametrize("name", ["convdiff3d_9", "random_600"])
def test_parilu_sync_sweep_matches_oracle_sweep(dev, name):
    # one and three deterministic sweeps from the reference's initial guess;
    # the GPU sweeps run over precomputed update lists (random_600: a
    # nonsymmetric pattern, so entries off the diagonal also get products)
    A = gen.convdiff3d(9) if name == "convdiff3d_9" else random_sparse(600, 5, 9)
    n = len(A[0]) - 1
    from tests.test_oracle import _split_for_sweep
    lu0, uptr = oracle.ilu0(A)
    L0, U0, _, _ = _split_for_sweep(A, A[2], uptr)
    l, u = L0[2], U0[2]
    for sweeps in (1, 3):
        for _ in range(sweeps if sweeps == 1 else 2):
            l, u = oracle.parilu_sweep(A, (L0[0], L0[1], l), (U0[0], U0[1], u), n)
        S = XSolver()
        S.mat_setup(*A)
        S.ksp_settype("cg")
        S.pc_settype("ilu0")
        S.set_option("parilu_async", 0)
        S.set_option("parilu_scale", 0)   # the oracle sweeps the unscaled values
        S.set_option("parilu_sweeps", sweeps)
        S.pc_setup()
        rp, ci, lu, dpos = S.factors(n, len(A[2]))
        Lg, Ug, _, _ = _split_for_sweep(A, lu, uptr)
        assert rel_err(Lg[2], l) < 1e-14 and rel_err(Ug[2], u) < 1e-14
        S.close()


PARILUT_MATS = {
    "lognormal27_10": lambda: gen.lognormal27(10, seed=2),
    "convdiff3d_14": lambda: gen.convdiff3d(14),
    "grf2d_40": lambda: gen.vardiff2d(gen.grf_kappa(40, 0.1, 4)),
}


PARILUT_CASES = [(m, 0) for m in PARILUT_MATS] + [("lognormal27_10", 128), ("lognormal27_10", 512)]


@pytest.mark.parametrize("name", ["lognormal27_10", "longrows_1500"])
def test_parilut_small_sets_same_factors(dev, name):
    """The candidate counts of every ParILUT step come from 512-slot sets,
    the rows that fill theirs counted again in 2048-slot sets
    (longrows_1500: rows of 600 and 450 entries, and the rows whose lower part
    reaches them, take the second set).  Same counts, so the same factor as
    counting every row in the 2048-slot set: same pattern, values to the
    rounding of the sweeps' atomic sums."""
    A = (gen.lognormal27(10, seed=2) if name == "lognormal27_10"
         else random_sparse(1500, 4, 29, long_rows=[(3, 600), (300, 450)]))
    n = len(A[0]) - 1
    out = []
    for small in (1, 0):
        S = XSolver()
        S.mat_setup(*A)
        S.ksp_settype("gmres")
        S.pc_settype("ilut")
        S.pc_setilut(1e-4, 2)
        S.set_option("parilut_small_sets", small)
        S.pc_setup()
        rp, ci, lu, dpos = S.factors(n, 4 * len(A[2]) + n)
        out.append((rp.copy(), ci.copy(), lu.copy()))
        S.close()
    say(f"[parilut small sets] {name}: nnz {len(out[0][1])} / {len(out[1][1])}")
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert rel_err(out[0][2], out[1][2]) < 1e-12


@pytest.mark.parametrize("name,rows", PARILUT_CASES, ids=[f"{m}-rows{r}" for m, r in PARILUT_CASES])
def test_parilut_matches_oracle(dev, name, rows):
    """GPU ParILUT (10 steps, fill 2, drop 1e-4) against the oracle's
    deterministic restatement: same pattern up to threshold ties, same values
    to rounding, pivot always present, per-factor counts within the keep.
    rows: the row table of the candidate and sweep kernels (0 = from the row
    lengths; 128 sends the 27-point candidate rows beyond 128 entries to the
    per-entry forms, 512 takes the two-wave workgroups)."""
    A = PARILUT_MATS[name]()
    n = len(A[0]) - 1
    say(f"[parilut] {name} n={n} nnz={len(A[2])} rows={rows}")
    L, U = oracle.parilut(A, 10, 2.0, 1e-4)
    S = XSolver()
    S.mat_setup(*A)
    S.ksp_settype("gmres")
    S.pc_settype("ilut")
    S.pc_setilut(1e-4, 2)
    S.set_option("parilut_rows", rows)
    S.pc_setup()
    cap = 4 * len(A[2]) + n
    rp, ci, lu, dpos = S.factors(n, cap)
    S.close()
    # combined oracle factor in the same layout
    orp = [0]; oci = []; ov = []
    for i in range(n):
        for e in range(L[0][i], L[0][i + 1]):
            oci.append(L[1][e]); ov.append(L[2][e])
        for e in range(U[0][i], U[0][i + 1]):
            oci.append(U[1][e]); ov.append(U[2][e])
        orp.append(len(oci))
    gset = {(i, int(c)) for i in range(n) for c in ci[rp[i]:rp[i + 1]]}
    oset = {(i, int(c)) for i in range(n) for c in oci[orp[i]:orp[i + 1]]}
    sym = len(gset ^ oset)
    say(f"   nnz gpu={len(ci)} oracle={len(oci)} pattern sym-diff={sym}")
    assert sym <= max(4, len(oset) // 1000)
    assert all(ci[dpos[i]] == i for i in range(n))
    nl0 = sum(1 for i in range(n) for c in A[1][A[0][i]:A[0][i + 1]] if c < i)
    nlg = sum(int(dpos[i] - rp[i]) for i in range(n))
    # the keep count (2x A's strict lower part) plus entries tied at the threshold
    assert nlg <= 2 * nl0 + max(sym, len(L[2]) - 2 * nl0)
    gval = {(i, int(ci[e])): lu[e] for i in range(n) for e in range(rp[i], rp[i + 1])}
    oval = {(i, int(oci[e])): ov[e] for i in range(n) for e in range(orp[i], orp[i + 1])}
    common = gset & oset
    diff = max(abs(gval[k] - oval[k]) for k in common)
    scale = max(abs(v) for v in oval.values())
    assert diff <= 1e-9 * scale


def test_gmres_parilut_solve_parity(dev):
    A = gen.lognormal27(16, seed=2)
    xs, b = gen.manufactured(A, [2, 1])
    say(f"[gmres+parilut] lognormal27_16")
    xo, sto, ito, _ = oracle.solve(A, b, "fgmres", "parilut", tol=1e-10, maxiter=300, restart=30,
                                   ilut_tol=1e-4, ilut_fill=2)
    S = XSolver()
    S.mat_setup(*A)
    S.ksp_settype("fgmres"); S.ksp_setoption(1e-10, 300, 30)
    S.pc_settype("ilut"); S.pc_setilut(1e-4, 2)
    x, st = S.solve(b)
    it = S.iterations
    S.close()
    relres = np.linalg.norm(b - gen.spmv(A, x)) / np.linalg.norm(b)
    say(f"   oracle it={ito} gpu it={it} relres={relres:.2e}")
    assert sto == 0 and st == 0 and abs(it - ito) <= 2
    assert relres < 1e-10


@pytest.mark.parametrize("pc,kl,ku", [("ilu0", 0, 0), ("ilu0", 1, 3), ("ilu0", 2, 2),
                                       ("ilu0", 4, 4), ("ilu0", 5, 6), ("ilu0", 20, 20),
                                       ("ilu0", 10, 15), ("ilut", 2, 3), ("ilut", 10, 15)])
def test_ilu_sweep_apply_matches_oracle(dev, pc, kl, ku):
    """The reference's iterative GPU ILU apply (kl / ku Jacobi sweeps per
    factor) against the oracle's restatement on the GPU's own factors; two or
    more sweeps run over the ELL copies of L and U (first two fused), one or
    none over the CSR factors."""
    import torch
    A = gen.convdiff3d(16)
    n = len(A[0]) - 1
    say(f"[sweeps] {pc} kl={kl} ku={ku}")
    S = XSolver()
    S.mat_setup(*A)
    S.ksp_settype("bicgstab")
    S.pc_settype(pc)
    if pc == "ilut":
        S.pc_setilut(1e-3, 3)
    S.set_option("lsolve_sweeps", kl)
    S.set_option("usolve_sweeps", ku)
    S.pc_setup()
    rp, ci, lu, dpos = S.factors(n, 8 * len(A[2]))
    b = np.random.default_rng(6).uniform(-1, 1, n)
    yd = torch.empty(n, dtype=torch.float64, device=dev)
    S.pc_apply(dev_tensor(b, dev), yd, torch_stream())
    torch.cuda.synchronize()
    ref = oracle.ilu_sweeps(rp, ci, lu, dpos, kl, ku, b)
    assert rel_err(yd.cpu().numpy(), ref) < 1e-13
    S.close()


@pytest.mark.parametrize("name", ["convdiff3d_20", "lognormal27_12", "random_4000"])
def test_trsv_level_order_same_result(dev, name):
    """Handing the row groups out in dependency-level order changes only the
    order of work: every row's value is bit-identical to the row-order solve
    (and to the oracle's sequential solve to rounding)."""
    import torch
    A = TRSV_MATS[name]()
    n = len(A[0]) - 1
    b = np.random.default_rng(8).uniform(-1, 1, n)
    out = []
    for sched in (0, 1):
        S = XSolver()
        S.mat_setup(*A)
        S.ksp_settype("bicgstab")
        S.pc_settype("ilu0")
        S.set_option("parilu_async", 0)
        S.set_option("trsv_schedule", sched)
        S.pc_setup()
        yd = torch.empty(n, dtype=torch.float64, device=dev)
        for _ in range(2):
            S.pc_apply(dev_tensor(b, dev), yd, torch_stream())
            torch.cuda.synchronize()
        out.append(yd.cpu().numpy())
        rp, ci, lu, dpos = S.factors(n, len(A[2]))
        S.close()
    assert np.array_equal(out[0], out[1])
    L, U, dinv = split_factors(rp, ci, lu, dpos)
    assert rel_err(out[1], oracle.upper_solve(U, dinv, oracle.lower_solve(L, b))) < 1e-12


def _rows_of_lengths(lens, n, seed):
    """CSR with the given row lengths (repeated), the diagonal among each row's
    columns and dominant."""
    rng = np.random.default_rng(seed)
    rp, ci, v = [0], [], []
    for i in range(n):
        m = min(lens[i % len(lens)], n)
        c = rng.choice(n - 1, m - 1, replace=False)
        c = np.sort(np.append(np.where(c >= i, c + 1, c), i))
        a = rng.uniform(-1, 1, m)
        a[c == i] = 1.5 * np.abs(a).sum() + 1.0
        ci.append(c)
        v.append(a)
        rp.append(rp[-1] + m)
    return np.array(rp, np.int32), np.concatenate(ci).astype(np.int32), np.concatenate(v)


# the last rows of lengths: at the rule's edges, 40 and 256 entries and ten
# times the mean, and at the rungs below which a lane sums a row
@pytest.mark.parametrize("lens", [(1, 15, 16, 17), (16, 17, 63, 64, 65), (2, 2047, 3), (1500, 1, 1),
                                  (17,), (1,) * 30 + (40,), (1,) * 30 + (41,), (256, 1), (257, 1),
                                  (6,) * 31 + (80,), (6,) * 31 + (90,),
                                  (2,) * 20 + (48, 49, 96, 97, 192, 193, 300)],
                         ids=lambda l: str(l) if len(l) < 8 else f"{len(l)}to{max(l)}")
def test_csr_row_blocks_mixed_lengths(dev, lens):
    """Rows at the edges of the lane / wave split of the LDS row blocks
    (xs_csr_lane_rows, csr_limit), FP64 products and epilogues and the FP32 inner
    solve over the same blocks.  Bound: a row of m products summed in any order
    is within m eps sum |a x| of the exact sum, and so is the oracle's."""
    import torch
    n = 2300 if max(lens) > 1000 else 1601
    A = _rows_of_lengths(lens, n, 5)
    say(f"[csr rows] lens={lens} n={n}")
    rng = np.random.default_rng(4)
    x, b = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
    bound = 2 * max(lens) * 2.3e-16 * (gen.spmv((A[0], A[1], np.abs(A[2])), np.abs(x)) + np.abs(b))
    S = XSolver()
    S.mat_setup(*A)
    S.set_option("spmv_kernel", 0)
    assert S.time_ms("spmv:kernel") == 0
    yd = torch.empty(n, dtype=torch.float64, device=dev)
    S.spmv(dev_tensor(x, dev), yd, torch_stream())
    assert np.all(np.abs(yd.cpu().numpy() - oracle.spmv(A, x)) <= bound)
    S.bmax(dev_tensor(b, dev), dev_tensor(x, dev), yd, torch_stream())
    assert np.all(np.abs(yd.cpu().numpy() - oracle.bmax(A, b, x)) <= bound)
    S.ksp_settype("bicgstab")
    S.ksp_setoption(1e-10, 200)
    S.pc_settype("jacobi")
    for precision in (0, 1):
        S.set_option("precision", precision)
        xs, st = S.solve(b)
        assert st == 0 and true_relres(A, b, xs) < 1e-10
    S.close()


def test_csr_row_blocks_time_per_entry(dev):
    """Rows a little past a limit of the lane / wave split cost about what
    shorter ones do per entry (summed by a wave each, rows of 17 took 3.4 times
    as long as rows of 16)."""
    import torch
    us = {}
    for L in (16, 17, 27, 60, 100):
        n = 3200000 // L
        rng = np.random.default_rng(L)
        # L ascending columns a row, about 40 apart, around the diagonal
        c = np.arange(n)[:, None] + np.cumsum(rng.integers(1, 80, (n, L)), 1) - 20 * L
        c = np.sort(np.clip(c, 0, None) % (n + 100 * L), 1).astype(np.int64)
        keep = np.ones_like(c, bool)
        keep[:, 1:] = c[:, 1:] != c[:, :-1]
        keep &= c < n
        rp = np.append(0, np.cumsum(keep.sum(1))).astype(np.int32)
        ci = c[keep].astype(np.int32)
        S = XSolver()
        S.mat_setup(rp, ci, rng.uniform(-1, 1, len(ci)))
        S.set_option("spmv_kernel", 0)
        assert S.time_ms("spmv:kernel") == 0
        x = torch.ones(n, dtype=torch.float64, device=dev)
        y = torch.empty_like(x)
        best = 1e30
        for _ in range(6):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(20):
                S.spmv(x, y, torch_stream())
            b.record()
            torch.cuda.synchronize()
            best = min(best, 50e6 * a.elapsed_time(b) / len(ci))   # ps per entry
        us[L] = best
        S.close()
    say("[csr time] ps per entry", {k: round(v, 1) for k, v in us.items()})
    assert max(us.values()) < 2 * us[16], us


def _grid_stencil(dims, offs, seed):
    """Random nonsymmetric stencil matrix on a grid, entries in [-1, 1], the
    diagonal 2.2 times their number."""
    cols, mask = gen._grid_offsets(dims, offs)
    n = len(cols)
    rng = np.random.default_rng(seed)
    v = np.where(mask, rng.uniform(-1, 1, cols.shape), 0.0)
    d = offs.index((0,) * len(dims))
    v[:, d] = 2.2 * (len(offs) - 1)
    return gen._assemble(n, cols, v, mask)


S5 = [(0, -1), (-1, 0), (0, 0), (1, 0), (0, 1)]
S7 = [(0, 0, -1), (0, -1, 0), (-1, 0, 0), (0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1)]
S9 = [(0, 0, -1), (0, -2, 0)] + S7[1:6] + [(0, 2, 0), (0, 0, 1)]
S9D = [(0, 0, -1), (1, 0, -1)] + S7[1:6] + [(-1, 0, 1), (0, 0, 1)]
CHAINS = {  # grid, stencil, chains of L (0: the general solve)
    "one_narrow": ((17, 40), S5, 1),          # part of a wave
    "one_full": ((64, 9), S5, 1),             # a step past a block of 8
    "carry_one_lane": ((65, 30), S5, 2),      # a group of one lane, carried
    "four": ((256, 300), S5, 4),              # chain 0 has less to do: the pace
    "next_workgroup": ((300, 100), S5, 5),
    "eight_waves": ((520, 30), S5, 9),        # more chains per step: 8 to a workgroup
    "planes": ((20, 20, 24), S7, 20),
    "planes_carry": ((70, 12, 10), S7, 24),
    "three_entries": ((128, 9, 16), S9, 18),  # and a carry
    "own_ring": ((60, 9, 16), S9D, 9),        # another lane of the chain's last step
    "three_blocks": ((130, 12, 10), S7, 36),
    "four_blocks": ((200, 20, 20), S7, 0),    # fewer levels by the general solve
    "four_blocks_one_row": ((193, 16, 16), S7, 64),   # which runs such groups together
    "four_blocks_many_lines": ((198, 90, 8), S7, 360),
    "groups_too_short": ((12, 12, 12), S7, 0),
    "chains_too_short": ((40, 40, 5), S7, 0),
}


@pytest.mark.parametrize("name", list(CHAINS))
def test_trsv_chains_edges(dev, name):
    """The triangular solves over chains against the oracle and, transposed,
    against the general solve.  The off-diagonal factor entries of every row
    and column sum to q < 0.5 of the pivot, so the error of x is at most
    1 / (1 - q) = 2 times a row's own, which a scan of 64 affine maps (two
    roundings each) and four products bound by 140 eps: 2 * 140 * 2.2e-16 =
    6.2e-14 of max |x|.  Over both triangles of two solves that differ by as
    much each: 2 * (6.2e-14 + 2 * 6.2e-14)."""
    import torch
    dims, offs, chains = CHAINS[name]
    A = _grid_stencil(dims, offs, 11)
    n = len(A[0]) - 1
    say(f"[chains] {name} n={n}")
    b = np.random.default_rng(6).uniform(-1, 1, n)
    bd = dev_tensor(b, dev)
    out = {}
    for on in (1, 0):
        S = XSolver()
        S.mat_setup(*A)
        S.pc_settype("ilu0")
        S.set_option("parilu_async", 0)
        S.set_option("trsv_chains", on)
        S.pc_setup()
        ld, ud, td = (torch.empty(n, dtype=torch.float64, device=dev) for _ in range(3))
        for rep in range(2):   # tickets reset themselves
            S.trsv(0, bd, ld, torch_stream())
            S.trsv(1, bd, ud, torch_stream())
            S.pc_apply_t(bd, td, torch_stream())
            torch.cuda.synchronize()
        assert S.time_ms("trsv:chains") == (chains if on else -1)   # -1: not looked at
        out[on] = [t.cpu().numpy() for t in (ld, ud, td)]
        if on:
            L, U, dinv = split_factors(*S.factors(n, len(A[2])))
        S.close()
    rl, ru = (np.repeat(np.arange(n), np.diff(T[0])) for T in (L, U))
    ad = np.abs(dinv)
    for idx, w in ((rl, np.abs(L[2])), (L[1], np.abs(L[2])), (ru, np.abs(U[2]) * ad[ru]),
                   (U[1], np.abs(U[2]) * ad[U[1]])):
        assert np.bincount(idx, w, n).max() < 0.5
    assert rel_err(out[1][0], oracle.lower_solve(L, b)) < 6.2e-14
    assert rel_err(out[1][1], oracle.upper_solve(U, dinv, b)) < 6.2e-14
    assert rel_err(out[1][2], out[0][2]) < 6 * 6.2e-14


@pytest.mark.parametrize("name", ["one_narrow", "four", "planes"])
def test_captured_exact_apply_follows_setup(dev, name):
    """An exact apply recorded into a graph solves with the factor of the last
    set-up, whichever came first, and can be recorded right after one."""
    import torch
    from xsolver_amd.autograd import solver_lib_update
    dims, offs, chains = CHAINS[name]
    A = _grid_stencil(dims, offs, 12)
    n = len(A[0]) - 1
    say(f"[captured apply] {name} n={n}")
    rng = np.random.default_rng(13)
    b = dev_tensor(rng.uniform(-1, 1, n), dev)
    y, ye = torch.empty_like(b), torch.empty_like(b)
    S = XSolver()
    S.mat_setup(*A)
    S.pc_settype("ilu0")
    S.set_option("parilu_async", 0)
    S.pc_setup()
    S.pc_apply(b, ye, torch_stream())   # the pattern's chains
    torch.cuda.synchronize()
    assert S.time_ms("trsv:chains") == chains

    def record():
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            S.pc_apply(b, y, torch_stream())
        return g

    graph = record()
    for step in range(3):
        if step:
            solver_lib_update(S, dev_tensor(A[2] * (1.0 + 0.3 * rng.uniform(size=len(A[2]))), dev))
            S.pc_setup()
        if step == 2:
            graph = record()
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        S.pc_apply(b, ye, torch_stream())
        torch.cuda.synchronize()
        assert torch.equal(y, ye), step
    S.close()
