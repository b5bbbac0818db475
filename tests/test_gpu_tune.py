"""Autotuner (xs_autotune): the chosen SpMV format / row-block size /
vector-CSR lanes and long-row threshold / k-RHS SpMM columns per thread, and
after a factorisation the triangular solves' workgroups / gather width /
group mode, are among the candidates; the SpMV, the SpMM, the triangular
solves and a solve with them still match the oracle; the per-matrix cache
file is written and then reused."""
import numpy as np
import pytest

import oracle
from tests.helpers import random_sparse, say, true_relres
from tests.test_gpu_kernels import S5, _grid_stencil
from xsolver_amd import XSolver, gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,build", [
    ("convdiff3d_48", lambda: gen.convdiff3d(48)),
    ("longrows_4000", lambda: random_sparse(4000, 5, 31, long_rows=[(10, 3000), (2000, 1500)])),
])
def test_autotune_choice_and_parity(dev, name, build, tmp_path, monkeypatch):
    import torch
    cache = tmp_path / "tune.txt"
    monkeypatch.setenv("XS_TUNE_CACHE", str(cache))
    A = build()
    n = len(A[0]) - 1
    S = XSolver()
    S.mat_setup(*A)
    chunk, ell, us = S.autotune()
    say(f"[tune] {name}: chunk={chunk} ell={ell} {us:.2f} us")
    # chunk 0 = the row-binned vector-CSR kernel
    assert chunk in (0, 512, 1024, 1536, 2048, 3072, 4096) and ell in (0, 1) and us > 0
    lanes, thr, cw = (int(S.time_ms(k)) for k in ("tune:vec_lanes", "tune:long_thr", "tune:spmm_cw"))
    say(f"   vector CSR {lanes} lanes, long rows past {thr}; SpMM {cw} columns per thread")
    assert lanes in (2, 4, 8, 16, 32, 64) and thr // lanes in (4, 8, 16) and thr % lanes == 0
    # the SpMM is tuned with the ELL copy (0: no copy for these row lengths)
    assert cw in ((2, 4) if ell else (0, 2, 4))
    lines = cache.read_text().split("\n")
    assert len([l for l in lines if l.strip()]) == 1
    x = np.random.default_rng(2).uniform(-1, 1, n)
    yd = torch.empty(n, dtype=torch.float64, device=dev)
    S.spmv(torch.from_numpy(x).to(dev), yd, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    scale = np.abs(A[2]).max() * np.diff(A[0]).max()
    assert np.abs(yd.cpu().numpy() - oracle.spmv(A, x)).max() <= 1e-14 * scale
    _, b = gen.manufactured(A, 1)
    S.ksp_settype("bicgstab")
    S.ksp_setoption(1e-10, 1000)
    S.pc_settype("jacobi")
    xg, st = S.solve(b)
    assert st == 0 and true_relres(A, b, xg) < 1e-10
    S.close()
    # a second context on the same matrix takes the cached choice
    T = XSolver()
    T.mat_setup(*A)
    assert T.autotune() == (chunk, ell, pytest.approx(us, rel=1e-3))
    assert len([l for l in cache.read_text().split("\n") if l.strip()]) == 1
    T.close()


def test_autotune_triangular_solves_and_spmm(dev, tmp_path, monkeypatch):
    """After ILU(0) set-up the tuner also picks the SpTRSV configuration; the
    exact triangular solves with it equal the oracle's, the k-RHS SpMM with
    the tuned columns per thread equals per-column SpMVs, and a second
    context takes both choices from the cache."""
    import torch
    cache = tmp_path / "tune.txt"
    monkeypatch.setenv("XS_TUNE_CACHE", str(cache))
    A = gen.convdiff3d(24)
    n = len(A[0]) - 1
    S = XSolver()
    S.mat_setup(*A)
    S.ksp_settype("bicgstab")
    S.ksp_setoption(1e-10, 500)
    S.pc_settype("ilu0")
    S.set_option("parilu_async", 0)
    S.set_option("parilu_sweeps", 400)
    S.set_option("parilu_scale", 0)
    S.pc_setup()
    S.autotune()
    wg, ga, pr, tus = (S.time_ms(k) for k in ("tune:trsv_wg", "tune:trsv_gather", "tune:trsv_prog",
                                               "tune:trsv_us"))
    say(f"[tune] convdiff3d_24 SpTRSV: {int(wg)} workgroups, gather {int(ga)}, mode {int(pr)}, "
        f"{tus:.1f} us per lower + upper solve")
    assert wg in (128, 256, 512, 1024) and ga in (4, 16) and pr in (0, 1) and tus > 0
    assert len([l for l in cache.read_text().split("\n") if l.strip()]) == 2
    # exact triangular solves with the tuned configuration: L U z = b for the
    # device factors (L unit lower, U with the pivots, one combined CSR)
    rng = np.random.default_rng(4)
    b = rng.uniform(-1, 1, n)
    bd = torch.from_numpy(b).to(dev)
    y = torch.empty_like(bd)
    z = torch.empty_like(bd)
    st = torch.cuda.current_stream().cuda_stream
    S.trsv(0, bd, y, st)
    S.trsv(1, y, z, st)
    torch.cuda.synchronize()
    rp, ci, lu, dpos = S.factors(n, len(A[2]))
    zz = z.cpu().numpy()
    u_z = np.zeros(n)
    for i in range(n):
        u_z[i] = sum(lu[e] * zz[ci[e]] for e in range(dpos[i], rp[i + 1]))
    lu_z = u_z.copy()
    for i in range(n):
        lu_z[i] += sum(lu[e] * u_z[ci[e]] for e in range(rp[i], dpos[i]))
    assert np.abs(lu_z - b).max() <= 1e-10 * np.abs(b).max()
    # the k-RHS SpMM with the tuned columns per thread
    k = 8
    X = rng.uniform(-1, 1, (n, k))
    Xd = torch.from_numpy(np.ascontiguousarray(X)).to(dev)
    Yd = torch.empty_like(Xd)
    S.spmm(Xd, Yd, st)
    torch.cuda.synchronize()
    Y = Yd.cpu().numpy()
    scale = np.abs(A[2]).max() * np.diff(A[0]).max()
    for j in range(k):
        assert np.abs(Y[:, j] - oracle.spmv(A, X[:, j])).max() <= 1e-14 * scale
    xs, bb = gen.manufactured(A, 1)
    S.set_option("lsolve_sweeps", -1)
    S.set_option("usolve_sweeps", -1)
    xg, stt = S.solve(bb)
    assert stt == 0 and true_relres(A, bb, xg) < 1e-10
    S.close()
    T = XSolver()
    T.mat_setup(*A)
    T.ksp_settype("bicgstab")
    T.pc_settype("ilu0")
    T.set_option("parilu_async", 0)
    T.set_option("parilu_sweeps", 400)
    T.set_option("parilu_scale", 0)
    T.pc_setup()
    T.autotune()
    assert (T.time_ms("tune:trsv_wg"), T.time_ms("tune:trsv_gather"),
            T.time_ms("tune:trsv_prog")) == (wg, ga, pr)
    assert len([l for l in cache.read_text().split("\n") if l.strip()]) == 2
    T.close()


def _chain_factor(**opts):
    """Dominant 5-point matrix on a 256 x 300 grid and its factor, whose
    triangular solves have 4 chains."""
    A = _grid_stencil((256, 300), S5, 11)
    S = XSolver()
    S.mat_setup(*A)
    S.pc_settype("ilu0")
    S.set_option("parilu_async", 0)
    for k, v in opts.items():
        S.set_option(k, v)
    S.pc_setup()
    return S, A


def _solves(S, b, dev):
    """L, U and transposed solves with the present factor."""
    import torch
    st = torch.cuda.current_stream().cuda_stream
    out = [torch.empty_like(b) for _ in range(3)]
    S.trsv(0, b, out[0], st)
    S.trsv(1, b, out[1], st)
    S.pc_apply_t(b, out[2], st)
    torch.cuda.synchronize()
    return out


def _refactor(S, A, dev):
    import torch
    from xsolver_amd.autograd import solver_lib_update
    solver_lib_update(S, torch.from_numpy(A[2]).to(dev))
    S.pc_setup()


def test_gather_width_leaves_the_chains(dev):
    """The gather width is the general solve's: a factor with chains keeps them
    over it and over a set-up with new values."""
    import torch
    S, A = _chain_factor()
    b = torch.ones(len(A[0]) - 1, dtype=torch.float64, device=dev)
    ref = _solves(S, b, dev)
    assert S.time_ms("trsv:chains") == 4
    for ga in (16, 4, 0):
        S.set_option("trsv_gather", ga)
        _refactor(S, A, dev)
        out = _solves(S, b, dev)
        assert S.time_ms("trsv:chains") == 4, ga
        assert all(torch.equal(x, y) for x, y in zip(out, ref))
    S.close()


def test_tuned_chains_stay_chosen(dev, tmp_path, monkeypatch):
    """A factor with chains: the tuner's choice between them and the general
    solve, either way (the cached line edited), holds over a set-up with new
    values, for the transposed solves, and in a context that reads the cache;
    a context that rules chains out has a line of its own."""
    import torch
    cache = tmp_path / "tune.txt"
    monkeypatch.setenv("XS_TUNE_CACHE", str(cache))
    S, A = _chain_factor()
    b = torch.from_numpy(np.random.default_rng(5).uniform(-1, 1, len(A[0]) - 1)).to(dev)
    ref = _solves(S, b, dev)
    assert S.time_ms("tune:trsv_chains") == -1
    S.autotune()
    chosen, us = S.time_ms("tune:trsv_chains"), S.time_ms("tune:trsv_us")
    say(f"[tune] 256 x 300: chains {chosen}, {us:.1f} us per lower + upper solve")
    assert chosen in (0, 1) and us > 0
    S.close()
    lines = cache.read_text().splitlines()
    assert len(lines) == 2 and lines[1].startswith("trsv+chains:")
    f = lines[1].split()
    # key, workgroups, gather, group mode, chains, us
    assert len(f) == 6 and f[4] == str(int(chosen))
    for pr, ch in (("0", "1"), ("1", "1"), ("0", "0"), ("1", "0")):
        f[2:5] = ["16" if pr == "1" else "4", pr, ch]
        cache.write_text(lines[0] + "\n" + " ".join(f) + "\n")
        S, _ = _chain_factor()
        _solves(S, b, dev)   # (chains of both are there before the tuner decides)
        S.autotune()
        assert S.time_ms("tune:trsv_chains") == int(ch)
        for rep in range(2):
            out = _solves(S, b, dev)
            assert S.time_ms("trsv:chains") == (4 if ch == "1" else 0), (pr, ch, rep)
            for x, y in zip(out, ref):
                # (the general solve: the bound of test_trsv_chains_edges)
                assert torch.equal(x, y) if ch == "1" else \
                    (x - y).abs().max() <= 6 * 6.2e-14 * y.abs().max(), (pr, ch, rep)
            _refactor(S, A, dev)
        S.close()
    assert len(cache.read_text().splitlines()) == 2
    S, _ = _chain_factor(trsv_chains=0)
    S.autotune()
    assert S.time_ms("tune:trsv_chains") == 0
    assert cache.read_text().splitlines()[2].startswith("trsv:")
    _solves(S, b, dev)
    assert S.time_ms("trsv:chains") in (0, -1)
    S.close()
