"""Batched persistent CG + Jacobi through the C-ABI (xs_batch_*), per system
against the oracle's CG on the same seeded systems."""
import numpy as np
import pytest

import oracle
import xsolver_amd
from tests.helpers import X_TOL, say
from xsolver_amd import XBatch, batch_concat, gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32inner"])
def test_batch_matches_per_system_oracle(dev, precision):
    sizes, systems = gen.batch_systems(count=40, smin=8, smax=48, seed=3)
    sys_ptr, rp, ci, v = batch_concat(systems)
    rng = np.random.default_rng(7)
    xs = rng.uniform(-1, 1, sys_ptr[-1])
    b = gen.spmv((rp, ci, v), xs)
    say(f"[batch] {len(systems)} systems, n={sys_ptr[-1]}, precision={precision}")
    B = XBatch(sys_ptr, rp, ci, v)
    x, st = B.solve(b, tol=1e-8, maxiter=3000, precision=precision)
    it, rr = B.results()
    B.close()
    assert st == 0
    for s, A in enumerate(systems):
        lo, hi = sys_ptr[s], sys_ptr[s + 1]
        xo, sto, ito, _ = oracle.solve(A, b[lo:hi], "cg", "jacobi", tol=1e-8, maxiter=3000)
        true = np.linalg.norm(b[lo:hi] - gen.spmv(A, x[lo:hi])) / np.linalg.norm(b[lo:hi])
        assert sto == 0
        assert true < 1.05e-8 and rr[s] == pytest.approx(true, rel=1e-6, abs=1e-14)
        if precision == 0:
            assert abs(int(it[s]) - ito) <= 2, (s, it[s], ito)
            assert np.linalg.norm(x[lo:hi] - xo) / np.linalg.norm(xo) <= X_TOL


def test_batch_uneven_sizes_and_zero_rhs(dev):
    sizes, systems = gen.batch_systems(count=12, smin=4, smax=70, seed=5)
    sys_ptr, rp, ci, v = batch_concat(systems)
    b = np.ones(sys_ptr[-1])
    b[sys_ptr[3]:sys_ptr[4]] = 0.0            # one system with a zero right-hand side
    B = XBatch(sys_ptr, rp, ci, v)
    x, st = B.solve(b, tol=1e-10, maxiter=5000)
    it, rr = B.results()
    B.close()
    assert st == 0 and it[3] == 0 and np.all(x[sys_ptr[3]:sys_ptr[4]] == 0)
    assert len(set(it.tolist())) > 3          # systems stop at their own counts


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32inner"])
def test_batch_nonzero_x0_uses_initial_residual_base(dev, precision):
    """Both precisions stop on ||b - A x|| < tol ||b - A x0|| and report relres
    on that base (the reference's convention, hip/Solver/xsolver_cg.cpp:16-74),
    as the oracle's CG started from the same x0 does."""
    sizes, systems = gen.batch_systems(count=10, smin=8, smax=40, seed=8)
    sys_ptr, rp, ci, v = batch_concat(systems)
    rng = np.random.default_rng(9)
    b = gen.spmv((rp, ci, v), rng.uniform(-1, 1, sys_ptr[-1]))
    x0 = rng.uniform(-1, 1, sys_ptr[-1])
    B = XBatch(sys_ptr, rp, ci, v)
    x, st = B.solve(b, tol=1e-9, maxiter=3000, precision=precision, x0=x0)
    it, rr = B.results()
    B.close()
    assert st == 0
    for s, A in enumerate(systems):
        lo, hi = sys_ptr[s], sys_ptr[s + 1]
        r0 = np.linalg.norm(b[lo:hi] - gen.spmv(A, x0[lo:hi]))
        true = np.linalg.norm(b[lo:hi] - gen.spmv(A, x[lo:hi])) / r0
        assert true < 1e-9 and rr[s] == pytest.approx(true, rel=1e-6, abs=1e-15)
        if precision == 0:
            xo, sto, ito, _ = oracle.solve(A, b[lo:hi], "cg", "jacobi", tol=1e-9, maxiter=3000,
                                           x0=x0[lo:hi])
            assert sto == 0 and abs(int(it[s]) - ito) <= 2
            assert np.linalg.norm(x[lo:hi] - xo) / np.linalg.norm(xo) <= X_TOL


# rows per system at the edges of k_batch_res: one row, a thread each, 8 rows a
# thread (its small form), 32 (d in registers), 39 (p in LDS), 50 (its limit),
# and beyond it (k_batch_cg)
RES_EDGES = (1, 2, 511, 512, 513, 4095, 4096, 4097, 16384, 16385, 19967, 19968, 19969, 25600,
             25601)


def _band_system(n, kind, rng):
    """Dominant symmetric systems: 'dia' tridiagonal plus a far pair (5 offsets,
    diagonal slots), 'wide' with 9 offsets (CSR, rows beyond the 6-entry
    window), 'unsorted' = tridiagonal with its columns in descending order."""
    offs = {"dia": (1, 37), "wide": (1, 2, 5, 23), "unsorted": (1,)}[kind]
    rows, cols, vals = [np.arange(n)], [np.arange(n)], [2.0 * len(offs) + rng.uniform(0.5, 1, n)]
    for o in offs:
        if o < n:
            a = -rng.uniform(0.2, 1, n - o)
            rows += [np.arange(n - o), np.arange(o, n)]
            cols += [np.arange(o, n), np.arange(n - o)]
            vals += [a, a]
    r, c, v = np.concatenate(rows), np.concatenate(cols), np.concatenate(vals)
    k = np.lexsort((-c if kind == "unsorted" else c, r))
    return np.append(0, np.cumsum(np.bincount(r, minlength=n))), c[k], v[k]


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32"])
@pytest.mark.parametrize("kind,sizes", [("dia", RES_EDGES), ("wide", RES_EDGES),
                                        ("unsorted", (1, 513, 4097, 19969)),
                                        ("dia", (1, 513, 4096)), ("wide", (7, 4095))],
                         ids=["dia", "wide", "unsorted", "dia-small", "wide-small"])
def test_batch_resident_edges(dev, kind, sizes, precision):
    import torch
    rng = np.random.default_rng(11)
    sys_ptr, rp, ci, v = batch_concat([_band_system(n, kind, rng) for n in sizes])
    A = (rp, ci, v)
    b = gen.spmv(A, rng.uniform(-1, 1, int(sys_ptr[-1])))
    say(f"[batch edges] {kind} rows={sys_ptr[-1]} precision={precision}")
    B = XBatch(sys_ptr, *A)
    x, st = B.solve(b, tol=1e-9, maxiter=500, precision=precision)
    it, rr = B.results()
    B.close()
    assert st == 0 and rr.max() < 1e-9
    xo, ito, _, bad = oracle.batch_cg(sys_ptr, A, b, tol=1e-9, maxiter=500)
    assert bad == 0
    for s, (lo, hi) in enumerate(zip(sys_ptr[:-1], sys_ptr[1:])):
        dx = np.linalg.norm(x[lo:hi] - xo[lo:hi]) / np.linalg.norm(xo[lo:hi])
        # FP64: the oracle's recurrence; FP32: both meet the residual
        # tolerance, and the matrices' condition is below 20
        assert dx <= (X_TOL if precision == 0 else 2 * 20 * 1e-9), (hi - lo, dx)
        if precision == 0:
            assert abs(int(it[s]) - int(ito[s])) <= 1, (hi - lo, it[s], ito[s])
    if precision == 0:   # the allocation-free entry: the same systems, bit for bit
        from tests.test_zz_no_alloc import _noalloc
        rc, x2, it2, rr2, _ = _noalloc(torch, dev, sys_ptr, rp, ci, v, b, 1e-9, 500)
        assert rc == 0 and np.array_equal(x2, x) and np.array_equal(it2, it)
        assert np.array_equal(rr2, rr)


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), 1e200], ids=["nan", "inf", "overflow"])
def test_batch_nonfinite_residual_is_not_converged(dev, value, precision):
    """A right-hand side with a NaN or an infinity, or one whose norm overflows
    (the base of relres is then infinite), in a system of each kernel and form:
    its relres is NaN and the batch has not converged; the others get what they
    get without it."""
    import torch
    rng = np.random.default_rng(12)
    for kind in ("dia", "wide"):
        sizes = (300, 513, 4097, 25600, 25601, 25700)   # the last two: k_batch_cg
        sys_ptr, rp, ci, v = batch_concat([_band_system(n, kind, rng) for n in sizes])
        b = gen.spmv((rp, ci, v), rng.uniform(-1, 1, int(sys_ptr[-1])))
        bad = b.copy()
        for s in (1, 3, 4):
            bad[sys_ptr[s] + 7] = value
        say(f"[batch nonfinite] {kind} {value} precision={precision}")
        B = XBatch(sys_ptr, rp, ci, v)
        x0, st0 = B.solve(b, tol=1e-9, maxiter=500, precision=precision)
        it0, rr0 = B.results()
        x1, st1 = B.solve(bad, tol=1e-9, maxiter=500, precision=precision)
        it1, rr1 = B.results()
        B.close()
        assert st0 == 0 and st1 == xsolver_amd.XS_NOT_CONVERGED
        for s, (lo, hi) in enumerate(zip(sys_ptr[:-1], sys_ptr[1:])):
            if s in (1, 3, 4):
                assert np.isnan(rr1[s]), (s, rr1[s])
            else:
                assert rr1[s] == rr0[s] and it1[s] == it0[s]
                assert np.array_equal(x1[lo:hi], x0[lo:hi])
        if precision == 0:
            from tests.test_zz_no_alloc import _noalloc
            rc, _, _, rr2, _ = _noalloc(torch, dev, sys_ptr, rp, ci, v, bad, 1e-9, 500)
            assert rc == 0 and np.array_equal(np.isnan(rr2), np.isnan(rr1))


def test_noalloc_small_systems_launch(dev):
    """A batch of mostly small systems runs in up to three launches of the
    allocation-free entry: the same results bit for bit as with the sizes
    known, each system solved by one of them, and a system whose columns leave
    its block reported by one, whatever its size."""
    import torch
    from tests.test_zz_no_alloc import _noalloc
    rng = np.random.default_rng(14)
    sizes = [10] * 60 + [4095, 25601, 1, 4096, 4097, 25600] + [37] * 60
    systems = [_band_system(n, "dia", rng) for n in sizes]
    sys_ptr, rp, ci, v = batch_concat(systems)
    n = int(sys_ptr[-1])
    assert 4096 < n and n // len(sizes) <= 1024
    b = gen.spmv((rp, ci, v), rng.uniform(-1, 1, n))
    say(f"[noalloc small] {len(sizes)} systems, n={n}")
    B = XBatch(sys_ptr, rp, ci, v)
    x, st = B.solve(b, tol=1e-9, maxiter=500)
    it, rr = B.results()
    B.close()
    assert st == 0
    for rep in range(2):
        rc, x2, it2, rr2, _ = _noalloc(torch, dev, sys_ptr, rp, ci, v, b, 1e-9, 500)
        assert rc == 0 and np.array_equal(x2, x) and np.array_equal(it2, it)
        assert np.array_equal(rr2, rr)
    bad = np.array(ci)
    off = [3, 60, 61, 64]   # 10, 4095, 25601 and 4097 rows
    for s in off:
        bad[rp[sys_ptr[s] + 1] - 1] = sys_ptr[s + 1]   # first row, into the next system
    rc, x3, it3, rr3, _ = _noalloc(torch, dev, sys_ptr, rp, bad, v, b, 1e-9, 500)
    ok = np.array([s not in off for s in range(len(sizes))])
    assert rc == 0 and np.all(it3[~ok] == -1) and np.all(np.isnan(rr3[~ok]))
    assert np.array_equal(it3[ok], it[ok]) and np.array_equal(rr3[ok], rr[ok])
