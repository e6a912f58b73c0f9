"""GPU tests of the generalized problem A x = lambda B x through the C-ABI:
the device LSPol solves, the generalized ChebAv and KPM against the dense
oracle (oracle/gen_oracle.py) on the same inputs, LanTrbounds against the
dense pencil spectrum, and the TESTS/Gen_Lap/LapPLanN.c flow with exact
per-slice counts.  Tolerances are written per test."""
import ctypes as C
import math

import numpy as np
import pytest
import scipy.linalg as sla
import scipy.sparse as sp

from oracle import gen_oracle as go
from oracle import oracle as orc
from pevsl_amd import capi, driver

pytestmark = pytest.mark.gpu


def banner(msg):
    print("\n[gpu case] " + msg, flush=True)


def dense(ia, ja, a, n):
    return sp.csr_matrix((a, ja, ia), shape=(n, n)).toarray()


class Gen:
    """A = 3-D Laplacian, B = chain Laplacian (the Gen_Lap pair) on the
    device, an instance in generalized mode with B-solve `bsol` ("host":
    exact Cholesky callback; "lspol": the library's LSPol B^{-1} on [2, 6])
    and L^T solve by LSPolSqrt(50, 1e-6, 2, 6)."""

    def __init__(self, lib, nx, ny, nz, bsol):
        self.lib = lib
        n = nx * ny * nz
        self.n = n
        self.Acsr = driver.laplacian3d(nx, ny, nz)
        self.Bcsr = driver.chain_laplacian(n)
        self.A = dense(*self.Acsr, n)
        self.B = dense(*self.Bcsr, n)
        self.MA = driver.Matrix(lib, *self.Acsr)
        self.MB = driver.Matrix(lib, *self.Bcsr)
        self.inst = driver.Instance(lib, self.MA)
        lib.pEVSL_SetBParcsr(self.inst.p, C.byref(self.MB.A))
        cho = sla.cho_factor(self.B)
        self.exact = lambda r: sla.cho_solve(cho, r)
        self.bdata = C.c_void_p()
        self.hs = None
        if bsol == "lspol":
            lib.pEVSL_SetupLSPolRec(50, 1e-12, 2.0, 6.0, C.byref(self.MB.A),
                                    C.byref(self.bdata))
            lib.pEVSL_SetBSol(self.inst.p, C.cast(lib.pEVSL_LSPolSol, C.c_void_p), self.bdata)
            mu, cc, dd = go.lspol_coeffs(lambda x: 1.0 / x, 2.0, 6.0, 50, 1e-12)
            self.solveB = lambda r: go.lspol_apply(self.B, mu, cc, dd, r)
        else:
            self.hs = driver.HostSolve(self.exact)
            self.hs.n = n
            lib.pEVSL_SetBSol(self.inst.p, self.hs.ptr(), None)
            self.solveB = self.exact
        self.lt = C.c_void_p()
        lib.pEVSL_SetupLSPolSqrt(50, 1e-6, 2.0, 6.0, C.byref(self.MB.A), C.byref(self.lt))
        lib.pEVSL_SetLTSol(self.inst.p, C.cast(lib.pEVSL_LSPolSol, C.c_void_p), self.lt)
        mus, ccs, dds = go.lspol_coeffs(lambda x: 1.0 / math.sqrt(x), 2.0, 6.0, 50, 1e-6)
        self.solveLT = lambda r: go.lspol_apply(self.B, mus, ccs, dds, r)
        assert lib.pEVSL_SetGenEig(self.inst.p) == 0
        self.lam = sla.eigh(self.A, self.B, eigvals_only=True)

    def close(self):
        self.inst.close()
        if self.bdata:
            self.lib.pEVSL_LSPolFree(self.bdata)
        self.lib.pEVSL_LSPolFree(self.lt)
        self.MA.free()
        self.MB.free()


def test_lspol_solves_on_device(lib):
    banner("LSPol B^{-1} and B^{-1/2} solves, chain Laplacian n=3000")
    n = 3000
    ia, ja, a = driver.chain_laplacian(n)
    M = driver.Matrix(lib, ia, ja, a)
    Bs = sp.csr_matrix((a, ja, ia), shape=(n, n))
    b = np.random.default_rng(1).standard_normal(n)
    try:
        for which, f, deg, tol in (("rec", lambda x: 1.0 / x, 50, 1e-12),
                                   ("sqrt", lambda x: 1.0 / math.sqrt(x), 50, 1e-6)):
            vd = C.c_void_p()
            setup = lib.pEVSL_SetupLSPolRec if which == "rec" else lib.pEVSL_SetupLSPolSqrt
            setup(deg, tol, 2.0, 6.0, C.byref(M.A), C.byref(vd))
            x = np.zeros(n)
            lib.pEVSL_LSPolSol(b.ctypes.data_as(capi.c_double_p),
                               x.ctypes.data_as(capi.c_double_p), vd)
            lib.pEVSL_LSPolFree(vd)
            mu, cc, dd = go.lspol_coeffs(f, 2.0, 6.0, deg, tol)
            ref = go.lspol_apply(Bs, mu, cc, dd, b)
            # same series, FP64 on both sides: relative 1e-12
            assert np.linalg.norm(x - ref) < 1e-12 * np.linalg.norm(ref)
            if which == "rec":
                ex = sp.linalg.spsolve(Bs.tocsc(), b)
                assert np.linalg.norm(x - ex) < 1e-10 * np.linalg.norm(ex)
    finally:
        M.free()


@pytest.mark.parametrize("bsol", ["host", "lspol"])
def test_chebav_generalized_matches_oracle(lib, bsol):
    banner("generalized ChebAv 8^3, B-solve %s" % bsol)
    g = Gen(lib, 8, 8, 8, bsol)
    try:
        lmin, lmax = g.lam[0] * 0.99, g.lam[-1] * 1.01
        pol, rc = driver.find_pol(lib, [1.5, 2.0, lmin, lmax])
        assert rc == 0
        mu = driver.pol_mu(pol)
        v = np.random.default_rng(2).uniform(-1, 1, g.n)
        y = np.zeros(g.n)
        X, Y = capi.Parvec(), capi.Parvec()
        lib.pEVSL_ParvecCreateShell(g.n, g.n, 0, 0, C.byref(X), v.ctypes.data_as(capi.c_double_p))
        lib.pEVSL_ParvecCreateShell(g.n, g.n, 0, 0, C.byref(Y), y.ctypes.data_as(capi.c_double_p))
        assert lib.pEVSL_ChebAv(g.inst.p, C.byref(pol), C.byref(X), C.byref(Y), None) == 0
        ref = go.cheb_av_gen(g.A, g.solveB, mu, pol.cc, pol.dd, v)
        # FP64 on both sides, same recurrence: relative 1e-11
        assert np.linalg.norm(y - ref) < 1e-11 * np.linalg.norm(ref), pol.deg
        lib.pEVSL_FreePol(C.byref(pol))
    finally:
        g.close()


@pytest.mark.parametrize("grid", [(5, 7, 3), (9, 3, 1), (3, 1, 1)])
def test_chebav_generalized_odd_order(lib, grid):
    """Odd orders: the work columns follow each other at odd offsets, and the
    last element of every vector takes part (two calls on other vectors, so
    that the work columns hold an earlier call's values)."""
    banner("generalized ChebAv, odd order %d x %d x %d" % grid)
    g = Gen(lib, *grid, "lspol")
    assert g.n % 2 == 1
    try:
        for seed in (3, 4):
            intv = [1.5, 2.5, 0.0, 6.0]
            pol, rc = driver.find_pol(lib, intv)
            assert rc == 0
            v = np.random.default_rng(seed).uniform(-1.0, 1.0, g.n)
            y = np.zeros(g.n)
            pv = [capi.Parvec() for _ in range(3)]
            for q, arr in zip(pv, (v, y, y)):
                lib.pEVSL_ParvecCreateShell(g.n, g.n, 0, 0, C.byref(q),
                                            arr.ctypes.data_as(capi.c_double_p))
            assert lib.pEVSL_ChebAv(g.inst.p, C.byref(pol), *[C.byref(q) for q in pv]) == 0
            mu = driver.pol_mu(pol)
            ref = go.cheb_av_gen(g.A, g.solveB, mu, pol.cc, pol.dd, v)
            lib.pEVSL_FreePol(C.byref(pol))
            # the same series in FP64 on both sides, as above
            assert np.linalg.norm(y - ref) < 1e-11 * np.linalg.norm(ref)
    finally:
        g.close()


def test_kpm_generalized_matches_oracle(lib):
    banner("generalized KPM 8^3, exact B-solve, LSPol L^T solve")
    g = Gen(lib, 8, 8, 8, "host")
    try:
        Mdeg, nvec = 30, 6
        lmin, lmax = g.lam[0] * 0.99, g.lam[-1] * 1.01
        xintv = np.array([1.5, 2.5, lmin, lmax])
        rc, mu, ecount = g.inst.kpmdos(Mdeg, 1, nvec, xintv)
        assert rc == 0
        # the same random vectors: the library's stream equals libc
        # srand(0)/rand() (pEVSL_Start seeds 0; KPM draws nvec x n values)
        orc.srand(0)
        vecs = np.array([orc.rand_vec(g.n) for _ in range(nvec)])
        ctr, wid = (lmax + lmin) / 2, (lmax - lmin) / 2
        dots = go.kpm_gen_dots(g.A, g.B, g.solveB, g.solveLT, vecs, Mdeg, ctr, wid)
        jac = orc.dampcf(Mdeg, 1)
        jac[0] = 1.0
        ref = np.zeros(Mdeg + 1)
        ref[0] = nvec * jac[0]
        ref[1:] = 2.0 * jac[1:] * dots.sum(0)
        ref /= nvec * np.pi
        # FP64 both sides; the L^T solve is the same series: relative 1e-10
        assert np.max(np.abs(mu - ref)) < 1e-10 * np.max(np.abs(ref))
        exact = np.sum((g.lam >= 1.5) & (g.lam <= 2.5))
        assert abs(ecount - exact) < 0.35 * exact  # 6 vectors: stochastic estimate
    finally:
        g.close()


def test_landos_generalized_matches_oracle(lib):
    """Generalized LanDosG (8^3 Gen_Lap pair, exact B-solve, LSPol L^T
    solve) against the dense oracle on the same random stream: the DOS curve
    to 1e-9 relative, the count within 30% of the dense pencil count."""
    banner("generalized LanDosG 8^3, 8 vectors, 30 steps")
    g = Gen(lib, 8, 8, 8, "host")
    try:
        lmin, lmax = g.lam[0] * 0.99, g.lam[-1] * 1.01
        xintv = [1.5, 2.5, lmin, lmax]
        rc, xd, yd, neig = g.inst.landos(8, 30, 200, xintv)
        assert rc == 0
        orc.srand(0)
        vecs = [orc.rand_vec(g.n) for _ in range(8)]
        oxd, oyd = go.landos_gen(g.A, g.B, g.solveB, g.solveLT, vecs, 30, 200, xintv)
        np.testing.assert_allclose(xd, oxd, rtol=0, atol=1e-15)
        assert np.max(np.abs(yd - oyd)) < 1e-9 * np.max(np.abs(oyd))
        oneig = orc.simpson(oxd, oyd)[-1] * g.n
        assert abs(neig - oneig) < 1e-8 * abs(oneig)
        exact = np.sum((g.lam >= 1.5) & (g.lam <= 2.5))
        assert abs(neig - exact) < 0.3 * exact
    finally:
        g.close()


@pytest.mark.parametrize("bsol", ["host", "lspol"])
def test_lantrbounds_generalized(lib, bsol):
    banner("generalized LanTrbounds 8^3, B-solve %s" % bsol)
    g = Gen(lib, 8, 8, 8, bsol)
    try:
        vinit = driver.rand_vinit(lib, g.n)
        rc, lo, hi = g.inst.lan_trbounds(50, 500, 1e-8, vinit, 1)
        assert rc == 0
        scale = max(abs(g.lam[0]), abs(g.lam[-1]))
        # bounds enclose the pencil's spectrum and are tight to the tolerance
        assert lo <= g.lam[0] + 1e-10 * scale and hi >= g.lam[-1] - 1e-10 * scale
        assert abs(lo - g.lam[0]) < 1e-6 * scale and abs(hi - g.lam[-1]) < 1e-6 * scale
    finally:
        g.close()


@pytest.mark.parametrize("deg", [1, 5, 40])
def test_chebiter_solves_match_oracle(lib, deg):
    """pEVSL_ChebIterSolv1/2 (device, host arrays) against the oracle's two
    forms on the same B and b: relative 1e-12; 40 steps on [2, 6] reach the
    exact solve (contraction (sqrt(3)-1)/(sqrt(3)+1) per step)."""
    banner("ChebIter solves, chain Laplacian n=3000, %d steps" % deg)
    n = 3000
    ia, ja, a = driver.chain_laplacian(n)
    M = driver.Matrix(lib, ia, ja, a)
    Bs = sp.csr_matrix((a, ja, ia), shape=(n, n))
    b = np.random.default_rng(3).standard_normal(n)
    cd = C.c_void_p()
    try:
        assert lib.pEVSL_ChebIterSetup(2.0, 6.0, deg, C.byref(M.A), C.byref(cd)) == 0
        for solv, ref in ((lib.pEVSL_ChebIterSolv1, go.chebiter_solv1(Bs, b, 2.0, 6.0, deg)),
                          (lib.pEVSL_ChebIterSolv2, go.chebiter_solv2(Bs, b, 2.0, 6.0, deg))):
            x = np.zeros(n)
            solv(b.ctypes.data_as(capi.c_double_p), x.ctypes.data_as(capi.c_double_p), cd)
            assert np.linalg.norm(x - ref) < 1e-12 * np.linalg.norm(ref)
            if deg == 40:
                ex = sp.linalg.spsolve(Bs.tocsc(), b)
                assert np.linalg.norm(x - ex) < 1e-10 * np.linalg.norm(ex)
    finally:
        if cd:
            lib.pEVSL_ChebIterFree(cd)
        M.free()


@pytest.mark.parametrize("bsol", ["host", "lspol", "chebiter"])
def test_gen_lap_flow_exact_counts(lib, bsol):
    """TESTS/Gen_Lap/LapPLanN.c defaults (8^3, [1.5, 2.5], 4 slices): every
    slice finds the dense pencil count, eigenvalues to 1e-10 relative,
    residuals ||A u - lambda B u|| < 1e-8."""
    banner("Gen_Lap flow 8^3 [1.5, 2.5] 4 slices, B-solve %s" % bsol)
    r = driver.gen_lap_run(8, 8, 8, 1.5, 2.5, 4, bsol=bsol)
    A = dense(*driver.laplacian3d(8, 8, 8), 512)
    B = dense(*driver.chain_laplacian(512), 512)
    lam = sla.eigh(A, B, eigvals_only=True)
    lmin, lmax = r["bounds"]
    assert lmin <= lam[0] + 1e-8 and lmax >= lam[-1] - 1e-8
    total = 0
    for s in r["slices"]:
        lo, hi = s["intv"]
        ex = lam[(lam >= lo) & (lam <= hi)]
        assert s["nev"] == len(ex), (s["slice"], s["nev"], len(ex))
        if len(ex):
            assert np.max(np.abs(s["lam"] - ex) / np.abs(ex)) < 1e-10
            assert np.all(np.asarray(s["res"]) < 1e-8)
        total += s["nev"]
    assert total == np.sum((lam >= r["sli"][0]) & (lam <= r["sli"][-1])) > 20


@pytest.mark.parametrize("bsol", ["tridiag", "chebiter"])
def test_genlap_c_driver(lib, bsol):
    """pevsl_amd/genlap_plan (C, TESTS/Gen_Lap/LapPLanN.c defaults) finds the
    dense pencil count in [1.5, 2.5]; "tridiag" is a host direct solver
    through pEVSL_SetBSol, the place of the reference's MUMPS solve."""
    import os
    import re
    import subprocess
    banner("genlap_plan C driver, B-solve %s" % bsol)
    exe = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pevsl_amd",
                       "genlap_plan")
    out = subprocess.run([exe, "-bsol", bsol], capture_output=True, text=True, timeout=240)
    print(out.stdout[-2000:], flush=True)
    assert out.returncode == 0, out.stderr
    total = int(re.search(r"total (\d+) eigenvalues", out.stdout).group(1))
    A = dense(*driver.laplacian3d(8, 8, 8), 512)
    B = dense(*driver.chain_laplacian(512), 512)
    lam = sla.eigh(A, B, eigvals_only=True)
    assert total == np.sum((lam >= 1.5) & (lam <= 2.5))
    for m in re.finditer(r"max res ([0-9.e+-]+)", out.stdout):
        assert float(m.group(1)) < 1e-8



@pytest.mark.parametrize("kind", [1, 2])
def test_lapchebiter_flow(lib, kind):
    """TESTS0/Chebiter/LapChebiter.c defaults: A = ParcsrLaplace(512, 1, 1),
    bounds by LanTrbounds(50, 200, 1e-8), 10 Chebyshev-iteration steps; the
    device solve equals the oracle's on the same b (1e-12), and for Saad's
    form the residual equals the closed-form residual polynomial
    T_10((theta - A)/delta)/T_10(theta/delta) b on the exact spectrum."""
    banner("LapChebiter flow, type %d" % kind)
    n, deg = 512, 10
    ia, ja, a = driver.chain_laplacian(n)
    M = driver.Matrix(lib, ia, ja, a)
    As = sp.csr_matrix((a, ja, ia), shape=(n, n))
    cd = C.c_void_p()
    try:
        inst = driver.Instance(lib, M)
        try:
            rc, lmin, lmax = inst.lan_trbounds(50, 200, 1e-8)
            assert rc == 0
        finally:
            inst.close()
        ex = 4 - 2 * np.cos(np.arange(1, n + 1) * np.pi / (n + 1))
        assert lmin <= ex.min() + 1e-8 and lmax >= ex.max() - 1e-8
        b = np.random.default_rng(5).uniform(-1, 1, n)
        x = np.zeros(n)
        assert lib.pEVSL_ChebIterSetup(lmin, lmax, deg, C.byref(M.A), C.byref(cd)) == 0
        solv = lib.pEVSL_ChebIterSolv1 if kind == 1 else lib.pEVSL_ChebIterSolv2
        solv(b.ctypes.data_as(capi.c_double_p), x.ctypes.data_as(capi.c_double_p), cd)
        ref = (go.chebiter_solv1 if kind == 1 else go.chebiter_solv2)(As, b, lmin, lmax, deg)
        assert np.linalg.norm(x - ref) < 1e-12 * np.linalg.norm(ref)
        res = b - As @ x
        if kind == 2:
            U = np.sin(np.outer(np.arange(1, n + 1), np.arange(1, n + 1)) * np.pi / (n + 1))
            U *= math.sqrt(2.0 / (n + 1))
            theta, delta = 0.5 * (lmax + lmin), 0.5 * (lmax - lmin)
            tk = np.polynomial.chebyshev.chebval((theta - ex) / delta, [0] * deg + [1])
            tk0 = np.polynomial.chebyshev.chebval(theta / delta, [0] * deg + [1])
            rref = U @ ((tk / tk0) * (U.T @ b))
            assert np.linalg.norm(res - rref) < 1e-12 * np.linalg.norm(b)
        # contraction of 10 steps on kappa ~ 3: far below the start residual
        assert np.linalg.norm(res) < 1e-4 * np.linalg.norm(b)
    finally:
        if cd:
            lib.pEVSL_ChebIterFree(cd)
        M.free()
