"""Diagonal layout: matrices of few constant diagonals (the main one may vary)
are read as a mask per row instead of CSR.  Every call that the layout takes
is compared with the plain CSR form of the same instance
(pEVSL_SetColumnOffsets16(0) switches both it and the 16-bit offsets off).

The filter's terms are the same in the same order, each rounded on its own,
so outputs are equal bit for bit; a product on the CSR side may sum a row in
several lanes, and both forms are compared with numpy to the rounding of a sum.
Which layout and which kernel a matrix gets is asserted as well
(pEVSL_DiagonalLayout, the per-kernel timers).
"""
import ctypes as C

import numpy as np
import pytest

from pevsl_amd import capi, driver

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    return capi.load()


def banded(n, offs, vary=None, drop=0.0, seed=0):
    """CSR with constant diagonals `offs` (value by diagonal), `vary` random
    diagonals among them, and a share `drop` of entries left out."""
    rng = np.random.default_rng(seed)
    r, c, v = [], [], []
    for o in sorted(offs):
        i = np.arange(max(0, -o), min(n, n - o))
        i = i[rng.random(len(i)) >= drop] if o != 0 else i
        r.append(i)
        c.append(i + o)
        val = np.full(len(i), 0.3 + 0.1 * (o % 7) - (0.05 if o > 0 else 0.0))
        if vary and o in vary:
            val = rng.uniform(1.0, 3.0, len(i))
        v.append(val)
    r, c, v = map(np.concatenate, (r, c, v))
    order = np.lexsort((c, r))
    ia = np.zeros(n + 1, np.int64)
    np.add.at(ia, r + 1, 1)
    return np.cumsum(ia).astype(np.int32), c[order].astype(np.int32), v[order]


def count_band(n, count):
    """Symmetric band of `count` diagonals, a varying main one among them if
    the count is odd."""
    up = [1 + k * k // 2 + k for k in range(count // 2)]
    ia, ja, a = banded(n, [-o for o in up] + up + [0] * (count % 2), vary=[0], seed=count)
    o = np.abs(ja - np.repeat(np.arange(n), np.diff(ia)))
    return ia, ja, np.where(o > 0, 0.3 + 0.1 * (o % 7), a)


CASES = {
    "1x1": lambda: banded(1, [0]),
    "one_row_block": lambda: banded(255, [-1, 0, 1]),
    "block_edge": lambda: banded(256, [-1, 0, 1]),
    "block_edge_1": lambda: banded(257, [-1, 0, 1], vary=[0]),
    "3_of_4_dropped": lambda: banded(1111, [-5, 0, 5], drop=0.3),
    "4_no_main": lambda: banded(1000, [-3, -1, 1, 3]),
    # several degrees per launch: one window, many windows, the widest band
    "chain_wide": lambda: banded(70001, [-1, 0, 1], vary=[0]),
    "band_31": lambda: banded(20011, [-31, -30, 0, 30, 31], drop=0.1),
    "band_400": lambda: banded(8000, [-400, -20, -1, 0, 1, 20, 400]),
    "lower_only": lambda: banded(5000, [-3, -2, 0]),
    "lap2d": lambda: driver.laplacian3d(31, 17, 1),
    "lap3d": lambda: driver.laplacian3d(13, 11, 7),
    "6_diags": lambda: banded(2000, [-90, -7, 0, 7, 90, 91], drop=0.1, vary=[0]),
    "8_diags": lambda: banded(3001, [-700, -31, -1, 0, 1, 31, 700, 2999], drop=0.1, vary=[0]),
    "9_diags": lambda: banded(3001, [-700, -31, -2, -1, 0, 1, 2, 31, 700], drop=0.1, vary=[0]),
    "32_diags": lambda: banded(2500, list(range(-16, 16)), vary=[0]),
    # the last count of each kernel above 8 diagonals, and the first of the next
    **{"count_%d" % k: (lambda k=k: count_band(1500 + k, k)) for k in
       (10, 13, 14, 19, 20, 27, 28)},
    "empty_rows": lambda: banded(700, [-9, 9], drop=0.45),
    # no such layout: 33 diagonals, a second varying diagonal, mostly absent
    "33_diags": lambda: banded(900, list(range(-16, 17))),
    "two_vary": lambda: banded(900, [-1, 0, 1], vary=[0, 1]),
    "sparse_diags": lambda: banded(900, [-40, -20, 0, 20, 40], drop=0.9),
    # ...and a value that FP32 does not hold, which zero must not multiply
    "beyond_fp32": lambda: (lambda ia, ja, a: (ia, ja, np.where(
        ja - np.repeat(np.arange(900), np.diff(ia)) == 3, 1e39, a)))(
            *banded(900, [-1, 0, 3], drop=0.2)),
}


def filt(lib, M, pol, v, prec, on):
    inst = driver.Instance(lib, M, prec=prec, col16=bool(on))
    try:
        y = np.full(M.n, np.nan)
        pv, py = capi.Parvec(), capi.Parvec()
        for p, a in ((pv, v), (py, y)):
            lib.pEVSL_ParvecCreateShell(M.n, M.n, 0, 0, C.byref(p),
                                        a.ctypes.data_as(capi.c_double_p))
        assert lib.pEVSL_ChebAv(inst.p, C.byref(pol), C.byref(pv), C.byref(py), None) == 0
    finally:
        inst.close()
    return y


@pytest.mark.parametrize("name", sorted(CASES))
def test_filter_equals_csr(lib, name):
    print("\n[gpu case] diagonal layout, filter, %s" % name, flush=True)
    ia, ja, a = CASES[name]()
    n = len(ia) - 1
    M = driver.Matrix(lib, ia, ja, a)
    rad = float(np.max(np.bincount(np.repeat(np.arange(n), np.diff(ia)), np.abs(a), n)))
    rng = np.random.default_rng(n)
    try:
        v = rng.uniform(-1, 1, n)
        # every way a run of degrees can end in the update of y
        for deg in (1, 2, 3, 4, 5, 6, 17, 70):
            mu = rng.uniform(-1, 1, deg + 1)
            pol = capi.Polparams()
            pol.deg, pol.cc, pol.dd = deg, 0.1 * rad, 1.1 * rad
            pol.mu = mu.ctypes.data_as(capi.c_double_p)
            for prec in (capi.PEVSL_PREC_FP64, capi.PEVSL_PREC_FP32):
                np.testing.assert_array_equal(filt(lib, M, pol, v, prec, 1),
                                              filt(lib, M, pol, v, prec, 0))
    finally:
        M.free()


@pytest.mark.parametrize("name", sorted(CASES))
def test_product_equals_csr(lib, name):
    print("\n[gpu case] diagonal layout, product, %s" % name, flush=True)
    ia, ja, a = CASES[name]()
    n = len(ia) - 1
    M = driver.Matrix(lib, ia, ja, a)
    try:
        x = np.random.default_rng(n).uniform(-1, 1, n)
        y = M.matvec(x)
        rows = np.repeat(np.arange(n), np.diff(ia))
        ref = np.bincount(rows, a * x[ja], n)
        mag = np.bincount(rows, np.abs(a * x[ja]), n)
        # two summation orders of at most 33 terms
        assert np.all(np.abs(y - ref) <= 33 * 2.3e-16 * mag)
    finally:
        M.free()


@pytest.mark.parametrize("mat", ["lap3d", "pot", "9_diags"])
@pytest.mark.parametrize("prec,kind,width", [(0, 1, 2), (0, 1, 4), (0, 1, 8), (0, 1, 16),
                                             (1, 1, 2), (1, 1, 4), (1, 2, 8), (1, 1, 16),
                                             (1, 2, 32)])
def test_block_steps_equal_csr(lib, mat, prec, kind, width):
    """Batched solves of 7 slices (groups of the width and a remainder), with
    slices whose degrees differ: same steps, eigenvalues and residuals."""
    print("\n[gpu case] diagonal layout, block %s prec %d kind %d width %d" % (
        mat, prec, kind, width), flush=True)
    if mat == "9_diags":
        ia, ja, a = banded(1201, [-90, -11, -2, -1, 0, 1, 2, 11, 90], vary=[0], seed=2)
        top = 20.0
        i = np.repeat(np.arange(1201), np.diff(ia))
        a = np.where(ja == i, 10.0 + a, 0.3 + 0.1 * (np.abs(ja - i) % 7))  # symmetric
    else:
        ia, ja, a = driver.laplacian3d(9, 8, 11)
        top = 12.0
        if mat == "pot":
            i = np.repeat(np.arange(len(ia) - 1), np.diff(ia))
            a = np.where(ja == i, a + np.random.default_rng(3).random(len(a)), a)
            top = 13.0
    M = driver.Matrix(lib, ia, ja, a)
    edges = np.array([0.02, 0.1, 0.15, 0.3, 0.33, 0.5, 0.55, 0.65]) * top
    intvs = [[edges[i], edges[i + 1], 0.0, top] for i in range(7)]
    pols = [driver.find_pol(lib, iv)[0] for iv in intvs]
    vinit = np.random.default_rng(5).uniform(-1, 1, M.n)
    runs = []
    try:
        for on in (True, False):
            inst = driver.Instance(lib, M, prec=prec, block_rowkernel=kind, block_width=width,
                                   col16=on)
            try:
                rc, outs = driver.cheblan_batch(inst, intvs, [60] * 7, 1e-8, vinit, pols)
                assert rc == 0
                runs.append(outs)
            finally:
                inst.close()
    finally:
        for p_ in pols:
            lib.pEVSL_FreePol(C.byref(p_))
        M.free()
    for x, y in zip(*runs):
        assert x["info"]["its"] == y["info"]["its"]
        assert x["info"]["tr"] == y["info"]["tr"]
        np.testing.assert_array_equal(x["lam"], y["lam"])
        np.testing.assert_array_equal(x["res"], y["res"])


def test_rectangular_product(lib):
    print("\n[gpu case] diagonal layout, rectangular products", flush=True)
    for nr, nc in ((300, 40), (40, 300)):
        k = min(nr, nc)
        ia = np.minimum(np.arange(nr + 1), k).astype(np.int32)
        ja, a = np.arange(k, dtype=np.int32), np.full(k, 2.5)
        csr = capi.Csr(nr, nc, ia.ctypes.data_as(capi.c_int_p), ja.ctypes.data_as(capi.c_int_p),
                       a.ctypes.data_as(capi.c_double_p))
        A = capi.Parcsr()
        assert lib.pEVSL_ParcsrCreate(nr, nc, None, None, C.byref(A), capi.MPI_COMM_WORLD) == 0
        assert lib.pEVSL_ParcsrSetup(C.byref(csr), C.byref(A)) == 0
        x, y = np.random.default_rng(1).uniform(-1, 1, nc), np.full(nr, np.nan)
        X, Y = capi.Parvec(), capi.Parvec()
        lib.pEVSL_ParvecCreateShell(nc, nc, 0, 0, C.byref(X), x.ctypes.data_as(capi.c_double_p))
        lib.pEVSL_ParvecCreateShell(nr, nr, 0, 0, C.byref(Y), y.ctypes.data_as(capi.c_double_p))
        lib.pEVSL_ParcsrMatvec(C.byref(A), C.byref(X), C.byref(Y))
        lib.pEVSL_ParcsrFree(C.byref(A))
        ref = np.zeros(nr)
        ref[:k] = 2.5 * x[:k]
        np.testing.assert_array_equal(y, ref)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("Mdeg,nvec", [(1, 1), (2, 3), (5, 33), (30, 70)])
def test_kpm_on_both_layouts(lib, prec, Mdeg, nvec):
    """Moments of odd and even counts, single vectors, padded groups and more
    vectors than one group holds, on the diagonal layout and as CSR, against
    the recurrence in FP64 numpy on the same rand() stream."""
    print("\n[gpu case] KPM Mdeg %d nvec %d prec %d" % (Mdeg, nvec, prec), flush=True)
    ia, ja, a = driver.laplacian3d(7, 9, 5)
    n = len(ia) - 1
    dense = np.zeros((n, n))
    dense[np.repeat(np.arange(n), np.diff(ia)), ja] = a
    libc = C.CDLL(None)
    libc.srand(7)
    t = 2147483647.0 / 2
    v = (np.array([libc.rand() for _ in range(n * nvec)], float).reshape(nvec, n).T - t) / t
    v /= np.linalg.norm(v, axis=0)
    u, um, dots = v, None, []
    for k in range(Mdeg):
        w = (dense @ u - 6.0 * u) * ((2.0 if k else 1.0) / 6.0) - (um if k else 0.0)
        um, u = u, w
        dots.append(float((w * v).sum()))
    # damping 0: mu_k = 2 / (nvec pi) sum of the dots
    ref = np.array([1.0 / np.pi] + [2.0 / (nvec * np.pi) * d for d in dots])
    M = driver.Matrix(lib, ia, ja, a)
    try:
        for on in (True, False):
            inst = driver.Instance(lib, M, prec=prec, col16=on)
            try:
                lib.pEVSL_RandSeed(7)
                rc, mu, _ = inst.kpmdos(Mdeg, 0, nvec, [3.0, 5.0, 0.0, 12.0])
            finally:
                inst.close()
            assert rc == 0
            # FP64: a few roundings of unit quantities; FP32 as CSR: the path's
            # 2e-5; on the layout: vectors rounded to FP32 once a step and
            # everything else in FP64, which numpy puts at up to 1.9e-9 here
            assert np.max(np.abs(mu - ref)) <= (1e-13 if prec == 0 else 6e-9 if on else 2e-5)
    finally:
        M.free()


@pytest.mark.parametrize("prec", [0, 1])
def test_kpm_several_runs_of_rows(lib, prec):
    """Enough rows that each workgroup takes several runs of them, the last
    ones partly or wholly past the end, against the recurrence in FP64."""
    print("\n[gpu case] KPM several runs, prec %d" % prec, flush=True)
    sp = pytest.importorskip("scipy.sparse")
    ia, ja, a = driver.laplacian3d(33, 33, 31)
    n, nvec, Mdeg = len(ia) - 1, 33, 5
    A = sp.csr_matrix((a, ja, ia), shape=(n, n))
    M = driver.Matrix(lib, ia, ja, a)
    try:
        inst = driver.Instance(lib, M, prec=prec)
        try:
            lib.pEVSL_RandSeed(11)
            rc, mu, _ = inst.kpmdos(Mdeg, 0, nvec, [3.0, 5.0, 0.0, 12.0])
        finally:
            inst.close()
    finally:
        M.free()
    assert rc == 0
    libc = C.CDLL(None)
    libc.srand(11)
    t = 2147483647.0 / 2
    v = (np.array([libc.rand() for _ in range(n * nvec)], float).reshape(nvec, n).T - t) / t
    v /= np.linalg.norm(v, axis=0)
    u, um, ref = v, None, [1.0 / np.pi]
    for k in range(Mdeg):
        w = (A @ u - 6.0 * u) * ((2.0 if k else 1.0) / 6.0) - (um if k else 0.0)
        um, u = u, w
        ref.append(2.0 / (nvec * np.pi) * float((w * v).sum()))
    # as in test_kpm_on_both_layouts; numpy: 9.4e-11 (1.4e-8 in FP32 arithmetic)
    assert np.max(np.abs(mu - np.array(ref))) <= (1e-13 if prec == 0 else 2e-9)


@pytest.mark.parametrize("grid,nvec", [((20, 20, 20), 1), ((7, 9, 5), 4)])
def test_kpm_fp32_rounds_once_a_step(lib, grid, nvec):
    """Two moments per product keep FP32 vectors' accuracy only with the row
    sums and the recurrence in FP64.  Bound: four times the error that numpy
    finds for that form on the same vectors; the same form in FP32 arithmetic
    throughout is beyond it."""
    print("\n[gpu case] KPM accuracy in FP32, %dx%dx%d, %d vectors" % (*grid, nvec), flush=True)
    sp = pytest.importorskip("scipy.sparse")
    ia, ja, a = driver.laplacian3d(*grid)
    n, Mdeg, f = len(ia) - 1, 200, np.float32
    A = sp.csr_matrix((a, ja, ia), shape=(n, n))
    libc = C.CDLL(None)
    libc.srand(7)
    t = 2147483647.0 / 2
    v = (np.array([libc.rand() for _ in range(n * nvec)], float).reshape(nvec, n).T - t) / t
    v /= np.linalg.norm(v, axis=0)

    def scaled(dots):
        return np.array([2.0 / (nvec * np.pi) * float(np.sum(d)) for d in dots])

    u, um, dots = v, 0.0, []
    for k in range(Mdeg):
        um, u = u, (A @ u - 6.0 * u) * ((2.0 if k else 1.0) / 6.0) - um
        dots.append((u * v).sum(0))
    ref = scaled(dots)

    def two_moments(arith):
        B, ctr = A.astype(arith), arith(6.0)
        U, um = [v.astype(f)], np.zeros((n, nvec), f)
        for k in range(Mdeg // 2):
            x = U[-1].astype(arith)
            w = (B @ x - ctr * x) * arith((2.0 if k else 1.0) / 6.0) - um.astype(arith)
            um = U[-1]
            U.append(w.astype(f))
        D = [x.astype(float) for x in U]
        vv, d1 = (D[0] * D[0]).sum(0), (D[1] * D[0]).sum(0)
        dots = [d1 / vv]
        for k in range(2, Mdeg + 1):
            j = k // 2
            dots.append(((2 * (D[j] * D[j]).sum(0) - vv) if k % 2 == 0
                         else (2 * (D[j + 1] * D[j]).sum(0) - d1)) / vv)
        return np.max(np.abs(scaled(dots) - ref))

    bound = 4 * two_moments(np.float64)
    assert two_moments(f) > bound
    M = driver.Matrix(lib, ia, ja, a)
    try:
        inst = driver.Instance(lib, M, prec=1)
        try:
            lib.pEVSL_RandSeed(7)
            rc, mu, _ = inst.kpmdos(Mdeg, 0, nvec, [3.0, 5.0, 0.0, 12.0])
        finally:
            inst.close()
    finally:
        M.free()
    assert rc == 0
    assert np.max(np.abs(mu[1:] - ref)) <= bound


def not_symmetric(which):
    """Matrices for which the products of neighbouring vectors give no
    moments, and one (unsorted columns) whose symmetry is not looked for."""
    rng = np.random.default_rng(21)
    if which == "diagonals":
        return banded(700, [-3, -2, 0, 1])
    if which == "values":  # symmetric pattern with a diagonal layout
        return banded(700, [-1, 0, 1])
    if which == "one_entry":  # a symmetric layout with one entry missing
        ia, ja, a = driver.laplacian3d(9, 8, 7)
        k = int(np.flatnonzero(ja != np.repeat(np.arange(len(ia) - 1), np.diff(ia)))[100])
        row = int(np.searchsorted(ia, k, side="right")) - 1
        ia = ia.copy()
        ia[row + 1:] -= 1
        return ia, np.delete(ja, k), np.delete(a, k)
    if which == "csr":
        n, m = 600, 5
        ja = np.concatenate([np.sort(rng.choice(n, m, replace=False)) for _ in range(n)])
        return (np.arange(n + 1, dtype=np.int32) * m, ja.astype(np.int32),
                rng.uniform(-1, 1, n * m))
    ia, ja, a = driver.laplacian3d(9, 8, 7)  # "unsorted"
    for i in range(len(ia) - 1):
        ja[ia[i]:ia[i + 1]] = ja[ia[i]:ia[i + 1]][::-1].copy()
        a[ia[i]:ia[i + 1]] = a[ia[i]:ia[i + 1]][::-1].copy()
    return ia, ja, a


@pytest.mark.parametrize("which", ["diagonals", "values", "one_entry", "csr", "unsorted"])
@pytest.mark.parametrize("prec", [0, 1])
def test_kpm_without_symmetry(lib, which, prec):
    """<v, T_k v> of a matrix that is not symmetric, against the recurrence in
    FP64 numpy: one product per moment, whatever the layout."""
    print("\n[gpu case] KPM without symmetry, %s prec %d" % (which, prec), flush=True)
    ia, ja, a = not_symmetric(which)
    n, nvec, Mdeg = len(ia) - 1, 5, 8
    dense = np.zeros((n, n))
    np.add.at(dense, (np.repeat(np.arange(n), np.diff(ia)), ja), a)
    # |A| <= sqrt(|A|_1 |A|_inf); T_k of a non-normal matrix may still grow
    c0 = 6.0 if which in ("one_entry", "unsorted") else 0.0
    off = np.abs(dense - c0 * np.eye(n))
    wid = 2.0 * float(np.sqrt(off.sum(0).max() * off.sum(1).max()))
    libc = C.CDLL(None)
    libc.srand(7)
    t = 2147483647.0 / 2
    v = (np.array([libc.rand() for _ in range(n * nvec)], float).reshape(nvec, n).T - t) / t
    v /= np.linalg.norm(v, axis=0)
    u, um, ref, top = v, None, [1.0 / np.pi], 1.0
    for k in range(Mdeg):
        w = (dense @ u - c0 * u) * ((2.0 if k else 1.0) / wid) - (um if k else 0.0)
        um, u = u, w
        top = max(top, float(np.linalg.norm(w, axis=0).max()))
        ref.append(2.0 / (nvec * np.pi) * float((w * v).sum()))
    M = driver.Matrix(lib, ia, ja, a)
    try:
        inst = driver.Instance(lib, M, prec=prec)
        try:
            lib.pEVSL_RandSeed(7)
            rc, mu, _ = inst.kpmdos(Mdeg, 0, nvec, [c0 - 0.1, c0 + 0.1, c0 - wid, c0 + wid])
            assert inst.stats()["n_mvA"] == nvec * Mdeg
        finally:
            inst.close()
    finally:
        M.free()
    assert rc == 0
    # as in test_kpm_on_both_layouts, times the vectors' largest norm
    assert np.max(np.abs(mu - np.array(ref))) <= top * (1e-13 if prec == 0 else 2e-5)


# diagonals and slots of each case's layout (0: none)
LAYOUT = {"1x1": 1, "one_row_block": 3, "block_edge": 3, "block_edge_1": 3, "3_of_4_dropped": 3,
          "4_no_main": 4, "chain_wide": 3, "band_31": 5, "band_400": 7, "lower_only": 3, "lap2d": 5,
          "lap3d": 7, "6_diags": 6, "8_diags": 8, "9_diags": 9, "32_diags": 32, "empty_rows": 2,
          "33_diags": 0, "two_vary": 0, "sparse_diags": 0, "beyond_fp32": 0,
          **{"count_%d" % k: k for k in (10, 13, 14, 19, 20, 27, 28)}}


@pytest.mark.parametrize("name", sorted(CASES))
def test_layout_is_taken(lib, name):
    """The cases above run, or do not run, on the layout they are meant for,
    with spare slots of at most a third from two diagonals on."""
    print("\n[gpu case] diagonal layout taken, %s" % name, flush=True)
    M = driver.Matrix(lib, *CASES[name]())
    slots = C.c_int(-1)
    try:
        for on in (True, False):
            inst = driver.Instance(lib, M, col16=on)
            try:
                nd = lib.pEVSL_DiagonalLayout(inst.p, C.byref(slots))
            finally:
                inst.close()
            assert nd == (LAYOUT[name] if on else 0)
            assert slots.value >= nd and (nd < 2 or 3 * (slots.value - nd) <= slots.value)
            assert nd > 0 or slots.value == 0
    finally:
        M.free()


COUNTS = [9, 10, 13, 14, 19, 20, 27, 28, 32]


@pytest.mark.parametrize("prec,kind,width", [(0, 1, 4), (1, 2, 8), (1, 1, 2)])
@pytest.mark.parametrize("count", COUNTS)
def test_block_steps_by_diagonal_count(lib, count, prec, kind, width):
    print("\n[gpu case] diagonal layout, block, %d diagonals prec %d kind %d width %d" % (
        count, prec, kind, width), flush=True)
    M = driver.Matrix(lib, *count_band(901, count))
    rad = 20.0
    intvs = [[0.05 * rad * i, 0.05 * rad * (i + 0.9), -rad, rad] for i in range(5)]
    pols = [driver.find_pol(lib, iv)[0] for iv in intvs]
    vinit = np.random.default_rng(5).uniform(-1, 1, M.n)
    runs = []
    try:
        for on in (True, False):
            inst = driver.Instance(lib, M, prec=prec, block_rowkernel=kind, block_width=width,
                                   col16=on)
            try:
                assert lib.pEVSL_DiagonalLayout(inst.p, None) == (count if on else 0)
                rc, outs = driver.cheblan_batch(inst, intvs, [40] * 5, 1e-8, vinit, pols)
                assert rc == 0
                runs.append(outs)
            finally:
                inst.close()
    finally:
        for p_ in pols:
            lib.pEVSL_FreePol(C.byref(p_))
        M.free()
    for x, y in zip(*runs):
        assert x["info"]["its"] == y["info"]["its"]
        assert x["info"]["tr"] == y["info"]["tr"]
        np.testing.assert_array_equal(x["lam"], y["lam"])
        np.testing.assert_array_equal(x["res"], y["res"])


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("count", COUNTS)
def test_kpm_by_diagonal_count(lib, count, prec):
    print("\n[gpu case] KPM, %d diagonals prec %d" % (count, prec), flush=True)
    ia, ja, a = count_band(901, count)
    n, nvec, Mdeg, rad = 901, 9, 11, 24.0
    dense = np.zeros((n, n))
    dense[np.repeat(np.arange(n), np.diff(ia)), ja] = a
    libc = C.CDLL(None)
    libc.srand(3)
    t = 2147483647.0 / 2
    v = (np.array([libc.rand() for _ in range(n * nvec)], float).reshape(nvec, n).T - t) / t
    v /= np.linalg.norm(v, axis=0)
    u, um, ref = v, None, [1.0 / np.pi]
    for k in range(Mdeg):
        w = (dense @ u) * ((2.0 if k else 1.0) / rad) - (um if k else 0.0)
        um, u = u, w
        ref.append(2.0 / (nvec * np.pi) * float((w * v).sum()))
    M = driver.Matrix(lib, ia, ja, a)
    try:
        inst = driver.Instance(lib, M, prec=prec)
        try:
            lib.pEVSL_RandSeed(3)
            rc, mu, _ = inst.kpmdos(Mdeg, 0, nvec, [1.0, 2.0, -rad, rad])
            assert inst.stats()["n_mvA"] == nvec * ((Mdeg + 1) // 2)  # on the layout
        finally:
            inst.close()
    finally:
        M.free()
    assert rc == 0
    # as in test_kpm_on_both_layouts (numpy: at most 1.6e-9)
    assert np.max(np.abs(mu - np.array(ref))) <= (1e-13 if prec == 0 else 5e-9)


# kernel of a filter of degree 70 in FP64: several degrees per launch on chains
# and bands of at most 8 diagonals, one above that or where the window of a
# workgroup would not fit the band, the CSR-stream kernel without a layout
STEP = {"chain_wide": "k_cheb_multi<double,3>", "band_31": "k_cheb_multi<double,5>",
        "lap2d": "k_cheb_multi<double,5>", "block_edge_1": "k_cheb_multi<double,3>",
        "band_400": "k_cheb_multi<double,7>", "8_diags": "k_cheb_dia<double,8>",
        "9_diags": "k_cheb_dia<double,9>",
        "count_10": "k_cheb_dia<double,13>", "32_diags": "k_cheb_dia<double,32>",
        "33_diags": "k_cheb_stream<double>", "two_vary": "k_cheb_stream<double>",
        "sparse_diags": "k_cheb_stream<double>"}


@pytest.mark.parametrize("name", sorted(STEP))
def test_filter_runs_the_kernel_meant_for_the_layout(lib, name):
    """...and its launches and bytes are counted as they ran."""
    print("\n[gpu case] filter kernel, %s" % name, flush=True)
    ia, ja, a = CASES[name]()
    n, deg = len(ia) - 1, 70
    M = driver.Matrix(lib, ia, ja, a)
    try:
        inst = driver.Instance(lib, M)
        try:
            mu = np.linspace(1, 2, deg + 1)
            pol = capi.Polparams()
            pol.deg, pol.cc, pol.dd = deg, 0.0, 1e3
            pol.mu = mu.ctypes.data_as(capi.c_double_p)
            v, y = np.ones(n), np.zeros(n)
            pv, py = capi.Parvec(), capi.Parvec()
            for p, x in ((pv, v), (py, y)):
                lib.pEVSL_ParvecCreateShell(n, n, 0, 0, C.byref(p),
                                            x.ctypes.data_as(capi.c_double_p))
            assert lib.pEVSL_ChebAv(inst.p, C.byref(pol), C.byref(pv), C.byref(py), None) == 0
            kt, ks = inst.kernel_times(), inst.kernel_stats()
        finally:
            inst.close()
    finally:
        M.free()
    assert list(kt) == [STEP[name]]
    t = kt[STEP[name]]
    assert ks["filter_steps"] == deg
    assert ks["filter_launches"] == t["launches"] and ks["filter_bytes"] == t["bytes"]
    if "multi" in STEP[name]:
        assert t["launches"] * 2 <= deg
    else:
        assert t["launches"] == deg
        # at least the two vectors that every degree reads or writes
        assert t["bytes"] >= 2.0 * 8 * n * deg


@pytest.mark.parametrize("name", sorted(CASES))
def test_product_on_and_off_the_layout(lib, name):
    """pEVSL_DeviceMatvec through the layout and through plain CSR: each within
    the rounding of the row's sum, in whichever order."""
    print("\n[gpu case] product on and off the layout, %s" % name, flush=True)
    ia, ja, a = CASES[name]()
    n = len(ia) - 1
    x = np.random.default_rng(n).uniform(-1, 1, n)
    rows = np.repeat(np.arange(n), np.diff(ia))
    ref = np.bincount(rows, a * x[ja], n)
    mag = np.bincount(rows, np.abs(a * x[ja]), n)
    M = driver.Matrix(lib, ia, ja, a)
    hip, d, nb = C.CDLL("libamdhip64.so"), C.c_void_p(), C.c_size_t(8 * n)
    try:
        assert hip.hipMalloc(C.byref(d), C.c_size_t(16 * n)) == 0
        dx, dy = C.c_void_p(d.value), C.c_void_p(d.value + 8 * n)
        for on in (True, False):
            y = np.full(n, np.nan)
            inst = driver.Instance(lib, M, col16=on)
            try:
                assert hip.hipMemcpy(dx, x.ctypes.data_as(C.c_void_p), nb, 1) == 0
                assert hip.hipMemcpy(dy, y.ctypes.data_as(C.c_void_p), nb, 1) == 0
                assert lib.pEVSL_DeviceMatvec(inst.p, dx, dy) == 0
                assert hip.hipMemcpy(y.ctypes.data_as(C.c_void_p), dy, nb, 2) == 0
            finally:
                inst.close()
            # two summation orders of at most 33 terms
            assert np.all(np.abs(y - ref) <= 33 * 2.3e-16 * mag), on
    finally:
        if d.value:
            hip.hipFree(d)
        M.free()


@pytest.mark.parametrize("which", ["lap3d", "pot", "two_vary"])
@pytest.mark.parametrize("prec,kind", [(0, 0), (0, 1), (0, 3), (1, 1), (1, 2), (1, 4), (1, 5)])
def test_benchblock_counts_the_form_it_reads(lib, which, prec, kind):
    """Bytes of a timed block step: mask bytes (and the varying main diagonal)
    for the row steps of a matrix read through its diagonals, the CSR matrix
    for every other kernel; vector passes by kernel."""
    print("\n[gpu case] block step bytes, %s prec %d kind %d" % (which, prec, kind), flush=True)
    ia, ja, a = driver.laplacian3d(13, 11, 7) if which == "pot" else CASES[which]()
    n, nnz, B, elem = len(ia) - 1, int(ia[-1]), 8, 4 if prec else 8
    if which == "pot":
        a = np.where(ja == np.repeat(np.arange(n), np.diff(ia)),
                     a + np.random.default_rng(3).random(nnz), a)
    M = driver.Matrix(lib, ia, ja, a)
    sec, got = C.c_double(), C.c_double()
    try:
        for on in (True, False):
            inst = driver.Instance(lib, M, prec=prec, block_rowkernel=kind, col16=on)
            try:
                assert lib.pEVSL_BenchBlock(inst.p, B, 2, C.byref(sec), C.byref(got)) == 0
            finally:
                inst.close()
            if on and kind in (1, 2) and which != "two_vary":
                mat = n * (1 + (elem if which == "pot" else 0))
            else:
                idx = 2 if on and kind in (1, 2) else 4
                mat = nnz * (elem + idx) + 4 * (n + 1)
            passes = {0: 5.0, 1: 11 / 3.0, 3: 11 / 3.0}.get(kind, 4.0)
            assert abs(got.value - (mat + passes * n * B * elem)) <= 1e-9 * got.value
            assert sec.value > 0
    finally:
        M.free()
