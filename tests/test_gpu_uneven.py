"""CSR-stream kernels at row lengths around their limits: rows of up to
kUnevenRow = 64 entries are summed by one thread, longer ones by a wave, rows
beyond a block's 2,048 staged entries by the whole workgroup; blocks end at 256
rows or 2,048 entries."""
import ctypes as C

import numpy as np
import pytest

from pevsl_amd import capi, driver

pytestmark = pytest.mark.gpu

# row lengths, repeated over the matrix
LENGTHS = {
    "one": [1], "edge64": [63, 64, 65], "all_long": [129], "one_long": [2] * 300 + [2048],
    "beyond_block": [5, 2049, 0, 7], "waves": [65] * 9 + [1] * 250, "empty_tail": [70] + [0] * 600,
    "mixed": [3, 900, 64, 66, 0, 1000, 200],
}


@pytest.mark.parametrize("name", sorted(LENGTHS))
def test_rows_of_every_length(name):
    print("\n[gpu case] CSR-stream rows, %s" % name, flush=True)
    lib = capi.load()
    n, rng = 2500, np.random.default_rng(len(name))
    lens = np.resize(LENGTHS[name], n)
    ia = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ja = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in lens]).astype(np.int32)
    a = rng.uniform(-1, 1, len(ja))
    x = rng.uniform(-1, 1, n)
    rows = np.repeat(np.arange(n), lens)
    ref = np.bincount(rows, a * x[ja], n)
    mag = np.bincount(rows, np.abs(a * x[ja]), n)
    M = driver.Matrix(lib, ia, ja, a)
    inst = driver.Instance(lib, M)
    try:
        # any summation order of m terms is within m ulp of the absolute sum
        assert np.all(np.abs(M.matvec(x) - ref) <= 2.3e-16 * lens * mag)
        # degree 1 with cc = 0, dd = 1, mu = (0, 1): the filter is the product
        for prec, eps in ((capi.PEVSL_PREC_FP64, 2.3e-16), (capi.PEVSL_PREC_FP32, 1.2e-7)):
            lib.pEVSL_SetFilterPrecision(inst.p, prec)
            mu, y = np.array([0.0, 1.0]), np.full(n, np.nan)
            pol = capi.Polparams()
            pol.deg, pol.cc, pol.dd = 1, 0.0, 1.0
            pol.mu = mu.ctypes.data_as(capi.c_double_p)
            pv, py = capi.Parvec(), capi.Parvec()
            for p, arr in ((pv, x), (py, y)):
                lib.pEVSL_ParvecCreateShell(n, n, 0, 0, C.byref(p),
                                            arr.ctypes.data_as(capi.c_double_p))
            assert lib.pEVSL_ChebAv(inst.p, C.byref(pol), C.byref(pv), C.byref(py), None) == 0
            # two more roundings per product for the FP32 copies of a and x
            assert np.all(np.abs(y - ref) <= eps * (lens + 2) * mag)
    finally:
        inst.close()
        M.free()
