"""Timed cases of the library's work, through its public entry points.

Kinds of case:

matvec   pEVSL_DeviceMatvec: y = A x on HBM vectors.
filter   pEVSL_ChebAvNoAlloc: one application of a Chebyshev filter p(A) to an
         HBM vector, FP64 or FP32 filter.  A solve spends its time here.
kpm      pEVSL_Kpmdos: moments of the density of states and the eigenvalue
         count (the first stage of every run).
cheblan  pEVSL_ChebLanNr / pEVSL_ChebLanNrBatch: whole filtered-Lanczos solves
         of spectrum slices, one after the other or as columns of one batch.
bounds   pEVSL_LanTrbounds: spectrum bounds by thick-restart Lanczos.
gen      pEVSL_ChebAv of a generalized problem with the library's polynomial
         B-solve.
mlp      pEVSL_MlpLossGrad: forward and backward pass of the slicer network.

Matrices: `lap` 7-point Laplacians (nz = 1: 5-point), `pot` Laplacians with a
random diagonal potential (the slicer's training family), `plaw` symmetric
matrices with power-law row lengths (the irregular workload).
"""
import ctypes as C
import functools
import math
import sys

import numpy as np
import torch

from pevsl_amd import capi, driver, slicer


def listed():
    return [
        # one product on the 20^3 grid of the README run: the smallest call
        dict(name="matvec_c1", kind="matvec", mat="lap", nx=20, ny=20, nz=20),
        # the README run's filter (degrees 61-110 on 20^3)
        dict(name="filter_c1", kind="filter", mat="lap", nx=20, ny=20, nz=20, prec=64,
             a=0.87, b=0.99, deg=86),
        # a slice's filter of the 100^3 Laplacian, interval [0.6, 1.2] in 10 slices
        dict(name="filter_c2", kind="filter", mat="lap", nx=100, ny=100, nz=100, prec=64,
             a=0.87, b=0.93, deg=168),
        # FP32 filter on odd sides with a diagonal potential (slicer training family)
        dict(name="filter_pot", kind="filter", mat="pot", nx=113, ny=97, nz=83, prec=32, w=1.3,
             a=0.9, b=1.1, deg=97),
        # filter on uneven rows (the irregular workload's generator)
        dict(name="filter_plaw", kind="filter", mat="plaw", n=100000, prec=64, a=-20.0, b=20.0,
             deg=120),
        # density of states of the README run, rand() vectors
        dict(name="kpm_c1", kind="kpm", mat="lap", nx=20, ny=20, nz=20, prec=64, rand="libc",
             Mdeg=300, nvec=60, a=0.6, b=1.2),
        # density of states of the 100^3 run: 64 vectors drawn on the device
        dict(name="kpm_c2", kind="kpm", mat="lap", nx=100, ny=100, nz=100, prec=32,
             rand="rademacher", Mdeg=300, nvec=64, a=0.6, b=1.2),
        # the README run's solve: five slices, one call each, FP64
        dict(name="cheblan_c1", kind="cheblan", nx=20, ny=20, nz=20, prec=64, a=0.6, b=1.2,
             nslices=5, first=0, count=5, batch=False),
        # eight of twenty slices as one batch, FP32 filter, FP64 basis (the
        # headline solve's wave on a smaller grid with unequal sides)
        dict(name="cheblan_batch", kind="cheblan", nx=48, ny=40, nz=44, prec=32, a=0.6, b=1.2,
             nslices=20, first=0, count=8, batch=True),
        # bounds of an irregular matrix (every run on a matrix read from a file
        # starts with them)
        dict(name="bounds_plaw", kind="bounds", mat="plaw", n=100000),
        # filter of A x = lambda B x with the polynomial B-solve
        dict(name="gen_filter", kind="gen", nx=40, ny=40, nz=40, a=1.5, b=2.5, deg=40),
        # one training batch of the slicer network, default shape
        dict(name="mlp_grad", kind="mlp", batch=256, nhidden=256, nlayers=3),
    ]


def _loguni(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, nmin, nmax):
    """Sides of a grid of about nmin..nmax points, unequal, sometimes 2-D."""
    n = _loguni(rng, nmin, nmax)
    if rng.random() < 0.15:
        s = math.sqrt(n)
        nx = max(2, int(s * rng.uniform(0.6, 1.6)))
        return dict(nx=nx, ny=max(2, n // nx), nz=1)
    s = n ** (1.0 / 3.0)
    nx = max(2, int(s * rng.uniform(0.7, 1.4)))
    ny = max(2, int(s * rng.uniform(0.7, 1.4)))
    return dict(nx=nx, ny=ny, nz=max(2, n // (nx * ny)))


def _matrix_draw(rng, nmin, nmax):
    u = rng.random()
    if u < 0.5:
        return dict(mat="lap", **_grid(rng, nmin, nmax))
    if u < 0.75:
        return dict(mat="pot", w=round(rng.uniform(0.1, 2.0), 3), **_grid(rng, nmin, nmax))
    return dict(mat="plaw", n=_loguni(rng, max(nmin, 2000), min(nmax, 150000)))


def _window(rng, lo, hi):
    """An interval of 1-20% of [lo, hi] inside it."""
    wd = (hi - lo) * math.exp(rng.uniform(math.log(0.01), math.log(0.2)))
    a = rng.uniform(lo + 0.02 * (hi - lo), hi - wd - 0.02 * (hi - lo))
    return round(a, 6), round(a + wd, 6)


def draw(rng):
    kind = rng.choice(["matvec", "filter", "filter", "filter", "kpm", "kpm", "cheblan",
                       "cheblan", "bounds", "gen", "mlp"])
    if kind == "matvec":
        return dict(kind=kind, **_matrix_draw(rng, 500, 1000000))
    if kind == "filter":
        m = _matrix_draw(rng, 500, 1000000)
        lo, hi = (-60.0, 60.0) if m["mat"] == "plaw" else (0.0, 8.0 if m["nz"] == 1 else 12.0)
        a, b = _window(rng, lo, hi)
        return dict(kind=kind, prec=rng.choice([32, 64]), a=a, b=b, deg=_loguni(rng, 8, 400), **m)
    if kind == "kpm":
        m = _matrix_draw(rng, 500, 600000)
        lo, hi = (-60.0, 60.0) if m["mat"] == "plaw" else (0.0, 8.0 if m["nz"] == 1 else 12.0)
        a, b = _window(rng, lo, hi)
        n = m["n"] if m["mat"] == "plaw" else m["nx"] * m["ny"] * m["nz"]
        return dict(kind=kind, prec=rng.choice([32, 64]), a=a, b=b, Mdeg=_loguni(rng, 20, 300),
                    nvec=rng.randint(1, 64),
                    rand="libc" if n < 20000 and rng.random() < 0.6
                    else rng.choice(["rademacher", "uniform"]), **m)
    if kind == "cheblan":
        batch = rng.random() < 0.6
        s = [rng.randint(12, 44 if batch else 24) for _ in range(3)]
        n = s[0] * s[1] * s[2]
        return dict(kind=kind, nx=s[0], ny=s[1], nz=s[2],
                    prec=rng.choice([32, 32, 64]) if batch else 64,
                    a=0.6, b=1.2, nslices=max(3, int(round(n * 0.016 / 60.0))), first=0,
                    count=rng.randint(2, 8) if batch else rng.randint(1, 3), batch=batch)
    if kind == "bounds":
        return dict(kind=kind, **_matrix_draw(rng, 2000, 150000))
    if kind == "gen":
        g = _grid(rng, 500, 200000)
        g["nx"] += g["nx"] % 2  # an even order
        a, b = _window(rng, 0.0, 4.0)
        return dict(kind=kind, a=a, b=b, deg=_loguni(rng, 8, 60), **g)
    return dict(kind="mlp", batch=_loguni(rng, 1, 1024), nhidden=rng.choice([64, 128, 200, 256]),
                nlayers=rng.randint(1, 4))


# ------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=2)
def _lap(nx, ny, nz):
    return driver.laplacian3d(nx, ny, nz)


def _csr(case, seed):
    """(ia, ja, a, frame) of the case's matrix."""
    mat = case.get("mat", "lap")
    if mat == "plaw":
        ia, ja, a = driver.powerlaw_sym(case["n"], seed=seed % 100003)
        # Gershgorin frame
        r = float(np.add.reduceat(np.abs(a), ia[:-1]).max()) if len(a) else 1.0
        return ia, ja, a, (-r, r)
    ia, ja, a = _lap(case["nx"], case["ny"], case["nz"])
    top = 12.0 if case["nz"] > 1 else 8.0
    if mat == "pot":
        n = len(ia) - 1
        rows = np.repeat(np.arange(n, dtype=np.int32), np.diff(ia))
        a = a.copy()
        a[ja == rows] += case["w"] * np.random.default_rng(seed).random(n)
        top += case["w"]
    return ia, ja, a, (0.0, top)


def _vec(n, seed):
    return np.random.default_rng(seed + 17).uniform(-1.0, 1.0, n)


def _step_coeffs(deg, a, b, lmin, lmax):
    """Chebyshev coefficients of a sigma-damped step function on [a, b]."""
    cc, dd = 0.5 * (lmax + lmin), 0.5 * (lmax - lmin)
    th0, th1 = math.acos(max(-1.0, min(1.0, (b - cc) / dd))), \
        math.acos(max(-1.0, min(1.0, (a - cc) / dd)))
    k = np.arange(1, deg + 1)
    damp = np.sin(k * math.pi / (deg + 1)) / (k * math.pi / (deg + 1))
    mu = np.empty(deg + 1)
    mu[0] = (th1 - th0) / math.pi
    mu[1:] = 2.0 / math.pi * (np.sin(k * th1) - np.sin(k * th0)) / k * damp
    return mu, cc, dd


class _Held:
    """Library objects of one state, released with it."""

    def __init__(self):
        self._undo = []

    def add(self, obj, undo):
        self._undo.append(undo)
        return obj

    def __del__(self):
        if sys.is_finalizing():
            return
        while self._undo:
            self._undo.pop()()


def _pol(mu, cc, dd):
    pol = capi.Polparams()
    pol.deg = len(mu) - 1
    pol.max_deg = pol.deg
    pol.cc, pol.dd = cc, dd
    pol.mu = mu.ctypes.data_as(capi.c_double_p)
    return pol


def _cuts(nx, ny, nz, a, b, nslices):
    """Equal-count cuts of [a, b], each in the widest gap near its share."""
    # the closed-form spectrum
    s2 = [4.0 * np.sin(np.arange(1, m + 1) * 0.5 * np.pi / (m + 1)) ** 2 for m in (nx, ny, nz)]
    ev = np.sort((s2[0][:, None, None] + s2[1][None, :, None] + s2[2][None, None, :]).ravel())
    ev = ev[(ev >= a) & (ev <= b)]
    cuts, m = [a], len(ev)
    for s in range(1, nslices):
        i = s * m // nslices
        w = max(2, m // (4 * nslices))
        j0, j1 = max(1, i - w), min(m - 1, i + w)
        j = j0 + int(np.argmax(ev[j0:j1 + 1] - ev[j0 - 1:j1]))
        cuts.append(0.5 * (ev[j - 1] + ev[j]))
    return cuts + [b], ev


def prepare(case, seed):
    kind = case["kind"]
    lib = capi.load()
    held = _Held()
    st = dict(case=case, lib=lib, seed=seed, held=held)
    if kind == "mlp":
        net = slicer.Mlp(lib, nhidden=case["nhidden"], nlayers=case["nlayers"], seed=seed)
        held.add(net, net.free)
        net.set_weights(_mlp_weights(case, seed))
        st.update(net=net, **_mlp_batch(case, seed))
        return st
    ia, ja, a, frame = _csr(case, seed)
    M = driver.Matrix(lib, ia, ja, a)
    held.add(M, M.free)
    prec = capi.PEVSL_PREC_FP32 if case.get("prec", 64) == 32 else capi.PEVSL_PREC_FP64
    inst = driver.Instance(lib, M, prec=prec)
    held.add(inst, inst.close)
    n = M.n
    st.update(M=M, inst=inst, frame=frame)
    if kind in ("matvec", "filter"):
        st["x"] = torch.from_numpy(_vec(n, seed)).cuda()
        st["y"] = torch.empty_like(st["x"])
    if kind == "filter":
        mu, cc, dd = _step_coeffs(case["deg"], case["a"], case["b"], *frame)
        st.update(mu=mu, pol=_pol(mu, cc, dd))
    elif kind in ("bounds", "cheblan"):
        st["vinit"] = _vec(n, seed)
    elif kind == "gen":
        MB = driver.Matrix(lib, *driver.chain_laplacian(n))
        held.add(MB, MB.free)
        lib.pEVSL_SetBParcsr(inst.p, C.byref(MB.A))
        bsol = C.c_void_p()
        lib.pEVSL_SetupLSPolRec(50, 1e-12, 2.0, 6.0, C.byref(MB.A), C.byref(bsol))
        held.add(bsol, lambda: lib.pEVSL_LSPolFree(bsol))
        lib.pEVSL_SetBSol(inst.p, C.cast(lib.pEVSL_LSPolSol, C.c_void_p), bsol)
        lib.pEVSL_SetGenEig(inst.p)
        mu, cc, dd = _step_coeffs(case["deg"], case["a"], case["b"], 0.0, 0.5 * frame[1])
        x, y = _vec(n, seed), np.empty(n)
        pv = [capi.Parvec(), capi.Parvec(), capi.Parvec()]
        for p, v in zip(pv, (x, y, y)):
            lib.pEVSL_ParvecCreateShell(n, n, 0, 0, C.byref(p), v.ctypes.data_as(capi.c_double_p))
        st.update(MB=MB, mu=mu, pol=_pol(mu, cc, dd), x=x, y=y, pv=pv)
    if kind == "cheblan":
        cuts, ev = _cuts(case["nx"], case["ny"], case["nz"], case["a"], case["b"],
                         case["nslices"])
        top = frame[1]
        sel = range(case["first"], min(case["first"] + case["count"], case["nslices"]))
        intvs = [[cuts[s], cuts[s + 1], 0.0, top] for s in sel]
        pols = []
        for iv in intvs:
            pol, rc = driver.find_pol(lib, iv)
            if rc:
                raise RuntimeError("FindPol error %d" % rc)
            held.add(pol, functools.partial(lib.pEVSL_FreePol, C.byref(pol)))
            pols.append(pol)
        nev = int(1 + len(ev) / case["nslices"]) + 2
        st.update(intvs=intvs, pols=pols, mlan=min(max(5 * nev, 300), n))
    torch.cuda.synchronize()
    return st


def _mlp_dims(case):
    return [slicer.NIN] + [case["nhidden"]] * case["nlayers"] + [slicer.NOUT]


def _mlp_weights(case, seed):
    """Packed parameters W_l (out x in), b_l: He-normal weights, small biases."""
    rng = np.random.default_rng(seed + 2)
    dims = _mlp_dims(case)
    parts = []
    for i, o in zip(dims, dims[1:]):
        parts += [rng.normal(0.0, math.sqrt(2.0 / i), i * o), rng.normal(0.0, 0.02, o)]
    return np.concatenate(parts).astype(np.float32)


def _mlp_batch(case, seed):
    """Features, priors and targets of a training batch: standardized inputs,
    log-mass priors, target masses that sum to one and a log fraction."""
    rng = np.random.default_rng(seed + 1)
    b = case["batch"]
    X = rng.normal(0.0, 1.0, (b, slicer.NIN)).astype(np.float32)
    m = rng.gamma(2.0, 1.0, (b, slicer.NOUT - 1))
    m /= m.sum(1, keepdims=True)
    frac = rng.uniform(-4.0, -0.5, (b, 1))
    Q = np.concatenate([np.log(m * rng.uniform(0.7, 1.4, m.shape)), frac + 0.1], 1)
    T = np.concatenate([m, frac], 1)
    return dict(X=X, Q=Q.astype(np.float32), T=T.astype(np.float32))


# --------------------------------------------------------------------- run
_RAND = {"libc": capi.PEVSL_RAND_LIBC, "rademacher": capi.PEVSL_RAND_RADEMACHER,
         "uniform": capi.PEVSL_RAND_UNIFORM}


def _check(rc, what):
    if rc:
        raise RuntimeError("%s error %d" % (what, rc))


def run(st):
    case, lib, kind = st["case"], st["lib"], st["case"]["kind"]
    if kind == "mlp":
        loss, grad = st["net"].loss_grad(st["X"], st["Q"], st["T"])
        return [np.array([loss], np.float32), grad]
    inst = st["inst"]
    if kind == "matvec":
        _check(lib.pEVSL_DeviceMatvec(inst.p, C.c_void_p(st["x"].data_ptr()),
                                      C.c_void_p(st["y"].data_ptr())), "DeviceMatvec")
        return st["y"]
    if kind == "filter":
        _check(lib.pEVSL_ChebAvNoAlloc(inst.p, C.byref(st["pol"]), C.c_void_p(st["x"].data_ptr()),
                                       C.c_void_p(st["y"].data_ptr())), "ChebAvNoAlloc")
        return st["y"]
    if kind == "gen":
        pv = st["pv"]
        _check(lib.pEVSL_ChebAv(inst.p, C.byref(st["pol"]), C.byref(pv[0]), C.byref(pv[1]),
                                C.byref(pv[2])), "ChebAv")
        return st["y"]
    if kind == "kpm":
        # the stream of random vectors starts anew, as in a fresh run
        lib.pEVSL_RandSeed(st["seed"] & 0x7FFFFFFF)
        lib.pEVSL_SetRandMode(inst.p, _RAND[case["rand"]], st["seed"])
        rc, mu, ecnt = inst.kpmdos(case["Mdeg"], 1, case["nvec"],
                                   [case["a"], case["b"], *st["frame"]])
        _check(rc, "Kpmdos")
        return [mu, float(ecnt)]
    if kind == "bounds":
        rc, lmin, lmax = inst.lan_trbounds(50, 200, 1e-8, st["vinit"], 1)
        _check(rc, "LanTrbounds")
        return [float(lmin), float(lmax)]
    out = []
    groups = [range(len(st["pols"]))] if case["batch"] else [[s] for s in range(len(st["pols"]))]
    for g in groups:
        rc, res = driver.cheblan_batch(inst, [st["intvs"][s] for s in g], [st["mlan"]] * len(g),
                                       1e-8, st["vinit"], [st["pols"][s] for s in g])
        _check(rc, "ChebLanNr")
        out += [np.sort(r["lam"]) for r in res]
    return out


# -------------------------------------------------------------------- work
def _size(case):
    if case.get("mat") == "plaw":
        return case["n"], 33 * case["n"]
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    nnz = n * (7 if nz > 1 else 5) - 2 * (ny * nz + nx * nz + (nx * ny if nz > 1 else 0))
    return n, nnz


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        dims = _mlp_dims(case)
        nw = sum(i * o + o for i, o in zip(dims, dims[1:]))
        return dict(bytes=8 * nw + 4 * case["batch"] * (slicer.NIN + 2 * slicer.NOUT),
                    flops=6 * nw * case["batch"])
    n, nnz = _size(case)
    mat = 12 * nnz + 4 * (n + 1)
    if kind == "matvec":
        return dict(bytes=mat + 16 * n, flops=2 * nnz)
    if kind == "filter":
        return dict(bytes=mat + 16 * n, flops=case["deg"] * (2 * nnz + 6 * n))
    if kind == "gen":
        # A and the chain B once, about 22 degrees of the B-solve a product
        return dict(bytes=mat + 40 * n + 16 * n, flops=case["deg"] * (2 * nnz + 22 * 12 * n))
    if kind == "kpm":
        return dict(bytes=mat, flops=case["Mdeg"] * case["nvec"] * (2 * nnz + 6 * n))
    if kind == "bounds":
        return dict(bytes=mat + 8 * n, flops=100 * (2 * nnz + 4 * 50 * n))
    # steps about 3.6 per eigenvalue, degree about 8.5 / slice width
    nev = 0.016 * n / case["nslices"]
    its, deg = 3.6 * nev + 60, 8.5 * case["nslices"] / (case["b"] - case["a"])
    return dict(bytes=mat + 8 * n,
                flops=int(case["count"] * (its * deg * (2 * nnz + 6 * n) + 2 * its * its * n)))


# ------------------------------------------------------------------- exact
def _sparse(ia, ja, a, dev):
    n = len(ia) - 1
    return torch.sparse_csr_tensor(torch.from_numpy(ia.astype(np.int64)),
                                   torch.from_numpy(ja.astype(np.int64)),
                                   torch.from_numpy(a), (n, n), dtype=torch.float64).to(dev)


def _mix64(x):
    """The splitmix64 finalizer (Steele, Lea, Flood 2014) on uint64 arrays."""
    x = x + np.uint64(0x9E3779B97F4A7C15)
    x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return x ^ (x >> np.uint64(31))


def _kpm_vectors(case, seed, n):
    """The run's random vectors as the entry point documents them."""
    m = case["nvec"]
    if case["rand"] == "libc":
        libc = C.CDLL(None)
        libc.srand(C.c_uint(seed & 0x7FFFFFFF))
        t = 2147483647.0 / 2.0
        return (np.array([libc.rand() for _ in range(n * m)], dtype=np.float64).reshape(m, n) - t) / t
    with np.errstate(over="ignore"):
        r = _mix64(np.uint64(seed) ^ _mix64(np.arange(n * m, dtype=np.uint64)))
    if case["rand"] == "rademacher":
        v = np.where((r >> np.uint64(63)).astype(bool), 1.0, -1.0)
    else:
        v = (r >> np.uint64(11)).astype(np.float64) * (2.0 / 9007199254740992.0) - 1.0
    return v.reshape(m, n)


def _chain_inverse(b):
    """tridiag(-1, 4, -1)^{-1} b: the infinite Toeplitz inverse
    r^|i-j| / (2 sqrt 3), r = 2 - sqrt 3, on the odd extension of b."""
    r, n = 2.0 - math.sqrt(3.0), len(b)
    pad = min(n, 64)
    z = torch.zeros(1, dtype=torch.float64)
    e = torch.cat([-b[:pad].flip(0), z, b, z, -b[-pad:].flip(0)])

    def scan(v):
        s = 1
        f = r
        while s < len(v) and f > 1e-40:
            v = v.clone()
            v[s:] += f * v[:-s].clone()
            s, f = 2 * s, f * f
        return v
    g = (scan(e) + scan(e.flip(0)).flip(0) - e) / (2.0 * math.sqrt(3.0))
    return g[pad + 1:pad + 1 + n]


def _cheb_apply(mul, mu, cc, dd, v):
    y, vk, vm = mu[0] * v, v, None
    for k in range(1, len(mu)):
        w = (mul(vk) - cc * vk) * ((1.0 if k == 1 else 2.0) / dd)
        if vm is not None:
            w = w - vm
        vm, vk = vk, w
        y = y + mu[k] * w
    return y


def exact(case, seed):
    kind = case["kind"]
    if kind == "bounds":
        return None
    if kind == "mlp":
        return _mlp_exact(case, seed)
    if kind == "cheblan":
        cuts, ev = _cuts(case["nx"], case["ny"], case["nz"], case["a"], case["b"],
                         case["nslices"])
        out = []
        for s in range(case["first"], min(case["first"] + case["count"], case["nslices"])):
            out.append(ev[(ev >= cuts[s]) & (ev <= cuts[s + 1])])
        return out
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    ia, ja, a, frame = _csr(case, seed)
    n = len(ia) - 1
    if kind == "gen":
        A = _sparse(ia, ja, a, "cpu")
        mu, cc, dd = _step_coeffs(case["deg"], case["a"], case["b"], 0.0, 0.5 * frame[1])
        return _cheb_apply(lambda v: A @ _chain_inverse(v), mu, cc, dd,
                           torch.from_numpy(_vec(n, seed))).numpy()
    A = _sparse(ia, ja, a, dev)
    if kind in ("matvec", "filter"):
        v = torch.from_numpy(_vec(n, seed)).to(dev)
        if kind == "matvec":
            return A @ v
        mu, cc, dd = _step_coeffs(case["deg"], case["a"], case["b"], *frame)
        return _cheb_apply(lambda x: A @ x, mu, cc, dd, v)
    # kpm: mu_k = jac_k (2 - [k = 0]) / (nvec pi) sum_m <v_m, T_k(A) v_m>
    if n * case["nvec"] * case["Mdeg"] > 3e10:
        return None
    Mdeg, nvec = case["Mdeg"], case["nvec"]
    ctr, wid = 0.5 * (frame[1] + frame[0]), 0.5 * (frame[1] - frame[0])
    k = np.arange(Mdeg + 1)
    th = math.pi / (Mdeg + 2)
    jac = np.sin((k + 1) * th) / ((Mdeg + 2) * math.sin(th)) + \
        (1 - (k + 1) / (Mdeg + 2)) * np.cos(k * th)
    jac[0] = 1.0
    v0 = torch.from_numpy(np.ascontiguousarray(_kpm_vectors(case, seed, n).T)).to(dev)
    v0 = v0 / v0.norm(dim=0, keepdim=True)
    dots = np.zeros(Mdeg + 1)
    dots[0] = nvec
    vk, vm = v0, None
    for j in range(1, Mdeg + 1):
        w = (A @ vk - ctr * vk) * ((1.0 if j == 1 else 2.0) / wid)
        if vm is not None:
            w -= vm
        vm, vk = vk, w
        dots[j] = float((w * v0).sum())
    mu = dots * jac * np.where(k == 0, 1.0, 2.0) / (nvec * math.pi)
    eps = np.finfo(float).eps
    b1 = math.acos(max(-1.0 + eps, (max(case["a"], frame[0]) - ctr) / wid))
    b2 = math.acos(min(1.0 - eps, (min(case["b"], frame[1]) - ctr) / wid))
    kk = k[1:]
    ecnt = -n * (mu[0] * (b2 - b1) + float((mu[1:] * (np.sin(kk * b2) - np.sin(kk * b1)) / kk).sum()))
    return [mu, ecnt]


def _mlp_exact(case, seed):
    w, bt = _mlp_weights(case, seed), _mlp_batch(case, seed)
    X, Q, T = (torch.from_numpy(bt[k].astype(np.float64)) for k in ("X", "Q", "T"))
    p = torch.from_numpy(w.astype(np.float64)).requires_grad_(True)
    dims = _mlp_dims(case)
    h, off = X, 0
    for l, (i, o) in enumerate(zip(dims, dims[1:])):
        W = p[off:off + i * o].reshape(o, i)
        h = h @ W.T + p[off + i * o:off + i * o + o]
        off += i * o + o
        if l < len(dims) - 2:
            h = torch.nn.functional.gelu(h)
    y, ns = h + Q, slicer.NOUT - 1
    loss = (-(T[:, :ns] * torch.log_softmax(y[:, :ns], 1)).sum(1)
            + ((y[:, ns:] - T[:, ns:]) ** 2).sum(1)).mean()
    loss.backward()
    return [loss.detach().numpy().reshape(1), p.grad.numpy()]
