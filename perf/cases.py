"""What a user of this framework has it do, as cases to time and compare.

Every case goes through the public entry points, with the sizes of the
reference drivers and of bench.py.  A case is a dict of plain values; its
"kind" names the call:

  dos     kpmdos_ex on the current matrix: the density of states that slicing
          starts from (seeded Rademacher vectors)
  pool    kpmdos_batch: densities of a pool of matrices of uneven size
  filter  evsl_amd_cheb_av_cols on device-resident vectors: p(A) X, the inner
          step of every filtered solver (one column: the plain ChebLanNr; 2-8
          columns of different degrees: slices of one matrix; 16 and more:
          blocks of many slices and of subspace iteration)
  solve   the call sequence of the LapPLanN driver: SetAMatrix, kpmdos,
          spslicer, then find_pol and ChebLanNr for each slice (FP64)
  batch   the same slices as one ChebLanNr_batch in the mixed-precision form
  landos  the LanDos driver's calls: LanTrbounds and LanDos
  serve   the request loop over resident matrices: slices and densities

A matrix is fixed by its case, as a user's operator is; start vectors, blocks
and the seeds of random vectors come from the seed.  Solved boxes have pairwise
different side lengths, so their eigenvalues are simple and known in closed form.
"""
import ctypes
import functools
import math

import numpy as np
import torch

from evsl_amd import matrices as M
from evsl_amd.evsl import EVSL, PREC_FP64, PREC_MIXED, VEC_RADEMACHER, Server
from evsl_amd.types import PolParams, c_double_p

_LIBC = ctypes.CDLL(None)
_SLICING = 7  # seed of the vectors that a solve's slices come from: the slices stay


@functools.lru_cache(maxsize=1)
def _library():
    ev = EVSL()
    assert ev.start() == 0, ev.last_error()
    return ev


# ---- cases ---------------------------------------------------------------------

def listed():
    return [
        # the plain driver's density of states: a small 2-D grid, 60 vectors
        # (launches and latency, not bandwidth)
        dict(name="dos_lap2d_1e4", kind="dos", family="box", nx=100, ny=100, nz=1, mdeg=300,
             nvec=60),
        # the headline problem's density of states: 10^6 rows, 40 vectors
        dict(name="dos_lap3d_1e6", kind="dos", family="perturbed", nx=100, ny=100, nz=100,
             mdeg=300, nvec=40),
        # the batching form's first phase: 32 requests over 8 small matrices
        dict(name="dos_pool", kind="pool", mats=8, requests=32, log2lo=10.0, log2hi=14.0,
             mdeg=200, nvec=32, prec="mixed", pool=4242),
        # the smallest filter call: one vector, a small grid, a low degree
        dict(name="filter_small", kind="filter", family="box", nx=64, ny=64, nz=1, cols=1,
             deg_lo=30, deg_hi=30, prec="fp64"),
        # one Lanczos step's filter of the plain FP64 form on the headline problem
        dict(name="filter_lap3d_1e6_plain", kind="filter", family="perturbed", nx=100, ny=100,
             nz=100, cols=1, deg_lo=442, deg_hi=442, prec="fp64"),
        # the same step for the headline's 8 slices in the mixed form
        dict(name="filter_lap3d_1e6_mixed8", kind="filter", family="perturbed", nx=100, ny=100,
             nz=100, cols=8, deg_lo=357, deg_hi=519, prec="mixed"),
        # two slices of an irregular matrix (8-32 nonzeros a row, any column)
        dict(name="filter_random_1e5", kind="filter", family="random", n=131072, lo=8, hi=32,
             cols=2, deg_lo=300, deg_hi=300, prec="fp64"),
        # 16 narrow slices at the band centre of an Anderson lattice (high degree)
        dict(name="filter_anderson_16", kind="filter", family="anderson", L=80, cols=16,
             deg_lo=3000, deg_hi=3000, prec="mixed"),
        # a whole small driver run, FP64, two slices
        dict(name="solve_lap2d", kind="solve", nx=100, ny=97, nz=1, a=0.4, b=0.6, nslices=2,
             mdeg=300, nvec=60),
        # a whole mixed-precision batched solve, four slices of a 3-D box
        dict(name="batch_lap3d", kind="batch", nx=30, ny=32, nz=34, a=0.4, b=0.6, nslices=4,
             mdeg=300, nvec=40),
        # bounds and Lanczos density of a 20^3 grid
        dict(name="landos_20", kind="landos", nx=20, ny=20, nz=20, nvec=20, msteps=40, npts=200),
        # six slices and three densities over three resident matrices
        dict(name="serve", kind="serve", scale=10000, count=20, per=2, mdeg=200, nvec=32,
             prec="fp64"),
    ]


def _loguniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _sides(rng, n, dims):
    """Side lengths, pairwise different, of a box of about n points."""
    s = max(4, round(n ** (1.0 / dims)))
    d = rng.randint(1, max(1, s // 8))
    return (s, s + d, 1) if dims == 2 else (s, s + d, s + 2 * d)


def draw(rng):
    kind = rng.choice(["dos", "pool", "filter", "filter", "filter", "solve", "batch", "landos",
                       "serve"])
    if kind == "dos":
        nx, ny, nz = _sides(rng, _loguniform(rng, 2e3, 5e5), rng.choice([2, 3]))
        return dict(kind=kind, family=rng.choice(["box", "perturbed"]), nx=nx, ny=ny, nz=nz,
                    mdeg=rng.randint(60, 300), nvec=rng.randint(1, 60))
    if kind == "pool":
        lo = rng.uniform(9.0, 12.0)
        return dict(kind=kind, mats=rng.randint(2, 8), requests=rng.randint(2, 32), log2lo=lo,
                    log2hi=lo + 3.0, mdeg=rng.randint(60, 200), nvec=rng.randint(1, 40),
                    prec=rng.choice(["fp64", "mixed"]), pool=rng.randrange(1 << 20))
    if kind == "filter":
        cols = rng.choice([1, 1, 2, 3, 4, 5, 7, 8, 8, 11, 16, 24, 32])
        lo = rng.randint(20, 500)
        case = dict(kind=kind, cols=cols, deg_lo=lo, deg_hi=lo + rng.choice([0, 0, lo // 3]),
                    prec=rng.choice(["fp64", "mixed"]))
        fam = rng.choice(["box", "perturbed", "anderson", "random"])
        n = _loguniform(rng, 2e3, 1e6)
        if fam == "random":
            lo = rng.randint(3, 12)
            return dict(case, family=fam, n=int(min(n, 2e5)), lo=lo, hi=lo + rng.randint(1, 24))
        if fam == "anderson":
            return dict(case, family=fam, L=max(8, round(min(n, 5e5) ** (1 / 3))))
        nx, ny, nz = _sides(rng, n, rng.choice([2, 3]))
        return dict(case, family=fam, nx=nx, ny=ny, nz=nz)
    if kind in ("solve", "batch"):
        dims = 2 if kind == "solve" else 3
        n = _loguniform(rng, 2.5e3, 1e4) if dims == 2 else _loguniform(rng, 5e3, 3e4)
        nx, ny, nz = _sides(rng, n, dims)
        n, a, count = nx * ny * nz, rng.uniform(0.3, 1.0), rng.randint(30, 100)
        # eigenvalues below x: n x / (4 pi) in 2-D, n x^1.5 / (6 pi^2) in 3-D
        if dims == 2:
            b = a + 4.0 * math.pi * count / n
        else:
            b = (a ** 1.5 + 6.0 * math.pi ** 2 * count / n) ** (2.0 / 3.0)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, a=a, b=b,
                    nslices=rng.randint(1, 3) if kind == "solve" else rng.randint(2, 6),
                    mdeg=300, nvec=rng.randint(20, 60))
    if kind == "landos":
        nx, ny, nz = _sides(rng, _loguniform(rng, 1e3, 3e4), 3)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, nvec=rng.randint(2, 16),
                    msteps=rng.randint(30, 50), npts=rng.choice([100, 200, 333]))
    return dict(kind=kind, scale=int(_loguniform(rng, 2e3, 1e4)), count=rng.randint(10, 20),
                per=rng.randint(1, 2), mdeg=rng.randint(100, 200), nvec=rng.randint(8, 32),
                prec=rng.choice(["fp64", "mixed"]))


# ---- matrices, vectors and filters ------------------------------------------------

@functools.lru_cache(maxsize=4)
def _box(nx, ny, nz):
    return M.laplacian(nx, ny, nz)


@functools.lru_cache(maxsize=4)
def _made(family, *size):
    """(matrix, lower bound, upper bound of its spectrum)"""
    if family == "box":
        return _box(*size), 0.0, 8.0 if size[2] == 1 else 12.0
    if family == "perturbed":
        return M.perturb_diag(_box(*size), 1e-3, seed=1), 0.0, 8.001 if size[2] == 1 else 12.001
    A = M.anderson(size[0], 16.5, seed=2) if family == "anderson" else M.random_symmetric(
        *size, seed=3)
    return (A,) + M.gershgorin(A)


def _matrix(case):
    if case["family"] == "anderson":
        return _made("anderson", case["L"])
    if case["family"] == "random":
        return _made("random", case["n"], case["lo"], case["hi"])
    return _made(case["family"], case["nx"], case["ny"], case["nz"])


@functools.lru_cache(maxsize=4)
def _pool(mats, log2lo, log2hi, pool):
    """A pool as the batching form's: 2-D and 3-D grids and random matrices in
    turn, sizes log-uniform."""
    rng = np.random.default_rng(pool)
    out = []
    for i in range(mats):
        n = int(2 ** rng.uniform(log2lo, log2hi))
        if i % 3 == 0:
            s = max(2, round(n ** 0.5))
            A = M.laplacian(s, s, 1)
        elif i % 3 == 1:
            s = max(2, round(n ** (1 / 3)))
            A = M.laplacian(s, s, s)
        else:
            A = M.random_symmetric(n, 8, 32, seed=pool + i)
        out.append((A,) + M.gershgorin(A))
    return out


def _requests(case, seed):
    """(matrix, lmin, lmax, interval, seed of the vectors) of each density"""
    pool = _pool(case["mats"], case["log2lo"], case["log2hi"], case["pool"])
    rng = np.random.default_rng(seed)
    out = []
    for r in range(case["requests"]):
        A, lo, hi = pool[r % len(pool)]
        a = lo + (hi - lo) * rng.uniform(0.05, 0.85)
        out.append((A, lo, hi, np.array([a, a + 0.1 * (hi - lo), lo, hi]),
                    int(rng.integers(1 << 40))))
    return out


@functools.lru_cache(maxsize=4)
def _serve_pool(scale):
    s2, s3 = round(scale ** 0.5), round(scale ** (1 / 3))
    return [(M.laplacian(s2, s2 - 3, 1), 0.0, 8.0),
            (M.laplacian(s3, s3 + 1, s3 + 2), 0.0, 12.0),
            (lambda A: (A,) + M.gershgorin(A))(M.anderson(s3, 16.5, seed=2))]


def _serve_requests(case, seed):
    """("slice", matrix, a, b, start vector) and ("dos", matrix, a, b, seed)"""
    rng = np.random.default_rng(seed)
    out = []
    for m, (A, _, _) in enumerate(_serve_pool(case["scale"])):
        for i in range(case["per"]):
            if m == 0:  # about `count` eigenvalues in each slice
                a = 0.4 + 0.3 * i
                b = a + 4.0 * math.pi * case["count"] / A.n
            elif m == 1:
                a = 0.6 + 0.4 * i
                b = (a ** 1.5 + 6.0 * math.pi ** 2 * case["count"] / A.n) ** (2.0 / 3.0)
            else:
                a = -0.4 + 0.6 * i
                b = a + 18.0 * case["count"] / A.n
            out.append(("slice", m, a, b, rng.uniform(-1.0, 1.0, A.n)))
        out.append(("dos", m, 0.5, 1.5, int(rng.integers(1 << 40))))
    return out


def _coefficients(deg, centre, cc, dd):
    """Chebyshev coefficients of a Jackson-damped delta at `centre`, scaled to
    p(centre) = 1: a band-pass filter of the degree"""
    k = np.arange(deg + 1)
    th = math.acos((centre - cc) / dd)
    j = math.pi / (deg + 2)
    jac = ((deg + 2 - k) * np.cos(k * j) + np.sin(k * j) / math.tan(j)) / (deg + 2)
    mu = np.cos(k * th) * jac
    mu[0] *= 0.5
    return mu / np.dot(mu, np.cos(k * th))


def _filters(case, lo, hi):
    """(cc, dd, [coefficients of each column's filter]): degrees from deg_lo
    to deg_hi, centres in the lower half of the spectrum"""
    cc, dd = 0.5 * (lo + hi), 0.5 * (hi - lo)
    degs = np.linspace(case["deg_lo"], case["deg_hi"], case["cols"]).round().astype(int)
    mid = lo + (hi - lo) * np.linspace(0.15, 0.45, case["cols"])
    return cc, dd, [_coefficients(int(d), m, cc, dd) for d, m in zip(degs, mid)]


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _vectors(case, n, seed):
    """cols x n start vectors, U[-1, 1]"""
    g = torch.Generator(device=_device()).manual_seed(seed)
    return torch.rand(case["cols"], n, dtype=torch.float64, device=_device(),
                      generator=g) * 2.0 - 1.0


# ---- what a program has in hand, and one pass ----------------------------------------

def prepare(case, seed):
    ev, kind = _library(), case["kind"]
    st = dict(case=case, kind=kind, seed=seed)
    if kind in ("dos", "filter"):
        A, lo, hi = _matrix(case)
        assert ev.set_matrix(A) == 0, ev.last_error()
        st.update(n=A.n, intv=np.array([lo + 0.05 * (hi - lo), lo + 0.1 * (hi - lo), lo, hi]))
    if kind == "filter":
        cc, dd, mus = _filters(case, lo, hi)
        st["mus"] = mus  # the pols below point at these
        st["pols"] = (PolParams * case["cols"])()
        for p, mu in zip(st["pols"], mus):
            ev.lib.set_pol_def(ctypes.byref(p))
            p.mu, p.cc, p.dd, p.deg = mu.ctypes.data_as(c_double_p), cc, dd, len(mu) - 1
        st["X"] = _vectors(case, A.n, seed)
        st["Y"] = torch.empty_like(st["X"])
    elif kind == "pool":
        st["requests"] = _requests(case, seed)
    elif kind in ("solve", "batch"):
        st["A"] = _box(case["nx"], case["ny"], case["nz"])
        st["vinit"] = _vectors(dict(cols=1), st["A"].n, seed)
    elif kind == "landos":
        A = _box(case["nx"], case["ny"], case["nz"])
        assert ev.set_matrix(A) == 0, ev.last_error()
        st["vinit"] = np.random.default_rng(seed).uniform(-1.0, 1.0, A.n)
    elif kind == "serve":
        prec = PREC_MIXED if case["prec"] == "mixed" else PREC_FP64
        st["server"] = srv = Server(ev, 16 << 30, prec)
        st["n"] = []
        for A, lo, hi in _serve_pool(case["scale"]):
            assert srv.add_matrix(A, lo, hi) >= 0, ev.last_error()
            st["n"].append(A.n)
        st["requests"] = _serve_requests(case, seed)
    return st


def _sorted(lam, Y):
    order = np.argsort(lam, kind="stable")
    return {"lam": lam[order], "Y": Y[:, order]}


def _joined(pairs):
    """The eigenvalues of all slices in order, and each slice's vectors"""
    return {"lam": np.sort(np.concatenate([p["lam"] for p in pairs])),
            "Y": [p["Y"] for p in pairs]}


def _slices(ev, st):
    """SetAMatrix, the density, equal-count slices and their filters"""
    case, A = st["case"], st["A"]
    intv = np.array([case["a"], case["b"], 0.0, 8.0 if case["nz"] == 1 else 12.0])
    assert ev.set_matrix(A) == 0, ev.last_error()
    err, mu, ecnt = ev.kpmdos(case["mdeg"], 1, case["nvec"], intv, vec_kind=VEC_RADEMACHER,
                              seed=_SLICING)
    assert err == 0, ev.last_error()
    ns = case["nslices"]
    err, sli = ev.spslicer(mu, intv, ns, int(10 * ecnt))
    assert err == 0, err
    mlan = min(max(5 * (int(1 + ecnt / ns) + 2), 300), A.n)
    ivs, pols = [], []
    for s in range(ns):
        iv, pol = np.array([sli[s], sli[s + 1], intv[2], intv[3]]), ev.default_pol()
        pol.damping, pol.thresh_int, pol.thresh_ext, pol.max_deg = 2, 0.8, 0.2, 3000
        assert ev.find_pol(iv, pol) == 0
        ivs.append(iv)
        pols.append(pol)
    return mu, ivs, pols, mlan


def run(st):
    ev, kind, case = _library(), st["kind"], st["case"]
    if kind == "dos":
        err, mu, ecnt = ev.kpmdos(case["mdeg"], 1, case["nvec"], st["intv"],
                                  vec_kind=VEC_RADEMACHER, seed=st["seed"])
        assert err == 0, ev.last_error()
        return {"mu": mu, "count": ecnt}
    if kind == "pool":
        mats, _, _, intvs, seeds = zip(*st["requests"])
        err, mu, ecnt = ev.kpmdos_batch(list(mats), list(intvs), case["mdeg"], 1, case["nvec"],
                                        VEC_RADEMACHER, seeds,
                                        PREC_MIXED if case["prec"] == "mixed" else PREC_FP64)
        assert err == 0, ev.last_error()
        return {"mu": mu, "count": ecnt}
    if kind == "filter":
        err = ev.lib.evsl_amd_cheb_av_cols(
            case["cols"], st["pols"], ctypes.cast(st["X"].data_ptr(), c_double_p),
            ctypes.cast(st["Y"].data_ptr(), c_double_p),
            PREC_MIXED if case["prec"] == "mixed" else PREC_FP64)
        assert err == 0, ev.last_error()
        return {"Y": st["Y"]}
    if kind in ("solve", "batch"):
        mu, ivs, pols, mlan = _slices(ev, st)
        n, v0 = st["A"].n, st["vinit"].data_ptr()
        pairs = []
        if kind == "solve":
            for iv, pol in zip(ivs, pols):
                err, lam, Y, _ = ev.ChebLanNr(iv, mlan, 1e-8, v0, pol, n=n)
                assert err == 0, ev.last_error()
                pairs.append(_sorted(lam, Y))
        else:
            ev.set_precision(PREC_MIXED)
            err, outs = ev.ChebLanNr_batch(ivs, mlan, 1e-8, v0, pols, n=n)
            ev.set_precision(PREC_FP64)
            assert err == 0, ev.last_error()
            pairs = [_sorted(lam, Y) for lam, Y, _ in outs]
        for p in pols:
            ev.free_pol(p)
        return dict(_joined(pairs), mu=mu)
    if kind == "landos":
        err, lmin, lmax = ev.LanTrbounds(50, 200, 1e-8, st["vinit"], 1)
        assert err == 0, ev.last_error()
        _LIBC.srand(st["seed"])
        err, x, y, neig = ev.LanDos(case["nvec"], case["msteps"], case["npts"],
                                    np.array([0.0, 12.0, 0.0, 12.0]))
        assert err == 0, ev.last_error()
        return {"bounds": [lmin, lmax], "x": x, "y": y, "neig": neig}
    srv, ids = st["server"], []
    for what, m, a, b, x in st["requests"]:
        if what == "slice":
            ids.append(srv.submit_slice(m, a, b, max(5 * (case["count"] + 2), 300), 1e-8, x))
        else:
            ids.append(srv.submit_dos(m, a, b, case["mdeg"], 1, case["nvec"], VEC_RADEMACHER, x))
        assert ids[-1] >= 0, ev.last_error()
    left = 1
    while left:
        left = srv.step()
        assert left >= 0, ev.last_error()
    out = []
    for rid, (what, m, *_) in zip(ids, st["requests"]):
        if what == "slice":
            err, lam, Y, _ = srv.slice_result(rid, st["n"][m])
            out.append(_sorted(lam, Y))
        else:
            err, mu, ecnt = srv.dos_result(rid)
            out.append({"mu": mu, "count": ecnt})
        assert err == 0, ev.last_error()
    return out


# ---- what a pass cannot do without -----------------------------------------------------

def _recurrence(A, cols, steps, vs):
    """A three-term recurrence: the matrix once, and for each step, which needs
    the whole step before it, two vector blocks read and one written."""
    return {"bytes": A.nnz * (vs + 4.0) + 4.0 * A.n + 3.0 * steps * cols * A.n * vs,
            "flops": steps * cols * (2.0 * A.nnz + 4.0 * A.n)}


def _basis(n, steps):
    """Full re-orthogonalisation of `steps` Lanczos vectors in FP64."""
    return {"bytes": 8.0 * n * steps * steps, "flops": 2.0 * n * steps * steps}


def _sum(*parts):
    return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}


def work(case):
    kind = case["kind"]
    vs = 4 if case.get("prec") == "mixed" else 8
    if kind == "dos":
        return _recurrence(_matrix(case)[0], case["nvec"], case["mdeg"], 8)
    if kind == "pool":
        return _sum(*(_recurrence(r[0], case["nvec"], case["mdeg"], vs)
                      for r in _requests(case, 0)))
    if kind == "filter":
        A, lo, hi = _matrix(case)
        steps = sum(len(mu) - 1 for mu in _filters(case, lo, hi)[2]) / case["cols"]
        return _sum(_recurrence(A, case["cols"], steps, vs),
                    {"bytes": 16.0 * A.n * case["cols"], "flops": 0.0})
    if kind in ("solve", "batch"):
        # a solve needs about 2.5 Lanczos steps for each eigenpair, each one
        # filter of a degree about twice the spectrum's width in slice widths
        A, ns = _box(case["nx"], case["ny"], case["nz"]), case["nslices"]
        dims, n = (2, A.n) if case["nz"] == 1 else (3, A.n)
        below = (lambda x: n * x / (4 * math.pi)) if dims == 2 else (
            lambda x: n * x ** 1.5 / (6 * math.pi ** 2))
        steps = 2.5 * (below(case["b"]) - below(case["a"])) / ns
        deg = 2.0 * 4.0 * dims * ns / (case["b"] - case["a"])
        return _sum(_recurrence(A, case["nvec"], case["mdeg"], 8),
                    _recurrence(A, ns, steps * deg, 8 if kind == "solve" else 4),
                    *[_basis(n, steps)] * ns)
    if kind == "landos":
        A = _box(case["nx"], case["ny"], case["nz"])
        return _sum(_recurrence(A, case["nvec"], case["msteps"], 8),
                    *[_basis(A.n, case["msteps"])] * case["nvec"])
    parts = []
    for A, lo, hi in _serve_pool(case["scale"]):
        steps = 2.5 * case["count"]
        parts += [_recurrence(A, case["nvec"], case["mdeg"], 8),
                  _recurrence(A, case["per"], steps * 0.1 * A.n / case["count"], vs),
                  *[_basis(A.n, steps)] * case["per"]]
    return _sum(*parts)


# ---- the same outputs in 64 bits, from plain torch and numpy ------------------------------

class _Rows:
    """A CSR matrix with its rows padded to one length, for A X in FP64."""

    def __init__(self, A):
        ia, n = A.ia.astype(np.int64), A.n
        length = np.diff(ia)
        width = max(1, int(length.max()))
        ja, a = np.zeros((width, n), np.int64), np.zeros((width, n))
        row = np.repeat(np.arange(n), length)
        at = np.arange(int(ia[-1])) - ia[row]
        ja[at, row], a[at, row] = A.ja[:int(ia[-1])], A.a[:int(ia[-1])]
        self.ja, self.a = torch.from_numpy(ja).to(_device()), torch.from_numpy(a).to(_device())

    def __call__(self, X):
        """A X for the n x B block X"""
        out = torch.zeros_like(X)
        for j, a in zip(self.ja, self.a):
            out += a[:, None] * X[j]
        return out


def _mix64(z):
    with np.errstate(over="ignore"):
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _rademacher(n, nvec, seed):
    """The seeded +-1 vectors of the densities, unit columns (n x nvec)"""
    out = torch.empty(n, nvec, dtype=torch.float64, device=_device())
    with np.errstate(over="ignore"):
        rows = np.arange(n, dtype=np.uint64) * np.uint64(0xD1B54A32D192ED03)
        for c in range(nvec):
            col = _mix64(np.array([seed], np.uint64) +
                         np.uint64(0x9E3779B97F4A7C15) * np.uint64(c + 1))
            bit = _mix64(col ^ rows) >> np.uint64(63)
            out[:, c] = torch.from_numpy(2.0 * bit.astype(np.float64) - 1.0).to(_device())
    return out / math.sqrt(n)


def _moments(rows, n, intv, mdeg, nvec, seed):
    """Jackson-damped KPM moments and the eigenvalue count of [a, b]"""
    ctr, wid = (intv[3] + intv[2]) / 2, (intv[3] - intv[2]) / 2
    raw = np.zeros(mdeg + 1)
    raw[0] = nvec
    v = _rademacher(n, nvec, seed)
    prev, cur = None, v
    for k in range(1, mdeg + 1):
        nxt = (rows(cur) - ctr * cur) * ((1.0 if prev is None else 2.0) / wid)
        if prev is not None:
            nxt -= prev
        raw[k] = float((nxt * v).sum())
        prev, cur = cur, nxt
    k = np.arange(mdeg + 1)
    j = math.pi / (mdeg + 2)
    jac = ((1 - k / (mdeg + 2)) * math.sin(j) * np.cos(k * j) +
           math.cos(j) * np.sin(k * j) / (mdeg + 2)) / math.sin(j)
    jac[0] = 1.0
    mu = jac * raw * np.where(k == 0, 1.0, 2.0) / (nvec * math.pi)
    b1, b2 = (math.acos((min(max(x, intv[2]), intv[3]) - ctr) / wid) for x in intv[:2])
    kk = k[1:]
    count = -mu[0] * (b2 - b1) - np.sum(mu[1:] * (np.sin(kk * b2) - np.sin(kk * b1)) / kk)
    return mu, float(count * n)


def _box_eigenvalues(nx, ny, nz, a, b):
    t = [4.0 * np.sin(np.arange(1, s + 1) * (0.5 * math.pi / (s + 1))) ** 2 if s > 1 else
         np.zeros(1) for s in (nx, ny, nz)]
    ev = np.sort((t[0][:, None, None] + t[1][None, :, None] + t[2][None, None, :]).ravel())
    return ev[(ev >= a) & (ev <= b)]


def _landos(A, case, seed):
    """Lanczos density: Gauss quadrature of nvec runs, smoothed by Gaussians"""
    n, m, npts, top = A.n, case["msteps"], case["npts"], 12.0
    rows, x = _Rows(A), np.linspace(0.0, top, case["npts"])
    steps = min(m, 30)
    s2 = 2.0 * (top / (steps - 1)) ** 2 / (8.0 * math.log(1.25))
    width = math.sqrt(s2 / 2.0) * math.sqrt(-2.0 * math.log(1e-8))
    y = np.zeros(npts)
    _LIBC.srand(seed)
    draws = np.array([_LIBC.rand() for _ in range(2 * n * case["nvec"])], np.float64)
    for u in draws.reshape(case["nvec"], 2 * n) / 2147483647.0:
        v = torch.from_numpy(np.sqrt(-2.0 * np.log(u[0::2])) *
                             np.cos(2.0 * 3.1415926535 * u[1::2])).to(_device())
        V = torch.zeros(m + 1, n, dtype=torch.float64, device=_device())
        V[0] = v / v.norm()
        T = np.zeros((m, m))
        for j in range(m):
            w = rows(V[j][:, None])[:, 0]
            T[j, j] = float(w @ V[j])
            for _ in range(2):
                w = w - V[:j + 1].T @ (V[:j + 1] @ w)
            beta = float(w.norm())
            if j + 1 < m:
                T[j, j + 1] = T[j + 1, j] = beta
            V[j + 1] = w / beta
        theta, S = np.linalg.eigh(T)
        d = x[None, :] - theta[:, None]
        y += ((S[0] ** 2)[:, None] * np.exp(-d * d / s2) * (np.abs(d) < width)).sum(0)
    y /= case["nvec"] * math.sqrt(s2 * math.pi)
    total, i = 0.0, 1  # Simpson's rule, a trapezoid at the end where one interval is left
    while i < npts - 1:
        total += (x[i + 1] - x[i - 1]) * (y[i - 1] + 4 * y[i] + y[i + 1]) / 6.0
        i += 2
    if i == npts - 1:
        total += (x[i] - x[i - 1]) * (y[i] + y[i - 1]) / 2.0
    return {"bounds": [None, None], "x": x, "y": y, "neig": float(total * n)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "dos":
        A, lo, hi = _matrix(case)
        mu, count = _moments(_Rows(A), A.n, [lo + 0.05 * (hi - lo), lo + 0.1 * (hi - lo), lo, hi],
                             case["mdeg"], case["nvec"], seed)
        return {"mu": mu, "count": count}
    if kind == "pool":
        both = [_moments(_Rows(A), A.n, iv, case["mdeg"], case["nvec"], s)
                for A, _, _, iv, s in _requests(case, seed)]
        return {"mu": np.array([m for m, _ in both]), "count": np.array([c for _, c in both])}
    if kind == "filter":
        A, lo, hi = _matrix(case)
        cc, dd, mus = _filters(case, lo, hi)
        rows, deg = _Rows(A), max(len(mu) for mu in mus) - 1
        mu = torch.zeros(deg + 1, case["cols"], dtype=torch.float64)
        for c, m in enumerate(mus):
            mu[:len(m), c] = torch.from_numpy(m)
        mu = mu.to(_device())
        prev, cur = None, _vectors(case, A.n, seed).T.contiguous()
        y = mu[0] * cur
        for k in range(1, deg + 1):
            nxt = (rows(cur) - cc * cur) * ((1.0 if prev is None else 2.0) / dd)
            if prev is not None:
                nxt -= prev
            y += mu[k] * nxt
            prev, cur = cur, nxt
        return {"Y": y.T.contiguous()}
    if kind in ("solve", "batch"):
        # no value for the vectors: their signs are open
        A = _box(case["nx"], case["ny"], case["nz"])
        mu, _ = _moments(_Rows(A), A.n, [case["a"], case["b"], 0.0,
                                         8.0 if case["nz"] == 1 else 12.0],
                         case["mdeg"], case["nvec"], _SLICING)
        lam = _box_eigenvalues(case["nx"], case["ny"], case["nz"], case["a"], case["b"])
        return {"lam": lam, "Y": [None] * case["nslices"], "mu": mu}
    if kind == "landos":
        return _landos(_box(case["nx"], case["ny"], case["nz"]), case, seed)
    s2, s3 = round(case["scale"] ** 0.5), round(case["scale"] ** (1 / 3))
    sides = [(s2, s2 - 3, 1), (s3, s3 + 1, s3 + 2)]
    out, pool = [], _serve_pool(case["scale"])
    for what, m, a, b, x in _serve_requests(case, seed):
        if what == "dos":
            mu, count = _moments(_Rows(pool[m][0]), pool[m][0].n, [a, b, *pool[m][1:]],
                                 case["mdeg"], case["nvec"], x)
            out.append({"mu": mu, "count": count})
        else:
            lam = _box_eigenvalues(*sides[m], a, b) if m < 2 else None
            out.append({"lam": lam, "Y": None})
    return out
