"""GPU: whole Chebyshev series in one launch where values carry their tags.

Bars, against the filter run one launch a degree (bit for bit):
* symmetric band and lattice matrices from one row to the largest a series takes
  and one more, around a wave's, a workgroup's and a lane's shares; rows of at
  most six entries out of twelve pairs and rows of twelve; FP64 and the mixed
  form; one column to more than four turns;
* matrices of different sizes after each other and again, so that the rings hold
  older values of other layouts;
* a matrix with unpaired rows (not symmetric) gives the same result as well."""
import numpy as np
import pytest

from evsl_amd import matrices as M
from evsl_amd.evsl import PREC_FP64, PREC_MIXED
from evsl_amd.types import HostCsr

pytestmark = pytest.mark.gpu

POLLS = 200000


def sym_band(n, offsets, seed, keep=0.7):
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    S = sp.diags(rng.uniform(-1.0, 1.0, n)).tocsr()
    for o in offsets:
        if o >= n:
            continue
        r = np.arange(n - o)
        r = r[rng.random(r.size) < keep]
        U = sp.coo_matrix((np.full(r.size, rng.uniform(0.2, 1.0)), (r, r + o)), shape=(n, n))
        S = S + U + U.T
    S = sp.csr_matrix(S)
    S.sort_indices()
    return HostCsr.from_scipy(S)


def check(ev, A, cols, degs=(8, 9, 30, 65, 130, 41, 23, 12)):
    lo, hi = M.gershgorin(A)
    lo, hi = lo - 0.1, hi + 0.1
    assert ev.set_matrix(A) == 0, ev.last_error()
    X = np.random.default_rng(5).uniform(-1.0, 1.0, (A.n, max(cols)))
    pols = []
    for i in range(max(cols)):
        pol = ev.default_pol()
        pol.deg = degs[i % len(degs)]
        a = lo + (0.2 + 0.02 * i) * (hi - lo)
        assert ev.find_pol(np.array([a, a + 0.1 * (hi - lo), lo, hi]), pol) == 0
        pols.append(pol)
    try:
        for prec in (PREC_FP64, PREC_MIXED):
            ev.set_series_polls(0)
            err, ref = ev.cheb_av_cols(pols, X, prec)
            assert err == 0, ev.last_error()
            ev.set_series_polls(POLLS)
            for c in cols:
                for _ in range(2):
                    err, Y = ev.cheb_av_cols(pols[:c], X[:, :c], prec)
                    assert err == 0, ev.last_error()
                    assert np.array_equal(Y, ref[:, :c]), (prec, c)
    finally:
        ev.set_series_polls(POLLS)
        for p in pols:
            ev.free_pol(p)


@pytest.mark.parametrize("n", [1, 64, 65, 4096, 4097, 32768, 32769, 65536, 65537])
@pytest.mark.parametrize("offsets", [[1], [1, 7, 64], [1, 2, 5, 9, 40, 900]])
def test_tagged_series_same_bits(ev, n, offsets):
    check(ev, sym_band(n, offsets, seed=n), (1, 8, 9, 33) if n < 5000 else (1, 8, 9))


@pytest.mark.parametrize("L", [5, 16, 31, 40])
def test_tagged_series_lattice(ev, L):
    check(ev, M.anderson(L, 16.5, seed=L), (1, 8, 16))


def test_rings_of_other_layouts(ev):
    mats = [sym_band(3000, [1, 50], 1), M.anderson(14, 16.5, seed=3), sym_band(700, [1, 2, 3], 2)]
    for _ in range(3):
        for A in mats:
            check(ev, A, (1, 5, 24))


def test_unpaired_rows(ev):
    import scipy.sparse as sp
    S = sp.csr_matrix(sp.triu(sym_band(2000, [1, 2, 30], 4).to_scipy()))
    S.sort_indices()
    check(ev, HostCsr.from_scipy(S), (1, 8))
