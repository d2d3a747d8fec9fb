"""GPU: whole Chebyshev series in one launch (evsl_amd_set_series_polls).

Bars:
* the bits of the filter run one launch a degree (0 polls): sizes from one row
  to the largest a series takes and one more, around whole workgroup shares; one
  and eight columns, equal and different degrees; FP64 and the mixed form;
  offsets on one side only;
* a wait that is given a single look ends, the filter is run again by launches,
  and its result is the same;
* a batched solve, the plain ChebLanNr and the request loop give the same bits
  with series launches, without them and after a failed one."""
import numpy as np
import pytest

from evsl_amd import matrices as M
from evsl_amd.evsl import PREC_FP64, PREC_MIXED, Server
from evsl_amd.types import HostCsr

pytestmark = pytest.mark.gpu

POLLS = 200000


def banded(n, offsets, seed):
    rng = np.random.default_rng(seed)
    rows = [np.arange(n)]
    cols = [np.arange(n)]
    vals = [rng.uniform(-1.0, 1.0, n)]
    for o in offsets:
        r = np.arange(max(0, -o), min(n, n - o))
        r = r[rng.random(r.size) < 0.7]
        rows.append(r)
        cols.append(r + o)
        vals.append(np.full(r.size, rng.uniform(0.2, 1.0)))
    import scipy.sparse as sp
    m = sp.coo_matrix((np.concatenate(vals), (np.concatenate(rows), np.concatenate(cols))),
                      shape=(n, n)).tocsr()
    m.sort_indices()
    return HostCsr.from_scipy(m)


def filters(ev, lo, hi, degs):
    out = []
    for i, d in enumerate(degs):
        pol = ev.default_pol()
        pol.deg = d
        a = lo + (0.3 + 0.05 * i) * (hi - lo)
        assert ev.find_pol(np.array([a, a + 0.1 * (hi - lo), lo, hi]), pol) == 0
        out.append(pol)
    return out


@pytest.mark.parametrize("n", [1, 63, 2048, 2049, 16384, 16385, 65536, 65537])
@pytest.mark.parametrize("offsets", [[-1, 1], [-7, -3, -1, 1, 3, 7],
                                     [-900, -40, -9, -5, -2, -1, 1, 2, 5, 9, 40, 900],
                                     [1, 2, 5, 9, 31, 64]])
def test_series_same_bits(ev, n, offsets):
    A = banded(n, offsets, seed=n)
    lo, hi = M.gershgorin(A)
    lo, hi = lo - 0.1, hi + 0.1
    assert ev.set_matrix(A) == 0, ev.last_error()
    X = np.random.default_rng(5).uniform(-1.0, 1.0, (n, 8))
    pols = filters(ev, lo, hi, [8, 9, 30, 17, 8, 41, 23, 12])
    try:
        for prec in (PREC_FP64, PREC_MIXED):
            for cols in (1, 3, 8):
                ev.set_series_polls(0)
                err, ref = ev.cheb_av_cols(pols[:cols], X[:, :cols], prec)
                assert err == 0, ev.last_error()
                ev.set_series_polls(POLLS)
                err, Y = ev.cheb_av_cols(pols[:cols], X[:, :cols], prec)
                assert err == 0, ev.last_error()
                assert np.array_equal(Y, ref), (prec, cols)
                ev.set_series_polls(1)
                err, Y = ev.cheb_av_cols(pols[:cols], X[:, :cols], prec)
                assert err == 0, ev.last_error()
                assert np.array_equal(Y, ref), (prec, cols, "one look")
    finally:
        ev.set_series_polls(POLLS)
        for p in pols:
            ev.free_pol(p)


@pytest.mark.parametrize("polls", [1, POLLS])
def test_solvers_same_bits(ev, polls):
    A = M.laplacian(40, 37, 1)
    ivs = [np.array([0.3, 0.45, 0.0, 8.0]), np.array([0.45, 0.6, 0.0, 8.0])]
    pols = []
    for iv in ivs:
        pol = ev.default_pol()
        pol.damping, pol.thresh_int, pol.thresh_ext, pol.max_deg = 2, 0.8, 0.2, 3000
        assert ev.find_pol(iv, pol) == 0
        pols.append(pol)
    v0 = np.random.default_rng(3).uniform(-1.0, 1.0, A.n)
    assert ev.set_matrix(A) == 0, ev.last_error()
    out = {}
    try:
        for p in (0, polls):
            got = []
            for prec in (PREC_FP64, PREC_MIXED):
                ev.set_series_polls(p)
                ev.set_precision(prec)
                err, lam, Y, res = ev.ChebLanNr(ivs[0], 200, 1e-8, v0, pols[0])
                assert err == 0, ev.last_error()
                got.append((lam, Y, res))
                ev.set_series_polls(p)
                err, outs = ev.ChebLanNr_batch(ivs, 200, 1e-8, v0, pols)
                assert err == 0, ev.last_error()
                got += outs
                ev.set_precision(PREC_FP64)
                ev.set_series_polls(p)
                srv = Server(ev, 1 << 32, prec)
                mid = srv.add_matrix(A, 0.0, 8.0)
                ids = [srv.submit_slice(mid, iv[0], iv[1], 200, 1e-8, v0) for iv in ivs]
                while srv.step():
                    pass
                for i in ids:
                    err, lam, Y, res = srv.slice_result(i, A.n)
                    assert err == 0
                    got.append((lam, Y, res))
                srv.close()
            out[p] = got
    finally:
        ev.set_series_polls(POLLS)
        ev.set_precision(PREC_FP64)
        for p in pols:
            ev.free_pol(p)
    assert len(out[0][0][0]) > 5
    for a, b in zip(out[0], out[polls]):
        assert all(np.array_equal(x, y) for x, y in zip(a, b))
