"""GPU: what becomes of a series launch (evsl_amd_series_counts): that the filters
of small row-mask matrices run as one and succeed, and that a failed one is
noticed and its filter run again.

Bar: the bits of the filter run one launch a degree (0 polls)."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

from evsl_amd import matrices as M
from evsl_amd.evsl import PREC_FP64, PREC_MIXED, Server
from evsl_amd.types import HostCsr, PolParams
from test_gpu_series_tags import POLLS, sym_band

pytestmark = pytest.mark.gpu

ALL = 512  # workgroups of a series launch


def filters(ev, A, ncols, deg=30):
    lo, hi = M.gershgorin(A)
    lo, hi = lo - 0.1, hi + 0.1
    out = []
    for i in range(ncols):
        pol = ev.default_pol()
        pol.deg = deg + i % 3
        a = lo + (0.2 + 0.02 * i) * (hi - lo)
        assert ev.find_pol(np.array([a, a + 0.1 * (hi - lo), lo, hi]), pol) == 0
        out.append(pol)
    return out


def run(ev, pols, X, prec=PREC_FP64, polls=POLLS):
    """The filtered columns, and the series launches and failures they took."""
    ev.set_series_polls(polls)
    n0, f0, _ = ev.series_counts()
    err, Y = ev.cheb_av_cols(pols, X, prec)
    assert err == 0, ev.last_error()
    n1, f1, _ = ev.series_counts()
    return Y, n1 - n0, f1 - f0


@pytest.fixture
def series(ev):
    yield ev
    ev.set_series_polls(POLLS)
    ev.set_series_workgroups(ALL)


@pytest.mark.parametrize("n", [1, 63, 2049, 16385, 65536])
@pytest.mark.parametrize("offsets", [[1], [1, 3, 7], [1, 2, 5, 9, 40, 900]])
def test_series_run_and_fail(series, n, offsets):
    ev = series
    A = sym_band(n, offsets, seed=n)
    assert ev.set_matrix(A) == 0, ev.last_error()
    pols = filters(ev, A, 8)
    X = np.random.default_rng(5).uniform(-1.0, 1.0, (n, 8))
    for prec in (PREC_FP64, PREC_MIXED):
        for cols in (1, 3, 8):
            ref, launched, _ = run(ev, pols[:cols], X[:, :cols], prec, 0)
            assert launched == 0
            Y, launched, failed = run(ev, pols[:cols], X[:, :cols], prec)
            assert (launched, failed) == (1, 0) and np.array_equal(Y, ref)
            Y, launched, failed = run(ev, pols[:cols], X[:, :cols], prec, 1)
            assert launched == 1 and np.array_equal(Y, ref)
            if n > 2000:  # several waves: none of them sees the others at one look
                assert failed == 1 and ev.series_counts()[2]
    for p in pols:
        ev.free_pol(p)


@pytest.mark.parametrize("L", [5, 16, 31, 40])
def test_series_run_on_lattices(series, L):
    # rows of six entries out of twelve pairs; columns that take turns on an XCD
    ev = series
    A = M.anderson(L, 16.5, seed=L)
    assert ev.set_matrix(A) == 0, ev.last_error()
    pols = filters(ev, A, 33)
    X = np.random.default_rng(5).uniform(-1.0, 1.0, (A.n, 33))
    for prec in (PREC_FP64, PREC_MIXED):
        ref, _, _ = run(ev, pols, X, prec, 0)
        for cols in (1, 16, 33):
            Y, launched, failed = run(ev, pols[:cols], X[:, :cols], prec)
            assert (launched, failed) == (-(-cols // 16), 0)
            assert np.array_equal(Y, ref[:, :cols])
        if L > 5:
            Y, launched, failed = run(ev, pols, X, prec, 1)
            assert launched == 3 and failed > 0 and np.array_equal(Y, ref)
    for p in pols:
        ev.free_pol(p)


def test_a_failure_lasts_until_the_next_start(series):
    ev = series
    A = sym_band(5000, [1, 70], seed=1)
    X = np.random.default_rng(5).uniform(-1.0, 1.0, (A.n, 1))
    pols = filters(ev, A, 1)
    assert ev.set_matrix(A) == 0, ev.last_error()
    assert run(ev, pols, X, polls=1)[2] == 1
    n0 = ev.series_counts()[0]
    err, ref = ev.cheb_av_cols(pols, X)
    assert err == 0 and ev.series_counts()[0] == n0 and ev.series_counts()[2]
    assert ev.finish() == 0 and ev.start() == 0, ev.last_error()
    assert ev.series_counts() == (0, 0, False)
    assert ev.set_matrix(A) == 0, ev.last_error()
    ev.set_series_polls(POLLS)
    err, Y = ev.cheb_av_cols(pols, X)
    assert err == 0 and np.array_equal(Y, ref)
    assert ev.series_counts() == (1, 0, False)
    for p in pols:
        ev.free_pol(p)


@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED])
@pytest.mark.parametrize("matrix", ["diagonal", "blocks", "chain"])
def test_missing_workgroups(series, matrix, prec):
    ev = series
    n = 65536
    offsets = [] if matrix == "diagonal" else [1]
    A = sym_band(n, offsets, seed=2, keep=1.0)
    if matrix == "blocks":  # no entry across a multiple of 1024 rows, a workgroup's share
        S = A.to_scipy().tocoo()
        keep = S.row // 1024 == S.col // 1024
        S = sp.csr_matrix(sp.coo_matrix((S.data[keep], (S.row[keep], S.col[keep])), shape=(n, n)))
        S.sort_indices()
        A = HostCsr.from_scipy(S)
    assert ev.set_matrix(A) == 0, ev.last_error()
    pols = filters(ev, A, 9)
    X = np.random.default_rng(5).uniform(-1.0, 1.0, (n, 9))
    ref, _, _ = run(ev, pols, X, prec, 0)
    for groups in (1, ALL // 2, ALL - 8):
        assert ev.set_series_workgroups(groups) == 0
        Y, launched, failed = run(ev, pols, X, prec, 2000)
        assert (launched, failed) == (1, 1) and np.array_equal(Y, ref), groups
    for p in pols:
        ev.free_pol(p)


def on_device(ev, pols, p_in, p_out, prec):
    P = (PolParams * len(pols))(*pols)
    return ev.lib.evsl_amd_cheb_av_cols(len(pols), P, C.cast(p_in, C.POINTER(C.c_double)),
                                        C.cast(p_out, C.POINTER(C.c_double)), prec)


@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED])
@pytest.mark.parametrize("cols", [1, 9])
@pytest.mark.parametrize("n", [5000, 65536])
def test_in_place(series, n, cols, prec):
    ev = series
    A = sym_band(n, [1], seed=2, keep=1.0)
    assert ev.set_matrix(A) == 0, ev.last_error()
    pols = filters(ev, A, cols, deg=9)
    X = np.asfortranarray(np.random.default_rng(5).uniform(-1.0, 1.0, (n, cols)))
    ref, _, _ = run(ev, pols, X, prec, 0)
    # one workgroup of an XCD missing: the rows far from its share are done before
    # its neighbours' waits end
    for polls, groups in ((POLLS, ALL), (2000, ALL - 8), (1, ALL)):
        ev.set_series_workgroups(groups)
        ev.set_series_polls(polls)
        p = ev.to_device(X.T)
        assert on_device(ev, pols, p, p, prec) == 0, ev.last_error()
        Y = ev.from_device(p, n * cols).reshape(cols, n).T
        ev.free_device(p)
        assert np.array_equal(Y, ref), (polls, groups)
    for q in pols:
        ev.free_pol(q)


@pytest.mark.parametrize("shift", [-3, 1, 5])
@pytest.mark.parametrize("size,cols", [((64, 60, 1), 9), ((450, 450, 1), 20)])
def test_ranges_that_overlap(series, size, cols, shift):
    ev = series
    A = M.laplacian(*size)
    assert ev.set_matrix(A) == 0, ev.last_error()
    pols = filters(ev, A, cols, deg=9)
    X = np.asfortranarray(np.random.default_rng(5).uniform(-1.0, 1.0, (A.n, cols)))
    for prec in (PREC_FP64, PREC_MIXED):
        ref, _, _ = run(ev, pols, X, prec, 0)
        ev.set_series_polls(POLLS)
        at = max(0, -shift)
        whole = np.zeros((cols + abs(shift), A.n))
        whole[at:at + cols] = X.T
        p = ev.to_device(whole)
        assert on_device(ev, pols, p + 8 * A.n * at, p + 8 * A.n * (at + shift), prec) == 0
        Y = ev.from_device(p, whole.size).reshape(whole.shape)[at + shift:at + shift + cols].T
        ev.free_device(p)
        assert np.array_equal(Y, ref), prec
    for q in pols:
        ev.free_pol(q)


@pytest.mark.parametrize("polls", [POLLS, 1])
def test_many_launches_before_a_check(series, polls):
    # 33 matrices that are filtered each on its own (more than 32 MB a launch), two
    # launches of at most 16 columns for each
    ev = series
    A = M.laplacian(65536, 1, 1)
    lo, hi = M.gershgorin(A)
    pol = ev.default_pol()
    pol.damping, pol.thresh_int, pol.thresh_ext, pol.max_deg = 2, 0.8, 0.2, 300
    v = np.random.default_rng(3).uniform(-1.0, 1.0, A.n)
    got = []
    for p in (0, polls):
        ev.set_series_polls(p)
        n0, f0, _ = ev.series_counts()
        srv = Server(ev, 1 << 37, PREC_FP64)
        ids = []
        for m in range(33):
            mid = srv.add_matrix(A, lo, hi)
            for s in range(17):
                a = lo + 0.4 + 0.1 * s
                ids.append(srv.submit_slice(mid, a, a + 0.15, 3, 1e-8, v, pol))
        while (more := srv.step()) > 0:
            pass
        assert more == 0, ev.last_error()
        n1, f1, off = ev.series_counts()
        if p == POLLS:
            assert n1 - n0 >= 66 and f1 == f0 and not off
        elif p == 1:
            assert n1 - n0 >= 64 and f1 > f0 and off
        out = [srv.slice_result(i, A.n) for i in ids]
        got.append(out)
        srv.close()
    for a, b in zip(*got):
        assert a[0] == b[0] == 0 and all(np.array_equal(x, y) for x, y in zip(a[1:], b[1:]))


def test_forced_layout(series):
    ev = series
    A = M.laplacian(24, 24, 24)
    assert ev.set_matrix(A) == 0, ev.last_error()
    pols = filters(ev, A, 4)
    X = np.random.default_rng(5).uniform(-1.0, 1.0, (A.n, 4))
    ref, launched, _ = run(ev, pols, X)
    assert launched == 1
    assert ev.set_spmm_layout(4, PREC_FP64, 1, 11) == 0
    Y, launched, _ = run(ev, pols, X)
    assert launched == 0 and np.array_equal(Y, ref)
    assert run(ev, pols, X, PREC_MIXED)[1] == 1  # the mixed form's layouts are its own
    assert ev.set_spmm_layout(4, PREC_FP64, 1, -1) == 0
    assert run(ev, pols, X)[1] == 1
    for p in pols:
        ev.free_pol(p)
