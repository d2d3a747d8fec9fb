"""GPU: the Lanczos runs of LanBounds and LanDos (SRC/lanbounds.c,
SRC/landos.c:37-196) with a user's operator, whose steps end at a lucky break.

Bars: the operator is called once for every step that is used, with finite
vectors, and in the order of the reference (a vector is drawn from libc rand()
after the calls of the run before it); the results equal those of the same matrix
as a CSR operator to 1e-10."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

from evsl_amd import matrices as M

pytestmark = pytest.mark.gpu


class Operator:
    def __init__(self, ev, S):
        self.ev, self.S = ev, S
        self.calls, self.finite = 0, True

    def __call__(self, x, y, data):
        n = self.S.shape[0]
        v = self.ev.from_device(C.cast(x, C.c_void_p), n)
        self.finite = self.finite and bool(np.all(np.isfinite(v)))
        self.calls += 1
        w = np.ascontiguousarray(self.S @ v)
        self.ev.lib.evsl_memcpy_host_to_device(C.cast(y, C.c_void_p), w.ctypes.data, 8 * n)


@pytest.fixture
def matrix():
    # six distinct eigenvalues: a run ends after six steps
    T = sp.block_diag([M.laplacian(6, 1, 1).to_scipy()] * 120).tocoo()
    return M._csr_from_coo(T.shape[0], T.row, T.col, T.data)


def test_lanbounds(ev, matrix):
    v = np.random.default_rng(4).standard_normal(matrix.n)
    assert ev.set_matrix(matrix) == 0, ev.last_error()
    err, lo, hi = ev.LanBounds(40, v)
    assert err == 0
    op = Operator(ev, matrix.to_scipy())
    assert ev.set_matvec(matrix.n, op) == 0
    err, lo_u, hi_u = ev.LanBounds(40, v)
    assert err == 0 and op.finite and op.calls == 6
    assert lo_u == pytest.approx(lo, rel=1e-10) and hi_u == pytest.approx(hi, rel=1e-10)


def test_landos(ev, libc, matrix):
    iv = np.array([2.1, 5.9, 2.0, 6.0])
    assert ev.set_matrix(matrix) == 0, ev.last_error()
    libc.srand(31)
    err, x, y, cnt = ev.LanDos(5, 20, 64, iv)
    assert err == 0
    op = Operator(ev, matrix.to_scipy())
    assert ev.set_matvec(matrix.n, op) == 0
    libc.srand(31)
    err, x_u, y_u, cnt_u = ev.LanDos(5, 20, 64, iv)
    assert err == 0 and op.finite and op.calls == 5 * 6
    assert np.array_equal(x, x_u)
    np.testing.assert_allclose(y_u, y, rtol=1e-10, atol=1e-12)
    assert cnt_u == pytest.approx(cnt, rel=1e-10)


def test_draws_follow_the_calls(ev, libc):
    # an operator that draws itself: the start vectors of later runs depend on it;
    # the stated spectrum asks for replacement vectors as well
    A = M.laplacian(30, 29, 1)
    S, nvec, msteps = A.to_scipy(), 3, 9

    def seen(spectrum):
        op, first = Operator(ev, S), []

        def call(x, y, data):
            op(x, y, data)
            first.append(libc.rand())

        assert ev.set_matvec(A.n, call) == 0
        libc.srand(7)
        err = ev.LanDos(nvec, msteps, 64, np.array([0.5, 3.0, 0.0, spectrum]))[0]
        assert err == 0 and op.finite and op.calls == nvec * msteps
        return first

    got = seen(8.0)
    # the same stream by hand: a vector's draws, then one after each call
    libc.srand(7)
    want, out = [], np.empty(A.n)
    for _ in range(nvec):
        ev.lib.randn_double(A.n, out.ctypes.data_as(C.POINTER(C.c_double)))
        want += [libc.rand() for _ in range(msteps)]
    assert got == want
    replaced = seen(4.0e13)
    libc.srand(7)
    ev.lib.randn_double(A.n, out.ctypes.data_as(C.POINTER(C.c_double)))
    assert replaced[0] == libc.rand()
    assert replaced[1:] != got[1:]
