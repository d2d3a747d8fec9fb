"""GPU: LanDos runs several start vectors together; one vector, fewer, as many and
more than a group takes, and the two ways a run can change the ones after it: a
lucky break, which shortens all later runs, and a replacement vector, which takes
a draw that a later run would have started from.

Bars: the oracle's LanDos (SRC/landos.c:37-196) on the same libc draws, as the
parity test of one call: rtol 1e-9, atol 1e-12; and the same number of draws."""
import numpy as np
import pytest
import scipy.sparse as sp

from evsl_amd import matrices as M

pytestmark = pytest.mark.gpu


def both(ev, oracle, libc, A, nvec, msteps, npts, intv):
    assert ev.set_matrix(A) == 0, ev.last_error()
    oracle.set_csr(A)
    libc.srand(31)
    eg, xg, yg, ng = ev.LanDos(nvec, msteps, npts, intv)
    drawn_g = libc.rand()
    libc.srand(31)
    eo, xo, yo, no = oracle.LanDos(nvec, msteps, npts, intv)
    drawn_o = libc.rand()
    assert eg == eo == 0, ev.last_error()
    assert drawn_g == drawn_o
    assert np.array_equal(xg, xo)
    np.testing.assert_allclose(yg, yo, rtol=1e-9, atol=1e-12)
    assert ng == pytest.approx(no, rel=1e-9)


@pytest.mark.parametrize("nvec", [1, 2, 3, 7, 14, 23])
@pytest.mark.parametrize("size", [(31, 29, 1), (11, 12, 13)])
def test_group_sizes(ev, oracle, libc, nvec, size):
    both(ev, oracle, libc, M.laplacian(*size), nvec, 30, 101,
         np.array([0.5, 3.0, 0.0, 8.0 if size[2] == 1 else 12.0]))


def test_irregular_matrix(ev, oracle, libc):
    A = M.random_symmetric(3001, 2, 40, seed=9)
    lo, hi = M.gershgorin(A)
    both(ev, oracle, libc, A, 9, 30, 100, np.array([lo, hi, lo, hi]))


def test_too_large_for_groups(ev, oracle, libc):
    both(ev, oracle, libc, M.laplacian(270, 251, 1), 3, 12, 64, np.array([0.5, 3.0, 0.0, 8.0]))


def test_lucky_break_shortens_later_runs(ev, oracle, libc):
    # six distinct eigenvalues: every run ends after six steps
    T = sp.block_diag([M.laplacian(6, 1, 1).to_scipy()] * 120).tocoo()
    A = M._csr_from_coo(T.shape[0], T.row, T.col, T.data)
    both(ev, oracle, libc, A, 9, 20, 64, np.array([0.1, 3.9, 0.0, 4.0]))


def test_replacement_vectors_take_draws(ev, oracle, libc):
    # the stated spectrum sets the breakdown level (1e-13 of it) to 4.0, which the
    # squared norms of this grid's steps lie on both sides of: the number of draws
    # says how many steps of every run were replaced
    both(ev, oracle, libc, M.laplacian(30, 29, 1), 11, 16, 64, np.array([0.5, 3.0, 0.0, 4.0e13]))
