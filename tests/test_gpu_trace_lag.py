"""GPU: ChebLanNr's convergence tests, solved while the device goes on with the next
steps: runs that end at a lagging test, by maxit at and between tests, and by maxit
while a test is under way, on a filter short enough for the tests to lag.

Bars: ChebLanNr_batch, which waits for every test, bit for bit; no draw taken."""
import numpy as np
import pytest

from evsl_amd import matrices as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("maxit", [31, 90, 91, 95, 111, 130, 400])
def test_same_run_as_waiting_for_every_test(ev, libc, maxit):
    A = M.laplacian(71, 67, 1)
    v0 = np.random.default_rng(8).uniform(-1.0, 1.0, A.n)
    assert ev.set_matrix(A) == 0, ev.last_error()
    iv, pol = np.array([0.4, 0.5, 0.0, 8.0]), ev.default_pol()
    pol.damping, pol.thresh_int, pol.thresh_ext, pol.max_deg = 2, 0.8, 0.2, 3000
    assert ev.find_pol(iv, pol) == 0
    libc.srand(3)
    err, lam, Y, res = ev.ChebLanNr(iv, maxit, 1e-8, v0, pol)
    assert err == 0, ev.last_error()
    drawn = libc.rand()
    libc.srand(3)
    assert drawn == libc.rand()
    err, outs = ev.ChebLanNr_batch([iv], maxit, 1e-8, v0, [pol])
    assert err == 0, ev.last_error()
    lam1, Y1, res1 = outs[0]
    assert np.array_equal(lam, lam1) and np.array_equal(Y, Y1) and np.array_equal(res, res1)
    if maxit == 400:
        assert len(lam) == len(M.laplacian_eigs(71, 67, 1, 0.4, 0.5))
    ev.free_pol(pol)
