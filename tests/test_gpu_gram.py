"""GPU: the Gram product U^T U in small tiles, at row counts around its 64-row
stages and 8192-row splits and at block sizes that are no multiple of a tile,
through the mixed batched solver and ChebSI, whose Rayleigh-Ritz steps it carries.

Bar: eigenpairs of the closed-form spectrum within 1e-10, residuals below tol."""
import numpy as np
import pytest

from evsl_amd import matrices as M
from evsl_amd.evsl import PREC_FP64, PREC_MIXED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(15, 17, 1), (16, 16, 1), (64, 67, 1), (200, 203, 1)])
def test_gram_in_the_solvers(ev, size):
    nx, ny, nz = size
    A = M.perturb_diag(M.laplacian(nx, ny, nz), 1e-3, seed=2)
    n = A.n
    want_n = 14
    # the lowest eigenvalues by a dense or a sparse solver
    if n < 3000:
        w = np.linalg.eigvalsh(A.to_scipy().toarray())[:want_n + 2]
    else:
        import scipy.sparse.linalg as sla
        w = np.sort(sla.eigsh(A.to_scipy(), k=want_n + 2, sigma=0.0, tol=1e-13,
                              return_eigenvectors=False))
    b = 0.5 * (w[want_n - 1] + w[want_n])
    iv = np.array([0.0, b, 0.0, 8.001])
    assert ev.set_matrix(A) == 0, ev.last_error()
    pol = ev.default_pol()
    pol.damping, pol.thresh_int, pol.thresh_ext, pol.max_deg = 2, 0.8, 0.2, 1000
    assert ev.find_pol(iv, pol) == 0
    rng = np.random.default_rng(4)
    ev.lib.evsl_amd_set_mixed_degree_range(2, 20000)
    try:
        ev.set_precision(PREC_MIXED)
        err, outs = ev.ChebLanNr_batch([iv], min(n, 300), 1e-8, rng.uniform(-1, 1, n), [pol])
    finally:
        ev.set_precision(PREC_FP64)
        ev.lib.evsl_amd_set_mixed_degree_range(32, 20000)
    assert err == 0, ev.last_error()
    lam, _, res = outs[0]
    assert len(lam) == want_n and np.max(res) < 1e-8
    assert np.max(np.abs(np.sort(lam) - w[:want_n])) <= 1e-10 * 8
    err, lam, _, res = ev.ChebSI(want_n + 70, iv, 400, 1e-8, rng.standard_normal((n, want_n + 70)),
                                 pol)
    ev.free_pol(pol)
    assert err == 0, ev.last_error()
    assert len(lam) == want_n and np.max(res) < 1e-8
    assert np.max(np.abs(np.sort(lam) - w[:want_n])) <= 1e-10 * 8
