"""GPU: the replay of the QL rotations at Krylov dimensions where a block holds two
rows of the eigenvector matrix in LDS (up to 3072), and above, where the matrix
stays in global memory.

Bars: a plain ChebLanNr that ends at its last step with every Ritz pair of the
interval asked for (an interval of more eigenvalues than steps) returns vectors
that are orthonormal and diagonalise p(A), both to 1e-8, whether or not they have
converged."""
import numpy as np
import pytest

from evsl_amd import matrices as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [1600, 3072, 3073])
def test_ritz_vectors_of_large_krylov_spaces(ev, steps):
    n = 6000
    A = M.perturb_diag(M.laplacian(n, 1, 1), 1.0, seed=3)
    lo, hi = M.gershgorin(A)
    iv = np.array([lo + 0.1 * (hi - lo), lo + 0.9 * (hi - lo), lo, hi])
    assert ev.set_matrix(A) == 0, ev.last_error()
    pol = ev.default_pol()
    pol.damping, pol.thresh_int, pol.thresh_ext, pol.max_deg = 2, 0.8, 0.2, 300
    assert ev.find_pol(iv, pol) == 0
    v = np.random.default_rng(2).uniform(-1.0, 1.0, n)
    err, lam, Y, res = ev.ChebLanNr(iv, steps, 1e9, v, pol)
    assert err == 0, ev.last_error()
    assert steps // 3 < len(lam) <= steps
    print(f"  {steps} steps, degree {pol.deg}: {len(lam)} Ritz pairs", flush=True)
    m = len(lam)
    assert np.max(np.abs(Y.T @ Y - np.eye(m))) <= 1e-8
    P = np.empty_like(Y, order="F")
    for j in range(0, m, 256):
        c = min(256, m - j)
        err, P[:, j:j + c] = ev.cheb_av_cols([pol] * c, Y[:, j:j + c])
        assert err == 0, ev.last_error()
    ev.free_pol(pol)
    H = Y.T @ P
    assert np.max(np.abs(H - np.diag(np.diag(H)))) <= 1e-8
