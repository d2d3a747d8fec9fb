"""GPU: the replay of the QL rotations that turns a tridiagonal matrix's
eigenvectors into Ritz vectors, at Krylov dimensions where a block holds 16, 8
and 4 rows of the eigenvector matrix in LDS, where its last block is partly
empty, and where only a few sweeps or split blocks are recorded.

Bar: a plain ChebLanNr whose Krylov space is the whole space (n steps, so the
Ritz vectors are eigenvectors) finds every eigenvalue of a dense spectrum in the
interval within 1e-10, with residuals below 1e-8 and eigenvectors orthonormal to
1e-8."""
import numpy as np
import pytest

from evsl_amd import matrices as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [31, 64, 383, 385, 769, 1000])
def test_ritz_vectors_at_every_row_count(ev, n):
    A = M.perturb_diag(M.laplacian(n, 1, 1), 1.0, seed=n)
    D = A.to_scipy().toarray()
    lo, hi = M.gershgorin(A)
    w = np.linalg.eigvalsh(D)
    a, b = 0.5 * (w[n // 3] + w[n // 3 + 1]), 0.5 * (w[n // 3 + 12] + w[n // 3 + 13])
    assert ev.set_matrix(A) == 0, ev.last_error()
    pol = ev.default_pol()
    pol.damping, pol.thresh_int, pol.thresh_ext, pol.max_deg = 2, 0.8, 0.2, 1500
    assert ev.find_pol(np.array([a, b, lo, hi]), pol) == 0
    v = np.random.default_rng(2).uniform(-1.0, 1.0, n)
    err, lam, Y, res = ev.ChebLanNr(np.array([a, b, lo, hi]), n, 1e-8, v, pol)
    ev.free_pol(pol)
    assert err == 0, ev.last_error()
    want = w[(w >= a) & (w <= b)]
    assert len(lam) == len(want)
    assert np.max(np.abs(np.sort(lam) - want)) <= 1e-10
    assert np.max(res) < 1e-8
    assert np.max(np.abs(Y.T @ Y - np.eye(len(lam)))) <= 1e-8
