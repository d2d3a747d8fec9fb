"""GPU: the two moments a step of the FP64 KPM series, and the sums of several
degrees in one launch, at the numbers of moments where they can go wrong: one
moment, odd and even numbers, and one less and one more than a whole number of
summed groups of 16 steps.

Bar: with the same libc rand() vectors the moments agree with the oracle's
kpmdos (SRC/spslice.c:29-148), which forms every v^T T_k v, within 1e-12."""
import ctypes

import numpy as np
import pytest

from evsl_amd import matrices as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mdeg", [1, 2, 3, 31, 32, 33, 63, 64, 65, 97])
@pytest.mark.parametrize("nvec", [1, 7, 33])
def test_moments_at_every_kind_of_degree(ev, oracle, mdeg, nvec):
    A = M.perturb_diag(M.laplacian(23, 19, 1), 1e-3, seed=4)
    intv = np.array([0.5, 1.5, 0.0, 8.001])
    assert ev.set_matrix(A) == 0, ev.last_error()
    oracle.set_csr(A)
    libc = ctypes.CDLL(None)
    libc.srand(17)
    err, mu, ecnt = ev.kpmdos(mdeg, 1, nvec, intv)
    assert err == 0, ev.last_error()
    libc.srand(17)
    err, mu_o, ecnt_o = oracle.kpmdos(mdeg, 1, nvec, intv)
    assert err == 0
    assert np.max(np.abs(mu - mu_o)) <= 1e-12
    assert abs(ecnt - ecnt_o) <= 1e-9 * max(1.0, abs(ecnt_o))
