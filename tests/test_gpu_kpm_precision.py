"""GPU: the rounding of FP64 densities, against the same vectors' moments from an
80-bit recurrence (SRC/spslice.c:29-148 forms v^T T_k v at every step).

Bar, of the norm of the moments beyond the first: three times what the recurrence
and its dots give in plain float64 on the CPU, 2.9e-16, 5.8e-16 and 1.2e-16 for the
three spectra (half as many steps with two products each: 4.2e-15, 4.1e-15 and
8.1e-16)."""
import numpy as np
import pytest

from evsl_amd import matrices as M
from evsl_amd.evsl import PREC_FP64, VEC_RADEMACHER, Server

pytestmark = pytest.mark.gpu

MDEG, NVEC, SEED = 200, 20, 77
GRID, RANDOM = M.laplacian(64, 60, 1), M.random_symmetric(5000, 3, 20, seed=4)
CASES = {"grid": (GRID, 0.0, 8.0, 2.9e-16), "grid_wider": (GRID, -0.01, 8.02, 5.8e-16),
         "random": (RANDOM, *M.gershgorin(RANDOM), 1.2e-16)}


def mix64(z):
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def signs(n):
    """The seeded +-1 vectors of kpmdos_ex, one a column."""
    with np.errstate(over="ignore"):
        rows = np.arange(n, dtype=np.uint64) * np.uint64(0xD1B54A32D192ED03)
        col = mix64(np.uint64(SEED) +
                    np.uint64(0x9E3779B97F4A7C15) * np.arange(1, NVEC + 1, dtype=np.uint64))
        return 2.0 * (mix64(col[None, :] ^ rows[:, None]) >> np.uint64(63)).astype(np.float64) - 1.0


def times(A, X):
    """A X in X's precision, a row's products in their order."""
    out = np.zeros_like(X)
    length = np.diff(A.ia)
    for k in range(length.max()):
        r = np.nonzero(length > k)[0]
        at = A.ia[r] + k
        out[r] += A.a[at].astype(X.dtype)[:, None] * X[A.ja[at]]
    return out


def moments(A, lo, hi, dtype, products=False):
    """Undamped mu_k, k = 1..MDEG, of the mean over the vectors."""
    n, c, w = A.n, dtype((lo + hi) / 2), dtype((hi - lo) / 2)
    v = signs(n).astype(dtype) / np.sqrt(dtype(n))
    t0, t1, raw = v, (times(A, v) - c * v) * (dtype(1) / w), np.zeros(MDEG + 1, dtype)
    d1 = np.sum(v * t1)
    for k in range(1, (MDEG // 2 if products else MDEG) + 1):
        if products:
            raw[2 * k - 1] = 2 * np.sum(t1 * t0) - d1
            raw[2 * k] = 2 * np.sum(t1 * t1) - NVEC
        else:
            raw[k] = np.sum(v * t1)
        t0, t1 = t1, (dtype(2) / w) * (times(A, t1) - c * t1) - t0
    return 2 * raw[1:] / (NVEC * dtype(np.pi))


def off(mu, ref):
    return float(np.sqrt(np.sum((mu - ref) ** 2) / np.sum(ref ** 2)))


@pytest.mark.parametrize("name", sorted(CASES))
def test_rounding_of_moments(ev, name):
    A, lo, hi, model = CASES[name]
    intv = np.array([0.5, 1.0, lo, hi])
    assert ev.set_matrix(A) == 0, ev.last_error()
    err, mu, _ = ev.kpmdos(MDEG, 0, NVEC, intv, vec_kind=VEC_RADEMACHER, seed=SEED)
    assert err == 0, ev.last_error()
    err, many, _ = ev.kpmdos_batch([A], [intv], MDEG, 0, NVEC, VEC_RADEMACHER, [SEED], PREC_FP64)
    assert err == 0, ev.last_error()
    srv = Server(ev, 1 << 32, PREC_FP64)
    rid = srv.submit_dos(srv.add_matrix(A, lo, hi), 0.5, 1.0, MDEG, 0, NVEC, seed=SEED)
    while srv.step() > 0:
        pass
    err, served, _ = srv.dos_result(rid)
    srv.close()
    assert err == 0
    ref = moments(A, lo, hi, np.longdouble, products=True)
    for got in (mu, many[0], served):
        e = off(got[1:], ref)
        print(f"  {name}: {e:.2e}", flush=True)
        assert e <= 3 * model
