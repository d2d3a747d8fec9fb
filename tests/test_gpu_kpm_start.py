"""GPU: the start blocks of batched densities, made for all requests together, and
FP32 values shared by requests of one matrix, centre and scale.

Bars: in FP64 every request equal, bit for bit, to kpmdos_ex on its matrix with its
seed, for both kinds of vector, matrices from one row up and vector counts on
either side of the column blocks; in the mixed form every request equal to the
same request alone."""
import numpy as np
import pytest

from evsl_amd import matrices as M
from evsl_amd.evsl import PREC_FP64, PREC_MIXED, VEC_GAUSSIAN, VEC_RADEMACHER

pytestmark = pytest.mark.gpu


def requests():
    mats = [M.laplacian(1, 1, 1), M.laplacian(2, 1, 1), M.laplacian(37, 31, 1),
            M.random_symmetric(2049, 3, 70, seed=4), M.laplacian(24, 23, 22)]
    out = []
    for i, A in enumerate(mats):
        lo, hi = M.gershgorin(A)
        lo, hi = lo - 0.5, hi + 0.5
        w = 0.25 * (hi - lo)
        for iv in ([lo, lo + w, lo, hi], [lo + w, lo + 2 * w, lo, hi], [lo, lo + w, lo, hi + w]):
            out.append((A, np.array(iv), 1000 + 7 * len(out)))
    return out


@pytest.mark.parametrize("kind", [VEC_RADEMACHER, VEC_GAUSSIAN])
@pytest.mark.parametrize("nvec", [1, 5, 32, 35])
def test_fp64_equals_single_runs(ev, kind, nvec):
    mats, ivs, seeds = zip(*requests())
    err, mu, ecnt = ev.kpmdos_batch(list(mats), list(ivs), 33, 1, nvec, kind, seeds, PREC_FP64)
    assert err == 0, ev.last_error()
    for r, (A, iv, seed) in enumerate(requests()):
        assert ev.set_matrix(A) == 0, ev.last_error()
        err, mu1, ecnt1 = ev.kpmdos(33, 1, nvec, iv, vec_kind=kind, seed=seed)
        assert err == 0, ev.last_error()
        assert np.array_equal(mu[r], mu1) and ecnt[r] == ecnt1


@pytest.mark.parametrize("nvec", [3, 32, 40])
def test_mixed_equals_each_request_alone(ev, nvec):
    mats, ivs, seeds = zip(*requests())
    err, mu, ecnt = ev.kpmdos_batch(list(mats), list(ivs), 32, 1, nvec, VEC_GAUSSIAN, seeds,
                                    PREC_MIXED)
    assert err == 0, ev.last_error()
    for r, (A, iv, seed) in enumerate(requests()):
        err, mu1, ecnt1 = ev.kpmdos_batch([A], [iv], 32, 1, nvec, VEC_GAUSSIAN, [seed], PREC_MIXED)
        assert err == 0, ev.last_error()
        assert np.array_equal(mu[r], mu1[0]) and ecnt[r] == ecnt1[0]
