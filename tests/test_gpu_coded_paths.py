"""GPU: the kernels of coded matrices, each as the one that runs: the CSR kernel on
pattern codes (SRC/chebpoly.c:519-598 is what a filter computes) on matrices of too
many pairs for row masks, with 16-bit and 32-bit table offsets, and on row-mask
matrices under a forced layout; the row-mask kernel, one launch a degree, at every
block width with filters of different degrees.

Bar: the bits of the same matrix without codes."""
import numpy as np
import pytest

from evsl_amd import matrices as M
from evsl_amd.evsl import PREC_FP64, PREC_MIXED, VEC_RADEMACHER
from test_gpu_series_tags import POLLS, sym_band

pytestmark = pytest.mark.gpu

WIDTHS = (1, 2, 3, 4, 5, 6, 7, 8, 11, 16, 23, 32, 40)


def filters(ev, A, ncols):
    lo, hi = M.gershgorin(A)
    lo, hi = lo - 0.1, hi + 0.1
    out = []
    for i in range(ncols):
        pol = ev.default_pol()
        pol.deg = (9, 17, 30)[i % 3]
        a = lo + (0.2 + 0.01 * i) * (hi - lo)
        assert ev.find_pol(np.array([a, a + 0.1 * (hi - lo), lo, hi]), pol) == 0
        out.append(pol)
    return out


@pytest.fixture
def launches(ev):
    """Filters one launch a degree."""
    ev.set_series_polls(0)
    yield ev
    ev.set_series_polls(POLLS)
    ev.set_pattern_codes(1)


def both(ev, A, setup, widths):
    """Filters and moments without codes and, after setup(), with them."""
    X = np.random.default_rng(5).uniform(-1.0, 1.0, (A.n, max(widths)))
    pols = filters(ev, A, max(widths))
    lo, hi = M.gershgorin(A)
    out = []
    for on in (0, 1):
        ev.set_pattern_codes(on)
        assert ev.set_matrix(A) == 0, ev.last_error()
        if on:
            setup()
        got = {}
        for prec in (PREC_FP64, PREC_MIXED):
            for B in widths:
                err, got[prec, B] = ev.cheb_av_cols(pols[:B], X[:, :B], prec)
                assert err == 0, ev.last_error()
        err, mu, cnt = ev.kpmdos(40, 1, 8, np.array([lo, hi, lo, hi]), vec_kind=VEC_RADEMACHER,
                                 seed=3)
        assert err == 0, ev.last_error()
        got["moments"] = np.append(mu, cnt)
        out.append(got)
    for p in pols:
        ev.free_pol(p)
    for key in out[0]:
        assert np.array_equal(out[0][key], out[1][key]), key


@pytest.mark.parametrize("far,mode", [(900, 2), (40000, 3)])
def test_pattern_codes_of_many_pairs(launches, far, mode):
    ev = launches
    A = sym_band(90000, [1, 3, 17, 40, 113, 250, 399, 611, far], seed=2)

    def setup():
        assert ev.pattern_codes() == 18
        for B, prec in ((1, PREC_FP64), (1, PREC_MIXED), (2, PREC_MIXED)):
            assert ev.lib.evsl_amd_spmm_row_masks(B, prec, 1) == 0
            assert ev.lib.evsl_amd_spmm_index_mode(B, prec, 1) == mode

    both(ev, A, setup, (1, 2, 3, 4, 8))


@pytest.mark.parametrize("case,mode", [("grid", 2), ("lattice", 3)])
def test_pattern_codes_under_a_forced_layout(launches, case, mode):
    ev = launches
    A = M.laplacian(30, 29, 28) if case == "grid" else M.anderson(40, 16.5, seed=9)

    def setup():
        assert ev.lib.evsl_amd_spmm_row_masks(2, PREC_MIXED, 1) > 0
        assert ev.set_spmm_layout(2, PREC_MIXED, 1, 11) == 0
        assert ev.lib.evsl_amd_spmm_row_masks(2, PREC_MIXED, 1) == 0
        assert ev.lib.evsl_amd_spmm_index_mode(2, PREC_MIXED, 1) == mode

    both(ev, A, setup, (2,))


@pytest.mark.parametrize("case", ["grid", "lattice"])
def test_row_masks_at_every_width(launches, case):
    ev = launches
    A = M.laplacian(16, 17, 18) if case == "grid" else M.anderson(14, 16.5, seed=9)

    def setup():
        for B in (1, 8, 32):
            assert ev.lib.evsl_amd_spmm_row_masks(B, PREC_FP64, 1) > 0

    n0 = ev.series_counts()[0]
    both(ev, A, setup, WIDTHS)
    assert ev.series_counts()[0] == n0
