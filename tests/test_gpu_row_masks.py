"""GPU: the row-mask form of the fused step kernel (evsl_amd_spmm_row_masks) at
the edges of what it codes: one pair, whole groups of 6 pairs and one more, 8
pairs (one mask byte) and 9 (two), 16 and 17 (not coded); all offsets on one
side of the diagonal; a matrix of its diagonal alone; rows whose columns are not
in ascending order (not coded); row counts that end inside a block.

Bar: the bits of the CSR kernels (pattern codes off when the matrix is set) for
the blocked ChebAv (the block form of SRC/chebpoly.c:519-598) at every width in
FP64 and in the mixed form, and for the FP64 KPM moments
(SRC/spslice.c:29-148)."""
import numpy as np
import pytest

from evsl_amd import matrices as M
from evsl_amd.evsl import PREC_FP64, PREC_MIXED, VEC_RADEMACHER
from evsl_amd.types import HostCsr

pytestmark = pytest.mark.gpu

WIDTHS = (1, 2, 3, 4, 5, 6, 7, 8, 16, 32)


def coded_matrix(n, offsets, seed, shuffled=False):
    """Each row holds a random half of the pairs (offset, value), the diagonal
    always, in ascending or shuffled order."""
    rng = np.random.default_rng(seed)
    vals = {int(o): float(v) for o, v in zip(offsets, rng.uniform(0.2, 1.0, len(offsets)))}
    ia, ja, a = [0], [], []
    for r in range(n):
        cols = [r + o for o in offsets if 0 <= r + o < n and rng.random() < 0.5] + [r]
        cols = rng.permutation(cols) if shuffled else sorted(cols)
        diag = rng.uniform(-1.0, 1.0)
        for c in cols:
            ja.append(int(c))
            a.append(diag if c == r else vals[int(c) - r])
        ia.append(len(ja))
    return HostCsr(n, np.array(ia), np.array(ja), np.array(a))


def both_sides(k):
    step = [1, 3, 17, 40, 113, 250, 399, 611, 900]
    return sorted(([-s for s in step] + step)[:k] if k < 18 else [-s for s in step] + step)


CASES = [("pairs%d" % k, both_sides(k), False, 0 if k > 16 else 1 if k <= 8 else 2)
         for k in (1, 6, 7, 8, 9, 12, 16, 17)]
CASES += [("below", [-1, -2, -5, -9, -31, -64], False, 1),
          ("above", [1, 2, 5, 9, 31, 64], False, 1),
          ("diagonal", [], False, 1), ("shuffled", [-7, -1, 1, 7], True, 0)]


@pytest.mark.parametrize("name,offsets,shuffled,nbytes", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("n", [1, 255, 2049])
def test_row_masks_same_bits(ev, name, offsets, shuffled, nbytes, n):
    A = coded_matrix(n, offsets, seed=n + len(offsets), shuffled=shuffled)
    lo, hi = M.gershgorin(A)
    lo, hi = lo - 0.1, hi + 0.1
    X = np.random.default_rng(5).uniform(-1.0, 1.0, (n, 32))
    pol = ev.default_pol()
    pol.deg = 17
    assert ev.find_pol(np.array([lo + 0.4 * (hi - lo), lo + 0.6 * (hi - lo), lo, hi]), pol) == 0
    out = {}
    try:
        for on in (0, 1):
            ev.set_pattern_codes(on)
            assert ev.set_matrix(A) == 0, ev.last_error()
            for prec in (PREC_FP64, PREC_MIXED):
                for B in WIDTHS:
                    got = ev.lib.evsl_amd_spmm_row_masks(B, prec, 1)
                    if not on:
                        assert got == 0
                    elif n > 1000:
                        assert got == nbytes, (prec, B)
                    err, Y = ev.cheb_av_cols([pol] * B, X[:, :B], prec)
                    assert err == 0, ev.last_error()
                    out[(on, prec, B)] = Y
            for nvec in (1, 2, 4, 8, 16, 32):
                err, mu, cnt = ev.kpmdos(9, 1, nvec, np.array([lo, hi, lo, hi]),
                                         vec_kind=VEC_RADEMACHER, seed=3)
                assert err == 0, ev.last_error()
                out[(on, "kpm", nvec)] = np.append(mu, cnt)
    finally:
        ev.set_pattern_codes(1)
        ev.free_pol(pol)
    for key in [k for k in out if k[0] == 0]:
        assert np.array_equal(out[key], out[(1,) + key[1:]]), (name, key)
