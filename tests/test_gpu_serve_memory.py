"""GPU: the device memory that the request loop counts for a density
(evsl_amd_server_stats), by which it admits requests.

Bar: not less than the buffers of its widest column block -- four vector blocks, an
FP64 one for the start vectors, the dots, and the block partials of 16 degrees --
and not more than that and 2 MB for the sums of the partials, and four times the
partials (a narrower block has at most as many)."""
import pytest

from evsl_amd import matrices as M
from evsl_amd.evsl import PREC_FP64, PREC_MIXED, Server

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,size,width,rows", [
    (PREC_FP64, (100, 100, 1), 32, 32),   # 256 rows over 8 lanes of 4 columns
    (PREC_FP64, (68, 68, 68), 16, 64),
    (PREC_FP64, (90, 90, 90), 8, 128),    # 4 lane groups of 2 rows by 2 columns
    (PREC_MIXED, (100, 100, 1), 32, 256)])
@pytest.mark.parametrize("mdeg", [40, 3000])
def test_memory_of_a_density(ev, prec, size, width, rows, mdeg):
    A = M.laplacian(*size)
    lo, hi = M.gershgorin(A)
    srv = Server(ev, 1 << 35, prec)
    mid = srv.add_matrix(A, lo, hi)
    assert srv.submit_dos(mid, lo + 0.1, lo + 1.0, mdeg, 1, 40) >= 0
    assert srv.step() >= 0, ev.last_error()
    used = srv.stats()["mem_peak"]
    srv.close()
    vs = 4 if prec == PREC_MIXED else 8
    part = 16 * -(-A.n // rows) * width * 8
    own = A.n * width * (4 * vs + 8) + (mdeg + 1) * width * 8 + part
    assert own <= used <= own + 3 * part + (2 << 20)
