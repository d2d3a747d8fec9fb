"""GPU: LanDos where the device has room for the basis of two of its runs, but not
of the eight that it would run together.

Bar: the same curve, bit for bit, as with all of the memory."""
import ctypes as C

import numpy as np
import pytest

from evsl_amd import matrices as M

pytestmark = pytest.mark.gpu

GB = 1 << 30


def free_bytes(ev):
    free, total = C.c_size_t(), C.c_size_t()
    assert ev.lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_fewer_runs_where_memory_is_short(ev, libc):
    n, steps, nvec = 60000, 500, 8
    A = M.laplacian(300, 200, 1)
    one = (steps + 1) * n * 8
    iv = np.array([0.5, 3.0, 0.0, 8.0])
    assert ev.set_matrix(A) == 0, ev.last_error()

    def run():
        libc.srand(5)
        err, x, y, cnt = ev.LanDos(nvec, steps, 64, iv)
        assert err == 0, ev.last_error()
        return x, y, cnt

    ref = run()
    held, piece = [], 16 * GB
    try:
        while (room := free_bytes(ev) - 3 * one) > GB // 4 and piece > GB // 16:
            p = ev.lib._evsl_Malloc_device(min(room, piece))
            if p:
                held.append(p)
            else:
                ev.lib.hipGetLastError()
                piece //= 2
        got = run()
    finally:
        for p in held:
            ev.lib._evsl_Free_device(p)
    assert all(np.array_equal(a, b) for a, b in zip(ref, got))
