"""Large downloads and uploads through pageable memory (page-locked chunks,
several threads) give the bytes that small ones and page-locked memory give:
sizes around a whole number of chunks, and several threads at once."""
import ctypes as C
import threading

import numpy as np
import pytest

import lbm_amd as L
from test_gpu_march import state

pytestmark = pytest.mark.gpu


def box(nr, nc):
    return np.zeros((nc, nr), np.uint8)     # every node wet: every byte moves


# 72 bytes a node: below the threshold, just above it, and 12 MiB chunks' rounds with and without a remainder
@pytest.mark.parametrize("nr,nc", [(64, 64), (255, 343), (256, 342), (512, 1024), (513, 1023), (1001, 997)])
def test_round_trip(nr, nc):
    p = state(np.random.default_rng(nr), nc, nr)
    with L.Lattice(box(nr, nc), storage=L.F64) as lat:
        lat.upload_populations(p)
        assert np.array_equal(lat.populations(), p)
        lat.step(1, L.STEP_MACRO)
        rho, u = lat.macro()
        assert np.allclose(rho, p.sum(0), rtol=1e-14, atol=0)
        r2, u2 = np.empty_like(rho), np.empty_like(u)
        lat.wait(lat.macro_async(r2, u2))
        assert np.array_equal(rho, r2) and np.array_equal(u, u2)


def test_page_locked_memory():
    nr, nc = 700, 300
    ptr = C.c_void_p()
    assert L.lib().lbm_host_alloc(9 * nr * nc * 8, C.byref(ptr)) == 0
    p = np.frombuffer((C.c_double * (9 * nr * nc)).from_address(ptr.value)).reshape(9, nc, nr)
    p[:] = state(np.random.default_rng(1), nc, nr)
    with L.Lattice(box(nr, nc), storage=L.F64) as lat:
        lat.upload_populations(p)
        assert np.array_equal(lat.populations(), p)
    assert L.lib().lbm_host_free(ptr) == 0


def test_threads():
    nr, nc = 400, 500
    states = [state(np.random.default_rng(k), nc, nr) for k in range(4)]
    bad = []

    def work(k):
        with L.Lattice(box(nr, nc), storage=L.F64) as lat:
            for _ in range(4):
                lat.upload_populations(states[k])
                if not np.array_equal(lat.populations(), states[k]):
                    bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


# 24 bytes a node: either side of the size up to which a kernel writes the fields
@pytest.mark.parametrize("nr,nc", [(3, 3), (209, 209), (210, 209), (600, 400)])
def test_fields_into_page_locked_memory(nr, nc):
    n = nr * nc
    ptr = C.c_void_p()
    assert L.lib().lbm_host_alloc(3 * n * 8, C.byref(ptr)) == 0
    buf = np.frombuffer((C.c_double * (3 * n)).from_address(ptr.value))
    with L.Lattice(box(nr, nc), storage=L.F64, tau=0.8) as lat:
        lat.upload_populations(state(np.random.default_rng(nr), nc, nr))
        for k in range(3):
            lat.step(2, L.STEP_MACRO)
            rho, u = lat.macro()
            buf[:] = -1.0
            lat.wait(lat.macro_async(buf[:n].reshape(nc, nr), buf[n:].reshape(2, nc, nr)))
            assert np.array_equal(buf[:n].reshape(nc, nr), rho) and np.array_equal(buf[n:].reshape(2, nc, nr), u)
        # either part alone, and one of them in pageable memory
        t = C.c_int64()
        dp = C.POINTER(C.c_double)
        own = np.empty((nc, nr))
        buf[:] = -1.0
        assert L.lib().lbm_download_macro_async(lat._h, None, C.cast(ptr.value + 8 * n, dp), C.byref(t)) == 0
        lat.wait(t.value)
        assert np.array_equal(buf[n:].reshape(2, nc, nr), u) and (buf[:n] == -1.0).all()
        assert L.lib().lbm_download_macro_async(lat._h, own.ctypes.data_as(dp), C.cast(ptr.value + 8 * n, dp),
                                                C.byref(t)) == 0
        lat.wait(t.value)
        assert np.array_equal(own, rho)
    assert L.lib().lbm_host_free(ptr) == 0
