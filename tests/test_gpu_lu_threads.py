"""GPU: factorisations and solves of several host threads at once, each on a
stream of its own: every result is the one that the call gives alone."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ORDERS = [300, 700, 1030]   # strips of 2, 3 and 5 workgroups in FP64


@pytest.mark.parametrize("entry", ["qpms_hip_zgetrf_dev", "qpms_hip_zgetrf_dev_noalloc", "mixed"])
def test_calls_of_several_threads(gpu, entry):
    import qpms_amd
    L = qpms_amd.lib()
    if entry != "mixed":
        getattr(L, entry).argtypes = [ctypes.c_size_t] + [ctypes.c_void_p] * 3

    def call(n, stream, out):
        rng = np.random.default_rng(n)
        A = np.eye(n) + (rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))) / np.sqrt(8 * n)
        up = qpms_amd.DeviceBuffer.from_array
        dA, dp, db, dx = up(A), up(np.zeros(n, np.int32)), up(np.arange(n) + 1j), up(np.zeros(n, complex))
        for _ in range(5):
            if entry == "mixed":
                it = L.qpms_hip_solve_mixed_dev(n, 1, dA.ptr, db.ptr, dx.ptr, 1e-14, 20, stream)
                out.append((it, dx.to_array(complex, (n,)).tobytes()))
            else:
                dA = up(A)
                info = getattr(L, entry)(n, dA.ptr, dp.ptr, stream)
                out.append((info, dp.to_array(np.int32, (n,)).tobytes(), dA.to_array(complex, (n, n)).tobytes()))

    streams = [ctypes.c_void_p() for _ in ORDERS]
    for s in streams:   # through the HIP runtime that the library is linked with; 1: hipStreamNonBlocking
        assert L.hipStreamCreateWithFlags(ctypes.byref(s), ctypes.c_uint(1)) == 0
    alone, together = [[] for _ in ORDERS], [[] for _ in ORDERS]
    for n, s, o in zip(ORDERS, streams, alone):
        call(n, s, o)
    threads = [threading.Thread(target=call, args=(n, s, o)) for n, s, o in zip(ORDERS, streams, together)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(alone, together):
        assert len(set(a)) == 1 and len(b) == 5 and set(b) == set(a)
    L.qh_stream_release.argtypes = [ctypes.c_void_p]
    for s in streams:
        L.qh_stream_release(s)
        assert L.hipStreamDestroy(s) == 0
