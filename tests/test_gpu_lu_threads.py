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


def test_waiting_launches_of_several_streams(gpu):
    """Four streams at once, strips of 12 and 20 workgroups and solves with as many as
    a slab may have: none is left to one workgroup, and every result is the one of the
    call alone."""
    import qpms_amd
    L, vp, up = qpms_amd.lib(), ctypes.c_void_p, qpms_amd.DeviceBuffer.from_array
    L.qh_getrf_ws_bytes.restype = L.qh_getrs_ws_bytes.restype = ctypes.c_size_t

    def call(n, s, out, reps):
        rng = np.random.default_rng(n)
        A = rng.standard_normal((n, n), np.float32) + 1j * rng.standard_normal((n, n), np.float32)
        A = A.astype(complex)
        A[range(n), range(n)] += 3 * np.sqrt(n)
        dp, dq, di = qpms_amd.DeviceBuffer(4 * n), qpms_amd.DeviceBuffer(4 * n), up(np.zeros(1, np.int32))
        ws = qpms_amd.DeviceBuffer(max(L.qh_getrf_ws_bytes(64, n, 1), L.qh_getrs_ws_bytes(64, n, 1, 1)))
        for _ in range(reps):
            dA, dB = up(A), up(A[:, :1].copy())
            i = ctypes.c_int
            L.qh_getrf_batched_wsla_f64(i(n), i(1), vp(dA.ptr), ctypes.c_long(0), vp(dp.ptr), vp(dq.ptr), vp(di.ptr),
                                        vp(ws.ptr), i(1), s)
            for _ in range(20):
                L.qh_getrs_ws_f64(i(n), i(1), i(1), vp(dA.ptr), ctypes.c_long(0), vp(dq.ptr), vp(dB.ptr),
                                  ctypes.c_long(0), vp(ws.ptr), s)
            assert L.hipStreamSynchronize(s) == 0
            out.append(dB.to_array(complex, (n, 1)).tobytes())

    orders = [3000, 5000, 3000, 5000]
    streams = [ctypes.c_void_p() for _ in orders]
    for s in streams:
        assert L.hipStreamCreateWithFlags(ctypes.byref(s), ctypes.c_uint(1)) == 0
    alone, together = [[] for _ in orders], [[] for _ in orders]
    for n, s, o in zip(orders[:2], streams, alone):
        call(n, s, o, 1)
    before = L.qh_alone_count()
    threads = [threading.Thread(target=call, args=(n, s, o, 3)) for n, s, o in zip(orders, streams, together)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert L.qh_alone_count() == before
    for k, o in enumerate(together):
        assert len(o) == 3 and set(o) == set(alone[k % 2])
    L.qh_stream_release.argtypes = [ctypes.c_void_p]
    for s in streams:
        L.qh_stream_release(s)
        assert L.hipStreamDestroy(s) == 0
