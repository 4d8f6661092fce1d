"""GPU: entries that queue several nested calls leave the sync mode to other
threads: with it on (the default), a call has finished when it returns, also
while another thread is inside such an entry."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_calls_beside_nested_ones_have_finished_when_they_return(hip):
    rt = C.CDLL("libamdhip64.so.7")
    rnd = np.random.default_rng(1)
    R = np.triu(rnd.uniform(-1, 1, (400, 400)), 1) / 400 + np.diag(rnd.uniform(1, 2, 400))
    B = rnd.standard_normal((3000, 400))
    n = 2000
    X = rnd.integers(-3, 4, (n, n)).astype(float)
    want = float(X[-1] @ X[:, -1])
    dX, dC = hip.DeviceArray.from_numpy(X), hip.DeviceArray.zeros((n, n))
    stop = threading.Event()

    def nested():
        dR, dB, dG = (hip.DeviceArray.from_numpy(v) for v in (R, B, R))
        while not stop.is_set():
            hip.trsm_right_upper(3000, 400, 1.0, dR, dB)
            hip.cholesky_qr(3000, 400, hip.DeviceArray.from_numpy(B), dG, variant=2)

    t = threading.Thread(target=nested)
    t.start()
    try:
        for rep in range(1, 101):
            hip.dgemm(0, 0, n, n, n, float(rep), dX, dX, 0.0, dC)
            got = C.c_double(-1.0)                   # the last entry, read on a stream that does not wait for it
            assert rt.hipMemcpy(C.byref(got), C.c_void_p(dC.at(n * n - 1)), C.c_size_t(8), 2) == 0
            assert got.value == rep * want, rep
    finally:
        stop.set()
        t.join()
