"""GPU: products whose k is split over workgroups (a small C from a long k).

The partial sums are added in a fixed order, so integers are exact, two runs
give the same bits, and random inputs stay within k * u * (|A||B|)_ij of the
double-double product, as for any order of summation.  Under stream capture the
product runs unsplit, and calls of several threads share one buffer in turn."""
import ctypes as C
import threading

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
U = 2.0 ** -53

SIZES = [(64, 64, 2000), (30, 500, 2000), (101, 67, 5003), (1, 1, 4001), (128, 128, 20000), (600, 600, 12001)]


def _ints(rnd, m, n, k, ta, tb):
    return (rnd.integers(-9, 10, (k, m) if ta else (m, k)).astype(float),
            rnd.integers(-9, 10, (n, k) if tb else (k, n)).astype(float))


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_split_products(hip, ta, tb):
    rnd = np.random.default_rng(31 + 2 * ta + tb)
    for m, n, k in SIZES:
        A, B = _ints(rnd, m, n, k, ta, tb)
        C0 = rnd.integers(-50, 51, (m + 1, n)).astype(float)
        P = rnd.integers(-50, 51, (m, n)).astype(float)
        dA, dB = hip.DeviceArray.from_numpy(A), hip.DeviceArray.from_numpy(B)
        prod = (A.T if ta else A) @ (B.T if tb else B)
        dC = hip.DeviceArray.from_numpy(C0)
        hip.dgemm(ta, tb, m, n, k, 2.0, dA, dB, -3.0, dC, ldc=m + 1)
        got = dC.numpy()
        assert np.array_equal(got[:m], 2.0 * prod - 3.0 * C0[:m]) and np.array_equal(got[m], C0[m]), (m, n, k)
        dC = hip.DeviceArray.filled((m, n), 0xFF)
        hip.dgemm_fold(ta, tb, m, n, k, 1.0, dA, dB, 0.0, dC, [hip.DeviceArray.from_numpy(P)])
        assert np.array_equal(dC.numpy(), P + prod), (m, n, k)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_split_random_within_bound_and_repeatable(hip, ta, tb):
    m, n, k = 101, 67, 5003
    rnd = np.random.default_rng(41 + 2 * ta + tb)
    A, B = rnd.uniform(-1, 1, (k, m) if ta else (m, k)), rnd.uniform(-1, 1, (n, k) if tb else (k, n))
    dA, dB = hip.DeviceArray.from_numpy(A), hip.DeviceArray.from_numpy(B)
    out = []
    for _ in range(2):
        dC = hip.DeviceArray.filled((m, n), 0xFF)
        hip.dgemm(ta, tb, m, n, k, 1.0, dA, dB, 0.0, dC)
        out.append(dC.numpy())
    assert np.array_equal(out[0], out[1])
    ii, jj = (v.ravel().astype(np.int32) for v in np.indices((m, n)))
    Af, Bf = np.asfortranarray(A), np.asfortranarray(B)
    ref, ab = O.dd_sample(ta, tb, m, n, k, Af, Af.shape[0], Bf, Bf.shape[0], ii, jj)
    assert np.all(np.abs(out[0][ii, jj] - ref) <= k * U * ab)


def test_split_size_under_capture(hip):
    from ca3dmm_amd._lib import lib
    rt = C.CDLL("libamdhip64.so.7")
    m, n, k = 64, 64, 3000
    rnd = np.random.default_rng(3)
    A, B = _ints(rnd, m, n, k, 0, 0)
    dA, dB = hip.DeviceArray.from_numpy(A), hip.DeviceArray.from_numpy(B)
    dC = hip.DeviceArray.zeros((m, n))
    stream = C.c_void_p(lib.hip_proxy_stream())
    graph, gexec = C.c_void_p(), C.c_void_p()
    hip.sync()
    hip.set_sync(False)
    try:
        assert rt.hipStreamBeginCapture(stream, 1) == 0                 # thread-local mode
        hip.dgemm(0, 0, m, n, k, 1.0, dA, dB, 0.0, dC)
        assert rt.hipStreamEndCapture(stream, C.byref(graph)) == 0
        assert rt.hipGraphInstantiate(C.byref(gexec), graph, None, None, C.c_size_t(0)) == 0
        other = hip.DeviceArray.zeros((m, n))
        for rep in range(3):
            dC.upload(np.full((m, n), -1.0))
            hip.dgemm(0, 0, m, n, k, -1.0, dA, dB, 0.0, other)          # an eager (split) call in between
            assert rt.hipGraphLaunch(gexec, stream) == 0
            hip.sync()
            assert np.array_equal(dC.numpy(), A @ B), rep
            assert np.array_equal(other.numpy(), -(A @ B)), rep
    finally:
        hip.set_sync(True)
        if gexec:
            rt.hipGraphExecDestroy(gexec)
        if graph:
            rt.hipGraphDestroy(graph)


def test_split_products_of_two_threads(hip):
    rnd = np.random.default_rng(4)
    wrong = []

    def work(m, n, k, A, B):
        dA, dB = hip.DeviceArray.from_numpy(A), hip.DeviceArray.from_numpy(B)
        dC = hip.DeviceArray.zeros((m, n))
        for rep in range(30):
            hip.dgemm(0, 0, m, n, k, float(rep), dA, dB, 0.0, dC)
            if not np.array_equal(dC.numpy(), rep * (A @ B)):
                wrong.append((m, n, k, rep))

    threads = [threading.Thread(target=work, args=(m, n, k) + _ints(rnd, m, n, k, 0, 0))
               for m, n, k in ((64, 64, 2000), (100, 200, 4000))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
