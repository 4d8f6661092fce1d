"""GPU: what the tests of integers alone cannot tell about split products: that
a split is taken, that none is under stream capture, and that the
register-staged kernel splits with the same bits; and edge tiles on integers."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _captured(hip, rt, call):
    """call() captured on the library's stream: (number of graph nodes, replay)."""
    from ca3dmm_amd._lib import lib
    stream = C.c_void_p(lib.hip_proxy_stream())
    graph, gexec, nodes = C.c_void_p(), C.c_void_p(), C.c_size_t()
    hip.sync()
    hip.set_sync(False)
    try:
        assert rt.hipStreamBeginCapture(stream, 1) == 0                 # thread-local mode
        call()
        assert rt.hipStreamEndCapture(stream, C.byref(graph)) == 0
    finally:
        hip.set_sync(True)
    assert rt.hipGraphGetNodes(graph, None, C.byref(nodes)) == 0
    assert rt.hipGraphInstantiate(C.byref(gexec), graph, None, None, C.c_size_t(0)) == 0

    def replay():
        assert rt.hipGraphLaunch(gexec, stream) == 0
        hip.sync()

    def done():
        rt.hipGraphExecDestroy(gexec)
        rt.hipGraphDestroy(graph)
    return nodes.value, replay, done


def test_split_is_taken_and_not_under_capture(hip):
    rt = C.CDLL("libamdhip64.so.7")
    m, n, k = 64, 64, 20000
    rnd = np.random.default_rng(6)
    A, B = rnd.standard_normal((m, k)), rnd.standard_normal((k, n))
    dA, dB = hip.DeviceArray.from_numpy(A), hip.DeviceArray.from_numpy(B)
    dC = hip.DeviceArray.zeros((m, n))
    hip.dgemm(0, 0, m, n, k, 1.0, dA, dB, 0.0, dC)                      # the buffer exists
    split = dC.numpy()
    nodes, replay, done = _captured(hip, rt, lambda: hip.dgemm(0, 0, m, n, k, 1.0, dA, dB, 0.0, dC))
    assert nodes == 1                                                   # no second launch
    whole = []
    for _ in range(3):
        dC.upload(np.full((m, n), -1.0))
        replay()
        whole.append(dC.numpy())
        hip.dgemm(0, 0, m, n, k, 1.0, dA, dB, 0.0, dC)                  # eager work in between
        assert np.array_equal(dC.numpy(), split)
    done()
    assert all(np.array_equal(w, whole[0]) for w in whole)
    assert not np.array_equal(whole[0], split)                          # another order of summation
    assert np.abs(whole[0] - split).max() <= 2 * k * 2.0 ** -53 * (np.abs(A) @ np.abs(B)).max()


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k", [(64, 64, 2000), (30, 500, 2001), (101, 67, 5003), (600, 600, 12001)])
def test_register_staged_split_has_the_same_bits(hip, monkeypatch, ta, tb, m, n, k):
    rnd = np.random.default_rng(m + k + 2 * ta + tb)
    dA = hip.DeviceArray.from_numpy(rnd.standard_normal((k, m) if ta else (m, k)))
    dB = hip.DeviceArray.from_numpy(rnd.standard_normal((n, k) if tb else (k, n)))
    out = []
    for loads in ("", "reg"):
        monkeypatch.setenv("CA3DMM_DGEMM_LOADS", loads)
        dC = hip.DeviceArray.filled((m, n), 0xFF)
        hip.dgemm(ta, tb, m, n, k, 1.0, dA, dB, 0.0, dC)
        out.append(dC.numpy())
    assert np.array_equal(*out)


@pytest.mark.parametrize("ta,tb,m,n,k", [(0, 0, 1, 300, 5000), (0, 1, 1, 1, 4001), (0, 1, 77, 1, 9001), (1, 1, 200, 1, 3000)])
def test_split_of_a_single_row_or_column(hip, ta, tb, m, n, k):
    """A row (column) contiguous along m (n) is register-staged."""
    rnd = np.random.default_rng(k)
    A, B = rnd.integers(-9, 10, (m, k)).astype(float), rnd.integers(-9, 10, (k, n)).astype(float)
    dC = hip.DeviceArray.filled((m, n), 0xFF)
    hip.dgemm(ta, tb, m, n, k, 1.0, hip.DeviceArray.from_numpy(A.T if ta else A),
              hip.DeviceArray.from_numpy(B.T if tb else B), 0.0, dC)
    assert np.array_equal(dC.numpy(), A @ B)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("em,en,k", [(1, 80, 37), (63, 113, 40), (127, 1, 16)])
def test_edge_tiles_on_integers(hip, ta, tb, em, en, k):
    m, n = 5120 + em, 3456 + en                       # 41 x 28 tiles: above four rounds of 256 CUs
    rnd = np.random.default_rng(em + en + ta + 2 * tb)
    A, B = rnd.integers(-9, 10, (m, k)).astype(float), rnd.integers(-9, 10, (k, n)).astype(float)
    dC = hip.DeviceArray.filled((m, n), 0xFF)
    hip.dgemm(ta, tb, m, n, k, 1.0, hip.DeviceArray.from_numpy(A.T if ta else A),
              hip.DeviceArray.from_numpy(B.T if tb else B), 0.0, dC)
    assert np.array_equal(dC.numpy(), A @ B)
