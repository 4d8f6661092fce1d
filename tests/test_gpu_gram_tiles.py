"""GPU: the Gram product at the edges of its 64- and 128-wide tiles, diagonal
tiles included: exact on integers, the bits of the register-staged form on
random entries."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,pad", [(1, 16, 0), (16, 17, 1), (17, 64, 0), (63, 1000, 0), (65, 1031, 1), (127, 513, 0),
                                     (129, 4097, 2), (192, 20000, 0), (385, 9999, 1), (641, 2050, 0), (1100, 700, 1),
                                     (1281, 15, 0), (2050, 333, 0)])
def test_gram_tile_edges(hip, monkeypatch, n, k, pad):
    rnd = np.random.default_rng(n + 3 * k)
    for kind in ("int", "f"):
        A = rnd.integers(-4, 5, (k, n)).astype(np.float64) if kind == "int" else rnd.standard_normal((k, n))
        buf = np.full((k + pad, n), np.nan, order="F")       # padding is not read into any entry
        buf[:k] = A
        dA = hip.DeviceArray.from_numpy(buf)
        got, reg = hip.DeviceArray.filled((n, n), 0xFF), hip.DeviceArray.filled((n, n), 0xFF)
        print(f"[gram] n={n} k={k} {kind}", flush=True)
        hip.gram(n, k, dA, got)
        monkeypatch.setenv("CA3DMM_DGEMM_LOADS", "reg")
        hip.gram(n, k, dA, reg)
        monkeypatch.delenv("CA3DMM_DGEMM_LOADS")
        C = got.numpy()
        assert np.array_equal(C, reg.numpy()) and np.array_equal(C, C.T)
        if kind == "int":
            assert np.array_equal(C, A.T @ A)
