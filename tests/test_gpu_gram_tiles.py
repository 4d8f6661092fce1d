"""GPU: the Gram product at the edges of its 64- and 128-wide tiles, diagonal
tiles included: exact on integers, the bits of the register-staged form on
random entries; and the B^T B engine without its copies."""
import numpy as np
import pytest

from tests.simutil import single_engine
from ca3dmm_amd import engine as E

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


@pytest.mark.parametrize("n,k", [(1, 40), (70, 5000), (300, 301), (1000, 12345)])
def test_btb_engine_direct_and_redistributed(hip, monkeypatch, n, k):
    """With and without the redistribution: the same bits, symmetric, exact on integers."""
    rnd = np.random.default_rng(n)
    B = rnd.integers(-4, 5, (k, n)).astype(np.float64)
    dB = hip.DeviceArray.from_numpy(B)
    out = []
    for force in ("0", "1"):
        monkeypatch.setenv("CA3DMM_FORCE_REDIST", force)
        eng = single_engine(n, n, k, 0, 0, btb=True)
        dC = hip.DeviceArray.filled((n, n), 0xFF)
        E.lib.ca3dmm_engine_exec(eng, None, 1, dB.ptr, k, dC.ptr, n)
        out.append(dC.numpy())
        E.lib.ca3dmm_engine_free(E.C.byref(eng))
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], B.T @ B)
