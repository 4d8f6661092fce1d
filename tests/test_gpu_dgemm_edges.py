"""GPU: products of several rounds of 128 x 128 tiles whose last row and column
of tiles are partly outside C: every count of 16 x 16 blocks of an edge tile,
against the register-staged form bit for bit and exact on integers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("em,en,k", [(1, 80, 37), (16, 64, 16), (33, 17, 52), (48, 96, 33), (63, 113, 40), (79, 1, 31),
                                     (97, 32, 64), (111, 50, 35), (112, 127, 18), (127, 66, 49)])
def test_edge_tiles(hip, monkeypatch, ta, tb, em, en, k):
    m, n = 5120 + em, 3456 + en                       # 41 x 28 tiles: above four rounds of 256 CUs
    rnd = np.random.default_rng(em + 7 * en + ta + 2 * tb)
    A, B = rnd.standard_normal((m, k)), rnd.standard_normal((k, n))
    A[:, ::2] = rnd.integers(-4, 5, A[:, ::2].shape)
    dA, dB = hip.DeviceArray.from_numpy(A.T if ta else A), hip.DeviceArray.from_numpy(B.T if tb else B)
    got, reg = hip.DeviceArray.filled((m, n), 0xFF), hip.DeviceArray.filled((m, n), 0xFF)
    print(f"[edges] {m} x {n} x {k}", flush=True)
    hip.dgemm(ta, tb, m, n, k, 1.0, dA, dB, 0.0, got)
    monkeypatch.setenv("CA3DMM_DGEMM_LOADS", "reg")
    hip.dgemm(ta, tb, m, n, k, 1.0, dA, dB, 0.0, reg)
    C = got.numpy()
    assert np.array_equal(C, reg.numpy())
    # a sum of k rounded products in any order
    assert np.abs(C - A @ B).max() <= 2 * (k + 1) * 2.0 ** -53 * (np.abs(A).max() * np.abs(B).max() * k)
