"""GPU: the register-staged form in its 64- and 32-wide tiles (k below 16, a
single row or column contiguous along m or n, or by request) against the
128-wide one bit for bit, and exact on integers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (31, 33, 15), (32, 32, 3), (65, 1000, 8), (700, 900, 15), (2000, 2001, 12),
                                   (1, 300, 47), (1, 4097, 200), (129, 1, 33), (33, 65, 129), (640, 500, 300)])
def test_staged_tiles(hip, monkeypatch, ta, tb, m, n, k):
    rnd = np.random.default_rng(m + 3 * n + 7 * k + ta + 2 * tb)
    Af, Bf = rnd.standard_normal((m, k)), rnd.standard_normal((k, n))
    Ai, Bi = rnd.integers(-9, 10, (m, k)).astype(float), rnd.integers(-9, 10, (k, n)).astype(float)
    C0 = rnd.integers(-50, 51, (m + 1, n)).astype(float)

    def run(A, B):
        dC = hip.DeviceArray.from_numpy(C0)
        hip.dgemm(ta, tb, m, n, k, 2.0, hip.DeviceArray.from_numpy(A.T if ta else A),
                  hip.DeviceArray.from_numpy(B.T if tb else B), -3.0, dC, ldc=m + 1)
        return dC.numpy()
    monkeypatch.setenv("CA3DMM_DGEMM_LOADS", "reg")
    out = []
    for tile in ("", "128x128", "64x64", "32x32"):
        monkeypatch.setenv("CA3DMM_DGEMM_TILE", tile)
        out.append(run(Af, Bf))
        got = run(Ai, Bi)
        assert np.array_equal(got[:m], 2.0 * (Ai @ Bi) - 3.0 * C0[:m]) and np.array_equal(got[m], C0[m]), tile
    assert all(np.array_equal(o, out[0]) for o in out[1:])
