"""GPU: products whose number of columns or length of k nears 2^31: grids of
2^32 threads or more, ends of k ranges beyond the largest int."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

V = np.frombuffer(b"\x3f" * 8)[0]                    # the double of a 0x3f byte fill


def test_two_rows_times_very_many_columns(hip):
    """C = A B of 2 x 2^29 + 40 from 16: 69 GB of B, all entries alike, so that
    an entry of C is the sum of 16 equal products and exact up to its roundings."""
    m, n, k = 2, 2 ** 29 + 40, 16
    dA = hip.DeviceArray.from_numpy(np.array([np.arange(1.0, 17.0), np.full(16, -1.0)]))
    dB = hip.DeviceArray.filled((k, n), 0x3F)
    dC = hip.DeviceArray.filled((m, n), 0xFF)
    print("[wide]", flush=True)
    hip.dgemm(0, 0, m, n, k, 1.0, dA, dB, 0.0, dC)
    dB.free()
    got = dC.numpy()
    want = np.array([136.0, -16.0]) * V
    tol = 16 * 2.0 ** -53 * np.array([136.0, 16.0]) * V
    for i in (0, 1):
        lo, hi = got[i].min(), got[i].max()
        assert want[i] - tol[i] <= lo and hi <= want[i] + tol[i]


@pytest.mark.parametrize("k", [2 ** 31 - 8, 2 ** 31 - 10 ** 6])
def test_k_up_to_the_largest_int(hip, k):
    """C = A B^T of 2 x 2 from k with entries all alike (two operands of 34 GB):
    k equal products, summed in some order."""
    dA = hip.DeviceArray.filled((2, k), 0x3F)
    dB = hip.DeviceArray.filled((2, k), 0x3F)
    dC = hip.DeviceArray.filled((2, 2), 0xFF)
    print("[long]", k, flush=True)
    hip.dgemm(0, 1, 2, 2, k, 1.0, dA, dB, 0.0, dC)
    got = dC.numpy()
    assert np.abs(got / (k * V * V) - 1.0).max() <= k * 2.0 ** -53
