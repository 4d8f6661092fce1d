"""GPU: the direct-to-LDS DGEMM's workgroup tiles (128, 64 and 32 wide) and
the library's choice among them, at the edges of tiles and of k-stages.

Every tile adds the products of an entry in the order of k, as the register-
staged kernel does, so the tolerance is zero: the same bits on random inputs,
exact sums on integers.  The last k-stage reads some k a second time and
counts them as zero, so a non-finite operand entry there must show up where
the product puts it and nowhere else."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(16, 16, 16), (2, 3, 17), (31, 33, 18), (33, 65, 47), (64, 63, 32), (65, 127, 33), (129, 128, 100),
         (128, 129, 31), (257, 193, 63), (1, 40, 50), (40, 1, 50)]


def _product(hip, monkeypatch, tile, loads, ta, tb, A, B, m, n, k):
    for name, value in (("CA3DMM_DGEMM_TILE", tile), ("CA3DMM_DGEMM_LOADS", loads)):
        monkeypatch.delenv(name, raising=False)
        if value:
            monkeypatch.setenv(name, value)
    dA, dB = hip.DeviceArray.from_numpy(A), hip.DeviceArray.from_numpy(B)
    dC = hip.DeviceArray.filled((m, n), 0xFF)
    hip.dgemm(ta, tb, m, n, k, 1.0, dA, dB, 0.0, dC)
    return dC.numpy()


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("tile", [None, "128x128", "64x64", "32x32"])
def test_tiles_same_bits_as_register_staged(hip, monkeypatch, tile, ta, tb):
    rnd = np.random.default_rng(77 + 2 * ta + tb)
    for m, n, k in SIZES:
        sa, sb = ((k, m) if ta else (m, k)), ((n, k) if tb else (k, n))
        A, B = rnd.uniform(-1, 1, sa), rnd.uniform(-1, 1, sb)
        want = _product(hip, monkeypatch, None, "reg", ta, tb, A, B, m, n, k)
        got = _product(hip, monkeypatch, tile, None, ta, tb, A, B, m, n, k)
        assert np.array_equal(got, want), (tile, m, n, k)
        A, B = rnd.integers(-9, 10, sa).astype(float), rnd.integers(-9, 10, sb).astype(float)
        got = _product(hip, monkeypatch, tile, None, ta, tb, A, B, m, n, k)
        assert np.array_equal(got, (A.T if ta else A) @ (B.T if tb else B)), (tile, m, n, k)


@pytest.mark.parametrize("tile", ["128x128", "64x64", "32x32"])
def test_tail_stage_keeps_nonfinite_entries_in_place(hip, monkeypatch, tile):
    rnd = np.random.default_rng(5)
    m, n, k = 70, 90, 37                       # the last stage starts at k = 21 and reads 21..31 again
    A, B = rnd.uniform(1, 2, (m, k)), rnd.uniform(1, 2, (k, n))
    A[3, 25] = np.inf                          # read twice
    A[4, 36] = np.nan                          # read once
    B[30, 5] = -np.inf                         # read twice
    got = _product(hip, monkeypatch, tile, None, 0, 0, A, B, m, n, k)
    want = _product(hip, monkeypatch, None, "reg", 0, 0, A, B, m, n, k)
    assert np.array_equal(got, want, equal_nan=True)
    finite = np.ones((m, n), bool)
    finite[[3, 4], :] = False
    finite[:, 5] = False
    assert np.array_equal(np.isfinite(got), finite)
    assert np.all(got[3, np.arange(n) != 5] == np.inf) and np.all(np.isnan(got[4]))
