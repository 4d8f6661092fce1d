"""GPU: an infinity or a NaN in R reaches only those entries of R^{-1} that
depend on it (rows up to its own, columns from its own on), as in a column by
column inversion."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -53


@pytest.mark.parametrize("loads", ["", "reg"])
@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("n,i,c", [(64, 5, 40), (100, 3, 70), (128, 40, 90), (129, 63, 128), (300, 17, 250),
                                   (300, 130, 200), (577, 70, 100), (577, 300, 570)])
def test_nonfinite_entry_stays_in_its_rows_and_columns(hip, monkeypatch, n, i, c, value, loads):
    if loads:
        monkeypatch.setenv("CA3DMM_DGEMM_LOADS", loads)
    rnd = np.random.default_rng(n + i + c)
    R = np.triu(rnd.uniform(-1, 1, (n, n)), 1) / n + np.diag(rnd.uniform(1, 2, n))
    want = np.linalg.inv(R)
    R[i, c] = value
    dX = hip.DeviceArray.filled((n, n), 0xFF)
    hip.trtri_upper(n, hip.DeviceArray.from_numpy(R), dX)
    X = dX.numpy()
    hit = np.zeros((n, n), bool)
    hit[:i + 1, c:] = True
    assert np.all(np.isfinite(X[~hit]))
    # kappa(R) is below 4 (the diagonal in [1, 2], the rest at most 1 together)
    assert np.abs(X - want)[~hit].max() <= 64 * (n + 2) * U
    assert not np.any(np.isfinite(X[i, c:]))
    assert np.array_equal(np.tril(X, -1), np.zeros((n, n)))


@pytest.mark.parametrize("n,j", [(100, 70), (129, 20), (300, 299), (577, 100)])
def test_zero_on_the_diagonal_reaches_its_rows_and_columns_only(hip, n, j):
    rnd = np.random.default_rng(n + j)
    R = np.triu(rnd.uniform(-1, 1, (n, n)), 1) / n + np.diag(rnd.uniform(1, 2, n))
    want = np.linalg.inv(R)
    R[j, j] = 0.0
    dX = hip.DeviceArray.filled((n, n), 0xFF)
    hip.trtri_upper(n, hip.DeviceArray.from_numpy(R), dX)
    X = dX.numpy()
    hit = np.zeros((n, n), bool)
    hit[:j + 1, j:] = True
    assert np.abs(X - want)[~hit].max() <= 64 * (n + 2) * U
    assert X[j, j] == np.inf
