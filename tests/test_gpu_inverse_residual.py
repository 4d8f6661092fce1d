"""GPU: the inverse of an ill-conditioned triangular R, and a solve with it, have
residuals no larger than those of a back substitution of each column."""
import numpy as np
import pytest
import scipy.linalg as sl

pytestmark = pytest.mark.gpu


def _residuals(R, X, B, Y):
    Rl = R.astype(np.longdouble)
    inv = np.linalg.norm((Rl @ X.astype(np.longdouble) - np.eye(len(R))).astype(float))
    return inv, np.linalg.norm((Y.astype(np.longdouble) @ Rl - B.astype(np.longdouble)).astype(float))


@pytest.mark.parametrize("loads", ["", "reg"])
@pytest.mark.parametrize("n,kappa", [(100, 1e6), (200, 1e5), (300, 1e6), (400, 1e7), (449, 1e4)])
def test_residuals(hip, monkeypatch, n, kappa, loads):
    """Against LAPACK's back substitution and the product with its result; the
    two round differently, which over n^2 (50 n) entries leaves a few percent:
    1.25 of the inverse's, 1.15 of the solve's."""
    if loads:
        monkeypatch.setenv("CA3DMM_DGEMM_LOADS", loads)
    rnd = np.random.default_rng(n)
    V, _ = np.linalg.qr(rnd.standard_normal((n, n)))
    A = (rnd.standard_normal((4 * n, n)) / np.sqrt(4 * n) * np.logspace(0, -np.log10(kappa), n)) @ V.T
    R = sl.cholesky(A.T @ A)
    B = np.asfortranarray(rnd.standard_normal((50, n)) @ R)
    # what R does not hold below its diagonal is not referenced
    dR = hip.DeviceArray.from_numpy(np.triu(R) + np.tril(np.full((n, n), np.nan), -1))
    dX, dB = hip.DeviceArray.filled((n, n), 0xFF), hip.DeviceArray.from_numpy(B)
    hip.trtri_upper(n, dR, dX)
    hip.trsm_right_upper(50, n, 1.0, dR, dB)
    X0 = sl.solve_triangular(R, np.eye(n))
    got, want = _residuals(R, dX.numpy(), B, dB.numpy()), _residuals(R, X0, B, B @ X0)
    assert got[0] <= 1.25 * want[0] and got[1] <= 1.15 * want[1]
