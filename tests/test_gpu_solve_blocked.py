"""GPU: the blocked Cholesky, inverse and right solve at the edges of their
64- and 128-wide blocks, through the direct-to-LDS and the register-staged
forms, with odd leading dimensions."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -53


def _upper(rnd, n):
    """Upper R with kappa of a few units: unit-size diagonal, small rest."""
    return np.triu(rnd.uniform(-1, 1, (n, n)), 1) / max(n, 4) + np.diag(rnd.uniform(1, 2, n))


def _padded(hip, a, ld):
    buf = np.full((ld, a.shape[1]), 7.0, order="F")
    buf[:a.shape[0]] = a
    return hip.DeviceArray.from_numpy(buf)


@pytest.mark.parametrize("loads", ["", "reg"])
@pytest.mark.parametrize("n,pad", [(1, 0), (15, 1), (63, 0), (64, 1), (65, 0), (79, 2), (80, 1), (128, 0), (129, 1),
                                   (193, 0), (320, 3), (577, 0), (1025, 1)])
def test_factor_and_inverse(hip, monkeypatch, n, pad, loads):
    """||R^T R - S|| and ||R X - I|| within c n u of their scale (each entry
    is a sum of at most n products, and kappa(R) is below 4)."""
    if loads:
        monkeypatch.setenv("CA3DMM_DGEMM_LOADS", loads)
    rnd = np.random.default_rng(7 * n + pad)
    R0 = _upper(rnd, n)
    S = R0.T @ R0
    ld = n + pad
    print(f"[solve] n={n} ld={ld} loads={loads or 'default'}", flush=True)
    dS = _padded(hip, S, ld)
    assert hip.potrf_upper(n, dS) == 0
    got = dS.numpy()
    R = np.triu(got[:n])
    assert np.array_equal(np.tril(got[:n], -1), np.tril(S, -1)) and np.all(got[n:] == 7.0)
    assert np.abs(R.T @ R - S).max() <= 8 * (n + 2) * U * np.abs(S).max()
    dX = hip.DeviceArray.filled((ld, n), 0xFF)
    hip.trtri_upper(n, _padded(hip, R0, ld), dX)
    X = dX.numpy()
    assert np.array_equal(np.tril(X[:n], -1), np.zeros((n, n)))
    assert np.all(np.isnan(X[n:]))
    assert np.linalg.norm(R0 @ X[:n] - np.eye(n), 2) <= 64 * (n + 2) * U


@pytest.mark.parametrize("n,k", [(64, 0), (65, 64), (200, 130), (257, 256), (300, 17)])
def test_factor_reports_the_failing_pivot(hip, n, k):
    rnd = np.random.default_rng(n)
    R0 = _upper(rnd, n)
    S = R0.T @ R0
    S[k, k] = -1.0
    dS = _padded(hip, S, n)
    assert hip.potrf_upper(n, dS) == k + 1


def test_inverse_of_extreme_diagonals(hip):
    """Diagonals outside the range of the reciprocal form are divided by: the
    inverse of a diagonal matrix is the rounded reciprocal."""
    d = np.array([1.0, 3.0, 2.0 ** -600, 2.0 ** 600, 5e-308, -7.0, 1e300, 0.1] * 9)
    n = len(d)
    dX = hip.DeviceArray.filled((n, n), 0xFF)
    hip.trtri_upper(n, hip.DeviceArray.from_numpy(np.diag(d)), dX)
    assert np.array_equal(dX.numpy(), np.diag(1.0 / d))


@pytest.mark.parametrize("m,n,pad", [(129, 16, 0), (300, 129, 1), (4097, 257, 0), (1000, 500, 3), (20001, 128, 0)])
def test_orthogonalisation_of_odd_sizes(hip, monkeypatch, m, n, pad):
    """Q = A R^{-1} in one launch agrees with the in-place form (one product
    per column block), and Q R = A; kappa(A) is below 10."""
    rnd = np.random.default_rng(m + n)
    A = rnd.standard_normal((m, n))
    out = []
    for inplace in ("0", "1"):
        monkeypatch.setenv("CA3DMM_CHOLQR_INPLACE", inplace)
        dA, dR = _padded(hip, A, m + pad), hip.DeviceArray.filled((n, n), 0xFF)
        info, passes = hip.cholesky_qr(m, n, dA, dR, variant=2)
        assert info == 0 and passes == 2
        out.append((dA.numpy(), dR.numpy()))
    (Q, R), (Q1, R1) = out
    assert np.abs(Q - Q1).max() <= 1e-13 and np.abs(R - R1).max() <= 1e-13 * np.abs(R1).max()
    assert np.all(Q[m:] == 7.0)
    assert np.linalg.norm(Q[:m] @ R - A) <= 1e-13 * np.linalg.norm(A)
    assert np.linalg.norm(Q[:m].T @ Q[:m] - np.eye(n)) <= 1e-13 * n


@pytest.mark.parametrize("n,at", [(64, 0), (100, 40), (200, 150), (130, 129)])
def test_factor_with_extreme_pivots(hip, n, at):
    """Pivots outside the range of the iterated square root are taken by
    square root and division: a diagonal matrix gives the rounded root."""
    d = np.linspace(0.5, 900.0, n)
    d[at] = 2.0 ** -1001 * 1.7
    d[n // 2] = 2.0 ** 1001 * 1.3
    dS = hip.DeviceArray.from_numpy(np.diag(d))
    assert hip.potrf_upper(n, dS) == 0
    assert np.allclose(np.diag(dS.numpy()), np.sqrt(d), rtol=2 * U, atol=0)
    d[at] = np.nan
    dS = hip.DeviceArray.from_numpy(np.diag(d))
    assert hip.potrf_upper(n, dS) == at + 1
