"""GPU: the backward error of small Cholesky factors of graded matrices, against
the elimination row by row on the CPU."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rows(G):
    """R of G = R^T R, each row divided by its rounded root before it is used."""
    A = np.triu(G).copy()
    for k in range(len(A)):
        A[k, k] = np.sqrt(A[k, k])
        A[k, k + 1:] /= A[k, k]
        A[k + 1:, k + 1:] -= np.triu(np.outer(A[k, k + 1:], A[k, k + 1:]))
    return A


@pytest.mark.parametrize("n", [5, 8, 16, 17, 32, 48])
def test_backward_error(hip, n):
    """rms over 24 matrices of kappa 1e14: 24^-1/2 is 20 %, and a product
    rounded apart from its sum (the CPU's) adds to the CPU's error: the GPU's is
    at most 1.4 of it."""
    got, want = [], []
    for seed in range(24):
        rnd = np.random.default_rng(100 * n + seed)
        V, _ = np.linalg.qr(rnd.standard_normal((n, n)))
        A = (rnd.standard_normal((4 * n, n)) / np.sqrt(4 * n) * np.logspace(0, -7, n)) @ V.T
        G = A.T @ A
        G = (G + G.T) / 2
        d = hip.DeviceArray.from_numpy(G)
        assert hip.potrf_upper(n, d) == 0
        for R, out in ((np.triu(d.numpy()), got), (_rows(G), want)):
            Rl = R.astype(np.longdouble)
            out.append(np.linalg.norm((Rl.T @ Rl - G.astype(np.longdouble)).astype(float)) / np.linalg.norm(G))
    assert np.sqrt(np.mean(np.square(got))) <= 1.4 * np.sqrt(np.mean(np.square(want)))
