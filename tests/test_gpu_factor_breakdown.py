"""GPU: what hip_dpotrf leaves in A when a pivot fails."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -53
NB = 64                                               # rows of a block of the factorization


def _broken(n, k):
    """A symmetric S whose leading k x k part is positive definite and whose
    pivot k is negative, and the factor of the leading part's block rows."""
    rnd = np.random.default_rng(n + 3 * k)
    R = np.triu(rnd.uniform(-1, 1, (n, n)), 1) / n + np.diag(rnd.uniform(1, 2, n))
    S = R.T @ R
    S[k, k] = -1.0
    return S, R


@pytest.mark.parametrize("n,k", [(200, 70), (300, 0), (1000, 130), (2500, 1999), (4000, 64), (257, 256)])
def test_rows_from_the_failing_block_on_are_the_updated_rest(hip, n, k):
    """The block rows before the failing one are the factor's; right of the
    failing block and below it A holds what is left after those rows."""
    S, R = _broken(n, k)
    j0 = k // NB * NB
    d = hip.DeviceArray.from_numpy(S)
    print(f"[breakdown] n={n} k={k}", flush=True)
    assert hip.potrf_upper(n, d) == k + 1
    got = d.numpy()
    tol = 8 * (n + 2) * U * np.abs(S).max()
    up = np.triu(np.ones((n, n), bool))
    assert np.array_equal(got[~up], S[~up])
    # R is the factor of S's rows above j0: only S[k, k] was changed
    assert np.abs((got - R)[:j0][up[:j0]]).max(initial=0.0) <= tol
    rest = S - R[:j0].T @ R[:j0]
    for rows, cols in ((slice(j0, j0 + NB), slice(j0 + NB, n)), (slice(j0 + NB, n), slice(j0 + NB, n))):
        m = up[rows, cols]
        assert np.abs((got - rest)[rows, cols][m]).max(initial=0.0) <= tol


@pytest.mark.parametrize("n,k", [(64, 63), (200, 70), (300, 47), (300, 17), (130, 129), (1000, 150), (90, 64)])
def test_rows_before_the_failing_pivot_are_factor_rows(hip, n, k):
    """Inside the failing block: rows of the factor before the pivot, and in
    the others the block less those rows, as LAPACK's dpotf2 leaves it."""
    S, R = _broken(n, k)
    j0 = k // NB * NB
    j1 = min(n, j0 + NB)
    d = hip.DeviceArray.from_numpy(S)
    assert hip.potrf_upper(n, d) == k + 1
    got = d.numpy()[j0:j1, j0:j1]
    rest = (S - R[:k].T @ R[:k])[j0:j1, j0:j1]
    want = np.where(np.arange(j0, j1)[:, None] < k, R[j0:j1, j0:j1], rest)
    up = np.triu(np.ones(want.shape, bool))
    assert np.abs((got - want)[up]).max() <= 8 * (n + 2) * U * np.abs(S).max()
