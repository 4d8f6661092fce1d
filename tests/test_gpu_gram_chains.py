"""GPU: the diagonal of a Gram product (sums of squares, whose rounding errors
grow with the length of the chain they are added in) is as accurate as chains of
equal ranges of all 128-wide tiles over one round of the chip give it, where
the ranges of a workgroup are longer than that and where there are many more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _equal_ranges(n, k, cus=256):
    nt = -(-n // 128)
    split = max(1, min(2 * cus // (nt * (nt + 1) // 2), -(-k // 1024)))
    step = -(-(-(-k // split)) // 16) * 16
    return [(a, min(k, a + step)) for a in range(0, k, step)]


@pytest.mark.parametrize("loads", ["", "reg"])
@pytest.mark.parametrize("n,k", [(1300, 9000), (1000, 40000), (2048, 8192), (512, 100000), (1999, 3001),
                                 (64, 100000), (128, 150000)])
def test_diagonal_errors(hip, monkeypatch, n, k, loads):
    """rms over the n entries, against the same chains added one after the other
    on the CPU; two such rms of one distribution differ by about n^-1/2, so the
    bound is five times that."""
    if loads:
        monkeypatch.setenv("CA3DMM_DGEMM_LOADS", loads)
    rnd = np.random.default_rng(n + k)
    A = np.asfortranarray(rnd.standard_normal((k, n)))
    dC = hip.DeviceArray.zeros((n, n))
    print(f"[chains] {n} from {k}", flush=True)
    hip.gram(n, k, hip.DeviceArray.from_numpy(A), dC)
    got = np.diag(dC.numpy())
    exact, want = np.empty(n), np.empty(n)
    for j in range(n):
        q = A[:, j].astype(np.longdouble) ** 2
        exact[j] = q.sum()
        s = A[:, j] * A[:, j]
        want[j] = np.cumsum([np.cumsum(s[a:b])[-1] for a, b in _equal_ranges(n, k)])[-1]

    def rms(v):
        return np.sqrt(np.mean(((v - exact) / exact) ** 2))
    assert rms(got) <= (1.0 + 5.0 * n ** -0.5) * rms(want)
