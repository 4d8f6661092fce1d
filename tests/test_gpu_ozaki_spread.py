"""GPU: the sampled spread statistics behind hip_ozaki_choose at the edges of
their k ranges (8 k at a time, up to 128 ranges dealt to 8 XCDs)."""
import numpy as np
import pytest

from oracle import ozaki as Z
from tests.test_gpu_ozaki_choose import _near_boundary

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("k", [1, 7, 8, 9, 65, 1023, 1025, 1033])
def test_choose_at_range_edges(hip, ta, tb, k):
    rnd = np.random.default_rng(k)
    opA, opB = Z.phi_matrix(rnd, (37, k), 3.0), Z.phi_matrix(rnd, (k, 29), 3.0)
    opA[5] = 0.0                                      # an empty line
    opB[:, 3] = 0.0
    dA = hip.DeviceArray.from_numpy(opA.T if ta else opA)
    dB = hip.DeviceArray.from_numpy(opB.T if tb else opB)
    L, Ls = Z.spread(opA, opB)
    assert not _near_boundary(L, Ls, k)
    assert hip.ozaki_choose(ta, tb, 37, 29, k, dA, dB) == Z.counts_from_spread(L, Ls, k)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("m,n,k", [(1024, 1030, 1024), (4097, 1500, 1029), (20011, 9001, 1100)])
def test_choose_with_sorted_samples(hip, ta, tb, m, n, k):
    """Sizes from which the samples are taken in the order of their lines."""
    rnd = np.random.default_rng(m)
    opA, opB = Z.phi_matrix(rnd, (m, k), 1.5), Z.phi_matrix(rnd, (k, n), 1.5)
    dA = hip.DeviceArray.from_numpy(opA.T if ta else opA)
    dB = hip.DeviceArray.from_numpy(opB.T if tb else opB)
    L, Ls = Z.spread(opA, opB)
    assert not _near_boundary(L, Ls, k)
    assert hip.ozaki_choose(ta, tb, m, n, k, dA, dB) == Z.counts_from_spread(L, Ls, k)
