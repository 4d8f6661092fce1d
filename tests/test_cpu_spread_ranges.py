"""CPU: the k ranges of the count choice's statistics (hip_ozaki_choose and
ozaki_spread_kernel), restated in the types the code uses: they cover k without
a gap, stay within the 128 that the workspace is sized for, and no step passes
the largest int, up to k = 2^31 - 1."""
import numpy as np
import pytest

I32 = 2 ** 31


@pytest.mark.parametrize("k", [1, 7, 8, 9, 1000, 1024, 1025, 130000, 131071, 2 ** 23, 2 ** 30 + 1, I32 - 1024, I32 - 129,
                               I32 - 128, I32 - 9, I32 - 1])
def test_ranges(k):
    kstep = (max(8, (k + 127) // 128) + 7) // 8 * 8       # formed in 64 bits
    ranges = (k + kstep - 1) // kstep
    assert kstep < I32 and 1 <= ranges <= 128
    grid = (ranges + 7) // 8 * 8 * 16
    seen = {}
    for b in range(grid):
        e = b >> 3
        r = (e // 16) * 8 + (b & 7)
        first = r * kstep                                 # 64 bits
        if first >= k:
            continue
        k1 = k if k - first < kstep else first + kstep
        assert first < I32 and k1 < I32
        for l in (first, max(first, k1 - 9), k1 - 1, k1):  # the loop's test: k1 - l >= 8
            assert 0 <= k1 - l < I32
        seen.setdefault(r, []).append((e % 16, first, k1))
    assert sorted(seen) == list(range(ranges))
    ends = [seen[r][0][1:] for r in range(ranges)]
    assert ends[0][0] == 0 and ends[-1][1] == k and all(a[1] == b[0] for a, b in zip(ends, ends[1:]))
    assert all(sorted(p[0] for p in v) == list(range(16)) for v in seen.values())
    assert np.prod((4096, 7, ranges)) * 8 <= 30 * 2 ** 20
