"""CPU: the addresses and index maps of the direct-to-LDS tiles as the kernels
form them (dgemm_tile.h, dgemm.hip, gram.hip, solve.hip), for every tile width
and number of waves in use, restated in plain Python: each read lies inside the
operand, the LDS slot that an MFMA reads for (k, x) holds the element whose
product the epilogue stores for (k, x), and every tile and k range is taken
once."""
import pytest

BK = 16
# (W, waves) of Tile128w8 / Tile128e, Tile64, Tile32, Tile128
SHAPES = [(128, 8), (64, 8), (32, 4), (128, 4)]
EDGES = [1, 2, 3, 8, 9, 15, 16, 17, 31, 32, 33, 47, 63, 64, 65, 104, 113, 127, 128]


def dtl_index(xc, W, k, x):
    if xc:
        return k * W + 2 * ((x >> 1) ^ ((k & 1) << 3)) + (x & 1)
    return x * 16 + 2 * ((k >> 1) ^ ((x >> 1) & 7)) + (k & 1)


def dtl_shift(xc, xn):
    """The x whose products come out one further on, -2 for none."""
    return xn - 1 if xc and xn & 1 else -2


def stored_x(xc, W, xn):
    """The epilogue's map: slot x of the tile -> the x it stores, None for none."""
    s = dtl_shift(xc, xn)
    out = []
    for x in range(W):
        y = x - (x == s + 1)
        out.append(y if x != s and y < xn else None)
    assert sorted(y for y in out if y is not None) == list(range(xn))
    return out


def dtl_stage(xc, W, waves, ld, x0, xn, k0):
    """DtlLoader<xc, 4, W, waves>::init and issue at k0: {slot: element offset
    from the operand's origin}."""
    out = {}
    NB, RPB = W // (8 * waves), 128 // W
    for w in range(waves):
        for i in range(NB):
            b = NB * w + i
            for lane in range(64):
                if xc:
                    kr = lane // (W // 2)
                    k = RPB * b + kr
                    x = min(2 * ((lane % (W // 2)) ^ ((k & 1) << 3)), xn - 2)
                    back = xn == 1
                    base = x0 - back + RPB * b * ld + k0 * ld
                    off = kr * ld * 8 + 8 * (x + back)
                else:
                    xb, xl = min(8 * b, xn - 1), 8 * b + (lane >> 3)
                    x = min(xl, xn - 1)
                    base = (x0 + xb) * ld + k0
                    off = (x - xb) * ld * 8 + 16 * ((lane & 7) ^ ((xl >> 1) & 7))
                assert 0 <= off < 2 ** 32 and off % 8 == 0
                for h in (0, 1):
                    slot = b * 128 + 2 * lane + h
                    assert slot not in out
                    out[slot] = base + off // 8 + h
    assert len(out) == BK * W
    return out


def stages(kbeg, kend):
    """mainloop_blocks: (k0, lo) of the stages, whose k below lo count as zero."""
    nfull, rem = (kend - kbeg) // BK, (kend - kbeg) % BK
    assert kend >= BK or kbeg == 0
    out = [(min(kbeg + z * BK, kend - BK), 0) for z in range(nfull)]
    if rem:
        out.append((min(kbeg + nfull * BK, kend - BK), BK - rem))
    # each k of the range counts once, in order
    assert [k0 + k for k0, lo in out for k in range(lo, BK)] == list(range(kbeg, kend))
    return out


@pytest.mark.parametrize("W,waves", SHAPES)
@pytest.mark.parametrize("xc", [0, 1])
def test_every_slot_holds_its_element(xc, W, waves):
    for xn in (e for e in EDGES if e <= W):
        for x0 in (0, 3 * W):
            if xc and xn == 1 and x0 == 0:
                continue                              # one row (column) in all: register-staged
            X = x0 + xn
            for K in (16, 29):
                for ld in ((X, X + 1) if xc else (K, K + 1)):
                    last = (K - 1) * ld + X - 1 if xc else (X - 1) * ld + K - 1
                    for k0, lo in stages(0, K):
                        img = dtl_stage(xc, W, waves, ld, x0, xn, k0)
                        assert min(img.values()) >= 0 and max(img.values()) <= last, (xn, x0, K, ld)
                        for x, y in enumerate(stored_x(xc, W, xn)):
                            if y is None:
                                continue
                            for k in range(lo, BK):
                                want = (k0 + k) * ld + x0 + y if xc else (x0 + y) * ld + k0 + k
                                assert img[dtl_index(xc, W, k, x)] == want, (xn, x0, K, k, x)


@pytest.mark.parametrize("W", [128, 64, 32])
@pytest.mark.parametrize("xc", [0, 1])
def test_mfma_reads_are_free_of_bank_conflicts(xc, W):
    for X0 in range(0, W, 16):
        for ks in range(4):
            for half in (0, 32):
                banks = set()
                for lane in range(half, half + 32):
                    w = 2 * dtl_index(xc, W, 4 * ks + (lane >> 4), X0 + (lane & 15))
                    banks |= {w % 64, (w + 1) % 64}
                assert len(banks) == 64, (xc, W, X0, ks)


@pytest.mark.parametrize("n", [65, 66, 79, 80, 81, 97, 127, 129, 193, 200])
def test_join_reads_stay_inside_both_matrices(n):
    """trtri_join_kernel: the last block may be shorter than a stage, which
    then starts before it."""
    ld = n
    last = ld * n - 1
    s = 64
    while s < n:
        for pair in range((n - s + 2 * s - 1) // (2 * s)):
            o = 2 * s * pair
            w = min(s, n - o - s)
            assert w > 0
            x11, x22 = o * ld + o, (o + s) * ld + o + s
            x21, r12 = x11 + s, (o + s) * ld + o
            x12 = x11 + s * ld
            for part in (0, 1, 2):                    # (3 reads what 1 does)
                M, N = (s, w) if part == 1 else (w, s)
                org_a, org_b = ((x22, r12), (x11, x21), (x12, o * ld + o))[part]
                for m0 in range(0, M, 32):
                    for n0 in range(0, N, 32):
                        kbeg, kend = ((0, min(w, m0 + 32)), (m0, s), (n0 + 32, s))[part]
                        mn, nn = min(32, M - m0), min(32, N - n0)
                        for k0, _ in (stages(kbeg, kend) if kend >= BK else [(kend - BK, BK - kend)]):
                            for xc, org, x0, xn in ((part == 1, org_a, m0, mn), (1, org_b, n0, nn)):
                                img = dtl_stage(xc, 32, 4, ld, x0, xn, k0)
                                assert 0 <= org + min(img.values()) and org + max(img.values()) <= last
                        if part == 2:                 # join_triangle: k in [n0, n0 + 32)
                            assert n0 + 32 <= s and nn == 32
                            reads = [org_a + (m0 + min(x, mn - 1)) * ld + n0 + k for x in range(32) for k in range(32)]
                            reads += [org_b + (n0 + k) * ld + n0 + x for x in range(32) for k in range(32)]
                            assert min(reads) >= 0 and max(reads) <= last
        s *= 2


def test_join_triangle_fills_both_stages():
    for xc in (0, 1):
        seen = {}
        for e in range(1024):
            lo, hi = e & 31, e >> 5
            k, x = (hi, lo) if xc else (lo, hi)
            slot = (k >= BK, dtl_index(xc, 32, k % BK, x))
            assert slot not in seen and slot[1] < 512
            seen[slot] = (k, x)
        assert len(seen) == 1024


def tile_coords(t, M, N, W, G):
    tiles_m, tiles_n = -(-M // W), -(-N // W)
    grp = t // (G * tiles_n)
    gsz = min(tiles_m - grp * G, G)
    r = t - grp * G * tiles_n
    return grp * G + r % gsz, r // gsz


@pytest.mark.parametrize("W", [128, 64, 32])
@pytest.mark.parametrize("M,N,K,ksplit", [(1, 1, 16, 1), (600, 600, 12001, 20), (101, 67, 5003, 7), (2501, 503, 40, 1),
                                          (300, 40, 2000, 31)])
def test_locate_takes_every_tile_and_k_once(W, M, N, K, ksplit):
    """dgemm.hip locate, with the ranges of pick_cut."""
    stages_ = -(-K // BK)
    length = -(-stages_ // ksplit)
    ksplit, kstep = -(-stages_ // length), length * BK
    tiles = -(-M // W) * -(-N // W)
    nb = (tiles * ksplit + 7) // 8 * 8
    seen = []
    for b in range(nb):
        t = (b & 7) * (nb >> 3) + (b >> 3)
        if t >= tiles * ksplit:
            continue
        sp = t // tiles
        kbeg = sp * kstep
        kend = K if K - kbeg < kstep else kbeg + kstep
        assert kbeg < kend <= K and (kend >= BK or ksplit == 1)
        seen.append(tile_coords(t - sp * tiles, M, N, W, 16) + (kbeg, kend))
    assert len(set(seen)) == len(seen) == tiles * ksplit
    for i in range(-(-M // W)):
        for j in range(-(-N // W)):
            r = sorted(x[2:] for x in seen if x[:2] == (i, j))
            assert r[0][0] == 0 and r[-1][1] == K and all(a[1] == b[0] for a, b in zip(r, r[1:]))


@pytest.mark.parametrize("W", [128, 64, 32])
@pytest.mark.parametrize("problems", [[(1, 1)], [(130, 77), (65, 77), (130, 1), (1, 300)], [(502, 504), (501, 503)] * 6])
def test_batch_takes_every_tile_once(W, problems):
    bases, total = [], 0
    for M, N in problems:
        bases.append(total)
        total += -(-M // W) * -(-N // W)
    nb = (total + 7) // 8 * 8
    seen = []
    for b in range(nb):
        t = (b & 7) * (nb >> 3) + (b >> 3)
        if t < total:
            p = max(i for i, base in enumerate(bases) if base <= t)
            seen.append((p,) + tile_coords(t - bases[p], *problems[p], W, 16))
    want = [(p, i, j) for p, (M, N) in enumerate(problems) for i in range(-(-M // W)) for j in range(-(-N // W))]
    assert sorted(seen) == want


@pytest.mark.parametrize("nt", [1, 2, 3, 8, 31])
def test_gram_pairs_and_diagonal_tiles(nt):
    """gram.hip pair_of over the strict upper triangle, and the 16 x 16 blocks
    that DiagTile deals to 8 waves."""
    noff = nt * (nt - 1) // 2
    seen = []
    for p in range(noff):
        i, rem = 0, p
        while rem >= nt - 1 - i:
            rem -= nt - 1 - i
            i += 1
        seen.append((i, i + 1 + rem))
    assert sorted(seen) == [(i, j) for i in range(nt) for j in range(i + 1, nt)]
    for nb in (8, 4):
        blocks = nb * (nb + 1) // 2
        got = []
        for wave in range(8):
            for q in range((blocks - wave + 7) // 8):
                p, j = wave + 8 * q, 0
                assert p < blocks
                while (j + 1) * (j + 2) // 2 <= p:
                    j += 1
                got.append((p - j * (j + 1) // 2, j))
        assert sorted(got) == sorted((i, j) for j in range(nb) for i in range(j + 1))


@pytest.mark.parametrize("m,n", [(2, 16), (129, 300), (4097, 257), (20001, 128), (30011, 1999)])
def test_trmm_takes_every_tile_once(m, n):
    tiles_m, tiles_n = -(-m // 128), -(-n // 128)
    per = (tiles_m + 7) // 8
    seen = []
    for b in range(per * 8 * tiles_n):
        first = (b & 7) * per
        rows, e = min(per, tiles_m - first), b >> 3
        if e >= rows * tiles_n:
            continue
        grp = e // (32 * tiles_n)
        r, gsz = e - grp * 32 * tiles_n, min(rows - 32 * grp, 32)
        seen.append((first + 32 * grp + r % gsz, tiles_n - 1 - r // gsz))
    assert sorted(seen) == [(i, j) for i in range(tiles_m) for j in range(tiles_n)]
