"""The recursion over carries that cr_an_pairs takes for short multipliers:
the identity restated with Python integers against the oracle's pair counts
(CPU), and the kernels against the pair kernel and closed forms (GPU)."""
import math

import pytest

from oracle import oracle as O


def carry_distribution(A, k):
    """Ordered-pair distance distribution of A*i, i < 2^k, A odd, one bit a level."""
    Q = {(c, d): [int(b == (c ^ d).bit_count()) for b in range(A.bit_length() + 1)] for c in range(A) for d in range(A)}
    for _ in range(k):
        nb = len(Q[0, 0]) + 1
        R = {}
        for c in range(A):
            for d in range(A):
                out = [0] * nb
                for i in (0, 1):
                    for j in (0, 1):
                        v, w = c + A * i, d + A * j
                        e = (v ^ w) & 1
                        for b, x in enumerate(Q[v >> 1, w >> 1]):
                            out[b + e] += x
                R[c, d] = out
        Q = R
    return Q[0, 0]


@pytest.mark.parametrize("A,k", [(1, 5), (3, 6), (5, 7), (11, 6), (13, 8)])
def test_recursion_equals_pair_counts(A, k):
    got = carry_distribution(A, k)
    raw = O.an_pairs_raw(A, 1 << k, 65)
    assert got[0] == 1 << k
    assert [x // 2 for x in got[1:]] == raw[1:len(got)] and not any(raw[len(got):])


@pytest.mark.gpu
@pytest.mark.parametrize("A", [1, 3, 31, 33, 63, 127, 12 * 16, 255, 257, 511, 769])
@pytest.mark.parametrize("k", [13, 14, 15, 17, 18])
def test_carry_matches_pair_kernel(A, k):
    # multipliers at both ends of a bit length (2^T > A, the largest carry),
    # even ones, odd and even numbers of levels
    import coding_reliability_amd as cra
    with cra.Context(0) as ctx:
        auto, _ = ctx.an_pairs_auto(A, 1 << k)
        pair, _ = ctx.an_pairs(A, 1 << k)
    assert auto == pair


@pytest.mark.gpu
@pytest.mark.parametrize("A,k", [(61, 22), (641, 22), (1021, 23), (2047, 22), (2049, 24), (4095, 24), (61, 26)])
def test_carry_matches_spectrum(A, k):
    # 32-bit counters, then 64-bit ones from level 16 on (A = 61: k - 6 levels)
    import coding_reliability_amd as cra
    with cra.Context(0) as ctx:
        auto, _ = ctx.an_pairs_auto(A, 1 << k)
        spec, _ = ctx.an_pairs_spectral(A, k)
    assert auto == spec


@pytest.mark.gpu
@pytest.mark.parametrize("A,k", [(999, 16), (1023, 17), (2015, 18), (2017, 18), (4033, 18), (4095 * 4, 18)])
def test_carry_tiles_match_pair_kernel(A, k):
    # multipliers at the edges of a block of 2016 carries and of its 32-carry
    # tiles, several blocks, no to four levels after the table
    import coding_reliability_amd as cra
    with cra.Context(0) as ctx:
        pair, _ = ctx.an_pairs(A, 1 << k)
        for _ in range(3):
            assert ctx.an_pairs_auto(A, 1 << k)[0] == pair


@pytest.mark.gpu
@pytest.mark.parametrize("A,k", [(2047, 19), (4097, 21), (8191, 22), (8193, 22), (16385, 22), (32767, 23), (4033, 24),
                                 (16385, 24), (65535, 20), (58659, 21), (32769, 23), (58659, 24), (4097, 25)])
def test_carry_tiles_match_spectrum(A, k):
    # 12- to 16-bit multipliers; k - 8 more bits than the multiplier has: up to
    # 32 low parts a carry
    import coding_reliability_amd as cra
    with cra.Context(0) as ctx:
        auto, ms = ctx.an_pairs_auto(A, 1 << k)
        spec, ms_spec = ctx.an_pairs_spectral(A, k)
    print(f"A={A} k={k}: {ms:.1f} ms, spectral path {ms_spec:.1f} ms", flush=True)
    assert auto == spec


@pytest.mark.gpu
@pytest.mark.parametrize("A,k", [(1, 30), (1 << 9, 32), (3, 32), (511, 32)])
def test_carry_longest_words(A, k):
    import coding_reliability_amd as cra
    with cra.Context(0) as ctx:
        raw, ms = ctx.an_pairs_auto(A, 1 << k)
        assert ms < 100
        with pytest.raises(cra.CRError):
            ctx.an_pairs_auto(A, 1 << k, nbins=8)
    assert sum(raw) == (1 << k) * ((1 << k) - 1) // 2
    if A & (A - 1) == 0:
        assert raw[1:k + 1] == [(1 << (k - 1)) * math.comb(k, d) for d in range(1, k + 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("A", [1, 3, 61, 63, 65, 12, 129, 511, 513, 1000 * 2 + 1])
@pytest.mark.parametrize("n,m", [(16, 3), (17, 100), (20, 1001)])
def test_grid_rows_match_oracle(A, n, m):
    # the grid over all 2^n words through the recursion over carries (from
    # about A * n * 80 < 2^n) and, for the longer multipliers, the rectangle kernel
    import coding_reliability_amd as cra
    with cra.Context(0) as ctx:
        hist, _ = ctx.an_grid_ref(1, n, m, 0, A)
    ref, _, _ = O.an_grid_ref(1, n, m, 0, A)
    assert hist[: len(ref)] == ref[: len(hist)] and not any(hist[len(ref):])


@pytest.mark.gpu
@pytest.mark.parametrize("A,n", [(3, 33), (61, 40), (1, 48), (513, 26), (40, 34)])
def test_grid_rows_long_words(A, n):
    # 32- and 64-bit counters beyond what the oracle enumerates: the recursion
    # restated with Python integers on the oracle's sample list
    import coding_reliability_amd as cra
    m = 4
    with cra.Context(0) as ctx:
        hist, _ = ctx.an_grid_ref(1, n, m, 0, A)
    cfg = O.grid_ref_config(A, n, m, 0, 1)
    samples = [int(v) for v in O.grid1d_ref_samples(cfg["A"], n, cfg["step"], 3, cfg["cc"] <= 32)]
    want = [0] * 65
    z = (A & -A).bit_length() - 1
    a = A >> z
    for v in samples:
        below, w = (v & ((1 << z) - 1)).bit_count(), v >> z
        G = [[int(b == (c ^ (w >> n)).bit_count()) for b in range(65)] for c in range(a)]
        for r in range(n):
            bit = w >> (n - 1 - r) & 1
            H = []
            for c in range(a):
                e = (c & 1) ^ bit
                p, q = (G[c >> 1], G[(c + a) >> 1]) if e == 0 else (G[(c + a) >> 1], G[c >> 1])
                H.append([p[b] + (q[b - 1] if b else 0) for b in range(65)])
            G = H
        for b, x in enumerate(G[0]):
            if x:
                want[b + below] += x
    assert hist == want[: len(hist)]
