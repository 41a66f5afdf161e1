"""Codes of any word count by the recursion over carries: aligned blocks and a tail
restated with Python integers against the oracle (CPU), the kernels against the
pair kernel (GPU)."""
import pytest

from oracle import oracle as O


def ragged_ordered(A, N, T):
    """Ordered-pair distances of A*i, i < N, A odd, blocks of 2^T words and more."""
    bits = (A * (N - 1)).bit_length() + 1
    out = [0] * (bits + 1)
    F = {(0, 0): {0: 1}}
    for m in range(N.bit_length()):
        if m >= T and N >> m & 1:
            last = (N >> m) - 1
            for (c, cc), f in F.items():
                for s in range(last + 1):
                    e = ((c + A * s) ^ (cc + A * last)).bit_count()
                    for d, n in f.items():
                        out[d + e] += n * (1 if s == last else 2)
        G = {}
        for (c, cc), f in F.items():
            for b in (0, 1):
                for bb in (0, 1):
                    v, w = c + A * b, cc + A * bb
                    g = G.setdefault((v >> 1, w >> 1), {})
                    for d, n in f.items():
                        g[d + ((v ^ w) & 1)] = g.get(d + ((v ^ w) & 1), 0) + n
        F = G
    tail = range(N - (N & ((1 << T) - 1)), N)
    for j in tail:
        for i in range(N):
            out[(A * i ^ A * j).bit_count()] += 1 if i in tail else 2
    return out


@pytest.mark.parametrize("A,N,T", [(1, 13, 1), (3, 37, 2), (5, 64, 3), (7, 101, 3), (11, 75, 4)])
def test_blocks_and_tail_equal_pair_counts(A, N, T):
    got, raw = ragged_ordered(A, N, T), O.an_pairs_raw(A, N, 65)
    assert got[0] == N
    assert [x // 2 for x in got[1:]] == raw[1:len(got)] and not any(raw[len(got):])


@pytest.mark.gpu
@pytest.mark.parametrize("A", [1, 3, 31, 33, 61, 62, 127, 129, 255, 511, 61 * 16])
@pytest.mark.parametrize("N", [65535, 65537, 3 << 15, 100003, 131071, (1 << 18) - 128, (1 << 18) + 127, 262145])
def test_ragged_matches_pair_kernel(A, N):
    # no tail and the longest, one 1 bit above it and all, even multipliers
    import coding_reliability_amd as cra
    with cra.Context(0) as ctx:
        auto, ms = ctx.an_pairs_auto(A, N)
        pair, _ = ctx.an_pairs(A, N)
    assert auto == pair and ms > 0


@pytest.mark.gpu
@pytest.mark.parametrize("A,N", [(61, (1 << 20) + 1), (1021, (1 << 20) - 1), (1023, 1 << 20 | 3), (509, (1 << 21) - 1),
                                 (1, (1 << 21) - 1), (1025, (1 << 19) + 1), (61, (1 << 21) + 1)])
def test_largest_ragged_codes(A, N):
    # both sides of the largest multiplier and the largest word count
    import coding_reliability_amd as cra
    with cra.Context(0) as ctx:
        auto, _ = ctx.an_pairs_auto(A, N, nbins=40)
        pair, _ = ctx.an_pairs(A, N, nbins=40)
        with pytest.raises(cra.CRError):
            ctx.an_pairs_auto(A, N, nbins=9)
    assert auto == pair
