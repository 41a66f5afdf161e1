"""Range requests of the Extended Hamming weights by the recursion over data
bits: restated with Python integers against the oracle (CPU), and the kernel
against the oracle, the word lists' kernel and the MacWilliams closed form (GPU)."""
import random

import numpy as np
import pytest

import coding_reliability_amd as cra
from oracle import oracle as O


@pytest.mark.parametrize("k,lo,hi", [(1, 0, 2), (1, 1, 2), (5, 3, 29), (8, 0, 256), (11, 1, 2048), (16, 12345, 54321)])
def test_recursion_gives_the_weights(k, lo, hi):
    # whole extended codewords here: the bits of S are the codeword of a data bit
    S = [O.hamming_codeword_ext(1 << i, k) for i in range(k)]
    size, L = 1 << k, {}
    ends = [(lo, -1), (hi % size, 1)]
    if hi >= size:
        L[0] = 1
    for t in reversed(range(k)):
        nxt = {}
        for s, n in L.items():
            for x in (s, s ^ S[t]):
                nxt[x] = nxt.get(x, 0) + n
        for v, sign in ends:
            if v >> t & 1:  # the words below v that leave it at bit t
                x = 0
                for i in range(t + 1, k):
                    x ^= S[i] if v >> i & 1 else 0
                nxt[x] = nxt.get(x, 0) + sign
        L = nxt
    want = O.hamming_weights(k, lo, hi)
    ext = [0] * (len(want) + 1)
    for w, n in enumerate(want):
        ext[w + (w & 1)] += n
    got = [0] * len(ext)
    for s, n in L.items():
        got[s.bit_count()] += n
    assert got == ext


@pytest.fixture(scope="module")
def ctx():
    c = cra.Context(0)
    yield c
    c.close()


@pytest.mark.gpu
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 11, 12, 26, 27, 31, 32, 33, 57, 58, 63, 64])
def test_ranges_equal_word_lists(ctx, k):
    # any first word (also past 2^k), wraps past 2^k, whole turns, one word;
    # widths at both sides of a parity bit more and of 32 bits
    rnd, mask = random.Random(k), (1 << k) - 1
    reqs = []
    for _ in range(12):
        count = rnd.choice([1, 2, 3, 63, 64, 65, 1000, 4096, 40001])
        first = rnd.choice([0, mask, mask // 2, rnd.getrandbits(64), (mask - rnd.randrange(2000)) % (1 << 64)])
        reqs.append((first, count))
    rows, _ = ctx.hamming_weights_batch([dict(k=k, source=cra.HAM_RANGE, first=f, count=n) for f, n in reqs])
    for (first, count), row in zip(reqs, rows):
        words = np.array([(first + i) & mask for i in range(count)], dtype=np.uint64)
        want, _ = ctx.hamming_weights(k, cra.HAM_LIST, words=words)
        got, _ = ctx.hamming_weights(k, cra.HAM_RANGE, first=first, count=count)
        assert got == want and row == want, (first, count)
    words = np.array([i & mask for i in range(100)], dtype=np.uint64)
    assert ctx.hamming_weights(k, count=100)[0] == O.hamming_weights_list(k, words)[:cra.hamming_N(k)]


@pytest.mark.gpu
@pytest.mark.parametrize("k", [8, 32, 33, 40, 48, 57, 63, 64])
def test_whole_codes_and_their_parts(ctx, k):
    # all words of a width: the closed form; two parts of it at an odd place; turns
    full = cra.hamming_sdc_table(k, 2)[1][:cra.hamming_N(k)]
    size, at = 1 << k, (0x9E3779B97F4A7C15 >> (64 - k)) | 1
    a, _ = ctx.hamming_weights(k, count=at)
    b, _ = ctx.hamming_weights(k, first=at, count=size - at)
    assert [x + y for x, y in zip(a, b)] == full
    c, _ = ctx.hamming_weights(k, first=at, count=size - 1)  # all but the word before `at`
    d, _ = ctx.hamming_weights(k, first=at - 1, count=1)
    assert [x + y for x, y in zip(c, d)] == full
    if k < 62:
        assert ctx.hamming_weights(k, first=at, count=3 * size)[0] == [3 * x for x in full]
