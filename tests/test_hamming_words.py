"""Range requests of few words, alone and beside other requests: word by word in
the launch of those or by the recursion over their bits, the same counts as the
list of the words (GPU)."""
import random

import numpy as np
import pytest

import coding_reliability_amd as cra
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = cra.Context(0)
    yield c
    c.close()


def _words(first, count, k):
    return np.array([(first + i) & ((1 << k) - 1) for i in range(count)], dtype=np.uint64)


@pytest.mark.parametrize("k", [1, 8, 20, 32, 33, 57, 58, 64])
@pytest.mark.parametrize("others", [[32], [64], [64, 20], [64] * 6, [40] * 7 + [20], []])
def test_few_ranges_beside_other_requests(ctx, k, others):
    # one to five ranges (four go word by word), other widths' launches or none,
    # calls that stay below the counters of a small batch and calls that do not
    rnd, mask = random.Random(k * 100 + len(others)), (1 << k) - 1
    more = [dict(k=o, source=cra.HAM_MC, count=1000 + 64 * i, seed=i, stream=1) for i, o in enumerate(others)]
    want_more = [O.hamming_mc(q["k"], q["seed"], 1, 0, q["count"])[:cra.hamming_N(q["k"])] for q in more]
    for n in (1, 2, 4, 5):
        reqs, want = list(more), list(want_more)
        for _ in range(n):
            first = rnd.choice([0, mask, rnd.getrandbits(64), (mask - 100) % (1 << 64), (1 << 64) - 7])
            count = rnd.choice([1, 63, 64, 65, 1025, 5000])
            at = rnd.randrange(len(reqs) + 1)
            reqs.insert(at, dict(k=k, source=cra.HAM_RANGE, first=first, count=count))
            want.insert(at, O.hamming_weights_list(k, _words(first, count, k))[:cra.hamming_N(k)])
        got, _ = ctx.hamming_weights_batch(reqs)
        assert got == want, n


@pytest.mark.parametrize("k,edge", [(32, int(1.25e-6 * 2.5e12)), (58, int(1.25e-6 * 0.9e12)), (64, int(1.25e-6 * 0.9e12))])
def test_both_sides_of_the_rule(ctx, k, edge):
    # the same words in one range on either side of the rule and in two parts
    mc = dict(k=k, source=cra.HAM_MC, count=1024, seed=5, stream=2)
    want_mc = O.hamming_mc(k, 5, 2, 0, 1024)[:cra.hamming_N(k)]
    first = (0x9E3779B97F4A7C15 >> (64 - k)) - 1000
    for count in (edge - 1, edge, edge + 1, 2 * edge):
        half = count // 2 + 1
        parts = [ctx.hamming_weights(k, first=f, count=n)[0] for f, n in ((first, half), (first + half, count - half))]
        want = [a + b for a, b in zip(*parts)]
        assert ctx.hamming_weights(k, first=first, count=count)[0] == want
        got, _ = ctx.hamming_weights_batch([dict(k=k, first=first, count=count), mc])
        assert got == [want, want_mc]
