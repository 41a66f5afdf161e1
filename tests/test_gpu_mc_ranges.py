"""AN Monte Carlo sample ranges: each number of histogram copies (64 ranges share
64 of them), empty ranges among them, against the oracle's prefixes."""
import random

import pytest

import coding_reliability_amd as cra
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = cra.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("count", [2, 3, 4, 5, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("A,n", [(61, 9), (58659, 11), ((1 << 40) + 3, 6)])
def test_ranges_against_prefixes(ctx, A, n, count):
    rnd = random.Random(count)
    bounds = sorted(rnd.randrange(3000) for _ in range(count + 1))
    bounds[1] = bounds[0]  # an empty one
    rows, ms = ctx.an_mc_ranges(A, n, bounds, seed=7)
    for i, row in enumerate(rows):
        lo, hi = (O.an_mc(A, n, m, 7) if m else [0] * 65 for m in (bounds[i], bounds[i + 1]))
        assert row == [b - a for a, b in zip(lo, hi)], i
