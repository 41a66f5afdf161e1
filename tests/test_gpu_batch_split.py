"""Batches whose codes of 2^k words go to the sliced kernel, or with few pairs to
the pair kernel beside its own codes: each side of the rule against the oracle."""
import pytest

import coding_reliability_amd as cra
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = cra.Context(0)
    yield c
    c.close()


def _check(ctx, codes, rows):
    got, _ = ctx.an_batch(codes, rows_per_lane=rows)
    plan = ctx.batch_plan(codes, rows_per_lane=rows)
    again = [plan.run()[0] for _ in range(2)]
    plan.close()
    assert again == [got, got]
    for (A, N), h in zip(codes, got):
        assert h == O.an_pairs_raw(A, N, len(h)), (A, N)


# planes above the low k bits at both ends of each variant of the sliced kernel
@pytest.mark.parametrize("k", [11, 12, 13])
def test_sliced_codes_alone(ctx, k):
    _check(ctx, [(A, 1 << k) for A in (1, 3, 127, 129, 193, 255, 4095, 4097, 32767, 32769, 58659, 65535, 58659 << 3)], 0)


# the pair kernel's codes just short of and past 48 rows a lane; words just
# within and past 2048 a row, pairs below and past 2.5e7 a row (1e8 at least)
@pytest.mark.parametrize("rows", [2, 4, 8])
@pytest.mark.parametrize("others", [0, 1])
@pytest.mark.parametrize("k,count", [(11, 1), (11, 47), (11, 48), (12, 1), (13, 1), (13, 3), (14, 1)])
def test_both_sides_of_the_rule(ctx, rows, others, k, count):
    codes = [(61 + 2 * i, 48 * rows + others - i) for i in range(3)]
    codes += [(40001 + 2 * i, 1 << k) for i in range(count)]
    codes.insert(1, ((1 << 40) + 3, 40))
    _check(ctx, codes, rows)
