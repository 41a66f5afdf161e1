"""GPU parity of the sliced pair kernel (codes of 2^11 words and more, in
batches and single calls) against the pair kernel and the oracle."""
import pytest

import coding_reliability_amd as cra
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = cra.Context(0)
    yield c
    c.close()


# planes above the low k bits at both ends of each variant: 0, 1, 7 | 8, 12 | 13, 15 | 16;
# even multipliers, and one of 17 bits that stays in the pair kernel
AS = [1, 3, 127, 129, 193, 255, 4095, 4097, 32767, 32769, 58659, 65535, 58659 << 3, 65537, (1 << 16) + 3]


@pytest.mark.parametrize("k", [10, 11, 12, 13])
def test_small_codes_against_oracle(ctx, k):
    # one block of 64 words and a few, blocks shared by four workgroups
    got, _ = ctx.an_batch([(A, 1 << k) for A in AS])
    for A, h in zip(AS, got):
        assert h == O.an_pairs_raw(A, 1 << k, len(h)), A


def test_mixed_batch_against_pair_kernel(ctx):
    # sliced and pair-kernel codes in one call, blocks kept whole (many items)
    codes = [(A, 1 << k) for k in (14, 16, 17) for A in AS] + [(A, 1000 + 7 * k) for k in range(3) for A in AS]
    got, _ = ctx.an_batch(codes)
    for (A, N), h in zip(codes, got):
        assert h == ctx.an_pairs(A, N)[0], (A, N)


@pytest.mark.parametrize("A,k", [(58659, 14), (58659, 17), (32767, 18), (65535, 15), (58659 * 2, 16)])
def test_single_calls(ctx, A, k):
    pair, _ = ctx.an_pairs(A, 1 << k)
    for _ in range(3):
        assert ctx.an_pairs_auto(A, 1 << k)[0] == pair
    with pytest.raises(cra.CRError):
        ctx.an_pairs_auto(A, 1 << k, nbins=9)


def test_plan_replays(ctx):
    codes = [(58659, 1 << 15), (61, 1 << 11), (3, 700), (4097, 1 << 13)]
    want = ctx.an_batch(codes)[0]
    plan = ctx.batch_plan(codes)
    for _ in range(3):
        assert plan.run()[0] == want
        ctx.an_pairs_auto(641, 1 << 15)
    plan.close()
