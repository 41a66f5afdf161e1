"""GPU parity of the one-launch calls: short codes of any word count and
multiplier against the oracle, the result buffers' state from call to call."""
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


@pytest.mark.parametrize("A", [1, 2, 61, 58659, (1 << 31) + 11, (1 << 40) + 3, 0xFFFFFFFFFF1, 58659 << 4])
@pytest.mark.parametrize("N", [1, 2, 63, 64, 65, 255, 256, 257, 1000, 1025, 2047, 2048, 2049, 4097, 8191, 8192, 8193])
def test_short_codes_against_oracle(ctx, A, N):
    # row blocks of 64 and 256 words and their remainders, one workgroup and
    # several, 32- and 64-bit codewords; 8193 words go to the pair kernel
    if (N - 1) * A >= 1 << 64:
        pytest.skip("codewords exceed 64 bits")
    raw, ms = ctx.an_pairs_auto(A, N)
    assert raw == O.an_pairs_raw(A, N, len(raw))
    assert 0 < ms < 100


def test_widest_codewords(ctx):
    # 65 distances, extra bins the caller asks for stay zero
    for A, N in [((1 << 64) - 1, 2), ((1 << 62) + 7, 4), (0x5555555555555555, 3), ((1 << 51) - 1, 1 << 13)]:
        raw, _ = ctx.an_pairs_auto(A, N, nbins=75)
        assert raw == O.an_pairs_raw(A, N, 65) + [0] * 10
    with pytest.raises(cra.CRError):
        ctx.an_pairs_auto(61, 256, nbins=3)
    with pytest.raises(cra.CRError):
        ctx.an_pairs_auto(0, 256)
    with pytest.raises(cra.CRError):
        ctx.an_pairs_auto((1 << 63) + 1, 4)
    with pytest.raises(cra.CRError):
        ctx.an_pairs_auto(61, 0)


def test_calls_leave_the_buffers_clean(ctx):
    # one-launch calls of every kind and width in random order on one context:
    # each leaves the shared copies, queue head and ticket zero for the next
    rnd = random.Random(11)
    kinds = [lambda: ("an", 58659, 256), lambda: ("an", 61, 5000), lambda: ("an", (1 << 40) + 3, 8000),
             lambda: ("an", 58659, 1 << 14), lambda: ("an", 32767, 1 << 15), lambda: ("an", 61, 1 << 18),
             lambda: ("an", 7, 1 << 20), lambda: ("grid", 61, 20)]
    want = {}
    for _ in range(60):
        kind, A, N = rnd.choice(kinds)()
        if kind == "an":
            got = ctx.an_pairs_auto(A, N)[0]
            ref = lambda: ctx.an_pairs(A, N)[0] if N <= 1 << 18 else ctx.an_pairs_spectral(A, 20)[0]
        else:
            got = ctx.an_grid_ref(1, N, 100, 0, A)[0]
            ref = lambda: O.an_grid_ref(1, N, 100, 0, A)[0]
        if (kind, A, N) not in want:
            want[kind, A, N] = ref()
        w = want[kind, A, N]
        assert got[: len(w)] == w[: len(got)], (kind, A, N)


def test_single_requests_between_short_codes(ctx):
    # one-launch Hamming and sample calls of 1 to 66 bins between one-launch
    # codes: each against the oracle, so a copy or counter left over would show
    for k, count in [(1, 1), (4, 4), (8, 1000), (32, 4096), (33, 12346), (57, 77778), (64, 2)]:
        got, ms = ctx.hamming_weights(k, cra.HAM_MC, count=count, seed=7, stream=k)
        assert got == O.hamming_mc(k, 7, k, 0, count)[:len(got)] and ms > 0
        words = [(i * 0x9E3779B97F4A7C15) & ((1 << k) - 1) for i in range(count)]
        got, _ = ctx.hamming_weights(k, cra.HAM_LIST, words=words)
        assert got == O.hamming_weights_list(k, words)[:len(got)]
        got, _ = ctx.hamming_weights(k, cra.HAM_STRIDE, count=count, stride=0x9E3779B97F4A7C15)
        assert got == O.hamming_weights_list(k, words)[:len(got)]
        got, _ = ctx.an_pairs_auto(61, 256)
        assert got == O.an_pairs_raw(61, 256, len(got))
        n = min(k, 20)
        got, _ = ctx.an_mc(61, n, 33, seed=k)
        assert got == O.an_mc(61, n, 33, k)[:len(got)]


@pytest.mark.parametrize("A", [4097, 58659, 58659 * 4097, (1 << 40) + 1])
@pytest.mark.parametrize("N", [8195, 12289, 16383, 30000, 65535])
def test_longer_short_codes_match_the_pair_kernel(ctx, A, N):
    # every workgroup busy, waves that start and end inside row blocks; the last
    # word count of the short kernel
    assert ctx.an_pairs_auto(A, N)[0] == ctx.an_pairs(A, N)[0]
