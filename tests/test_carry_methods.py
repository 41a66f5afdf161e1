"""The recursions over carries at the codes that cr_an_pairs gives them, by name, so
that a change of the estimates shows; and the counters of the tiles, which hold
every sum but one."""
import numpy as np
import pytest

from conftest import pairs_methods

# multiplier and word bits: up to four levels after the table (word bits less those
# of the multiplier and 4), odd and even block edges of 2016 carries
TILES = [(32769, 20), (47001, 20), (16385, 19), (8193, 18), (4097, 17), (2015, 17),  # no level
         (32767, 20), (8193, 19), (4097, 18), (2017, 17),                            # one
         (8191, 19), (4099, 19), (1023, 16),                                         # two
         (4095, 19), (511, 16), (1021, 17), (2017, 18)]                              # three, four
# levels above the last kernel's 2^T > A: odd and even numbers, 32- and 64-bit counters
CARRY = [(1, 15), (1, 16), (3, 14), (31, 14), (31, 15), (33, 14), (63, 15), (127, 16), (129, 15), (192, 17), (255, 18),
         (257, 17), (61, 19), (3, 19), (3, 20)]
BLOCKS = [(61, 65537), (1, 100003), (255, 131071), (511, 524289), (1021, 1048575)]


@pytest.mark.parametrize("method,codes", [("tiles", [(A, 1 << k) for A, k in TILES]),
                                          ("carry", [(A, 1 << k) for A, k in CARRY]), ("blocks", BLOCKS)])
def test_methods_of_the_codes_below(method, codes):
    assert [c for c in codes if pairs_methods(*c)[0] != method] == []


def test_tile_counters_hold_the_sums():
    # the polynomials of levels 4 and 8 sum to 256 and 65536, one more than a byte
    # and a half word hold: no pair of carries c, c' has all pairs i, j < 16 at one
    # distance popcount((c + A*i) ^ (c' + A*j)), for any odd A < 2^16 (nor then
    # those of level 8, whose terms are level 4's).  At one distance all c + A*i
    # would have the parity of c, and all c' + A*j that of c'.
    parity = (np.bitwise_count(np.arange(1 << 20, dtype=np.uint32)) & 1).astype(np.uint8)
    candidates = 0
    for A in range(3, 1 << 16, 2):
        mixed = parity[0:A] ^ parity[A:2 * A]
        for i in range(2, 16):
            mixed |= parity[0:A] ^ parity[i * A:(i + 1) * A]
        c = np.flatnonzero(mixed == 0).astype(np.uint32)
        if len(c) == 0:
            continue
        candidates += len(c)
        a, b = (x.ravel() for x in np.meshgrid(c, c, indexing="ij"))
        distance = np.bitwise_count(a ^ b)
        for i, j in [(0, 1), (1, 0), (1, 1)] + [(i, j) for i in range(16) for j in range(16)]:
            keep = np.bitwise_count((a + A * i) ^ (b + A * j)) == distance
            a, b, distance = a[keep], b[keep], distance[keep]
            if len(a) == 0:
                break
        assert len(a) == 0, A
    assert candidates > 100000  # the parities alone leave some


@pytest.mark.gpu
@pytest.mark.parametrize("A,N", [(A, 1 << k) for A, k in TILES + CARRY] + BLOCKS)
def test_recursions_match_the_pair_kernel(A, N):
    import coding_reliability_amd as cra
    with cra.Context(0) as ctx:
        pair, _ = ctx.an_pairs(A, N)
        for _ in range(2):
            assert ctx.an_pairs_auto(A, N)[0] == pair
