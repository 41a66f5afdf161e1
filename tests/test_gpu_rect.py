"""GPU parity of short rectangle launches (grids beyond the recursion over
carries) with the oracle: chunks of 16 columns and their remainders, partial row
blocks, fewer and more waves than work-queue heads, one head and eight."""
import pytest

import coding_reliability_amd as cra
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = cra.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n,m", [(11, 3), (11, 16), (11, 17), (13, 1001), (16, 33), (16, 1024), (18, 301)])
@pytest.mark.parametrize("A", [1029, 65537])
def test_short_1d_grids(ctx, n, m, A):
    if A >> n:
        pytest.skip("multipliers are below 2^n")
    ref, _, _ = O.an_grid_ref(1, n, m, 0, A)
    for _ in range(2):
        hist, ms = ctx.an_grid_ref(1, n, m, 0, A)
        assert hist == ref[:len(hist)] and 0 < ms < 1000


@pytest.mark.parametrize("m1,m2", [(1, 1), (15, 511), (16, 512), (17, 513), (100, 4099), (3000, 65)])
@pytest.mark.parametrize("n,A", [(14, 61), (30, 58659)])
def test_short_2d_grids(ctx, n, A, m1, m2):
    ref, _, _ = O.an_grid_ref(2, n, m1, m2, A)
    for _ in range(2):
        hist, _ = ctx.an_grid_ref(2, n, m1, m2, A)
        assert hist == ref[:len(hist)]
