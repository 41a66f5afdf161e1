"""A code whose fastest method finds no device memory for its tables gets the
same histogram from another one."""
import pytest

import coding_reliability_amd as cra

pytestmark = pytest.mark.gpu


def test_carry_tables_that_do_not_fit():
    # A = 4093, 2^18 words: two tables of 1.2 GiB, 0.5 GiB left
    torch = pytest.importorskip("torch")
    A, N = 4093, 1 << 18
    with cra.Context(0) as ctx:
        want, _ = ctx.an_pairs(A, N)
        free, _ = torch.cuda.mem_get_info(0)
        held = torch.empty(free - (1 << 29), dtype=torch.uint8, device="cuda:0")
        try:
            short, _ = ctx.an_pairs_auto(A, N)
        finally:
            del held
            torch.cuda.empty_cache()
        again, _ = ctx.an_pairs_auto(A, N)
    assert short == want and again == want
