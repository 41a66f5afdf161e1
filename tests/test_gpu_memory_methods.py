"""cr_an_pairs with less device memory than the tables of its methods take: the
next method in order that needs less."""
import pytest

import coding_reliability_amd as cra
from conftest import pairs_methods

pytestmark = pytest.mark.gpu

MiB = 1 << 20


# words, MiB left, MiB that the methods take and which of them must fail:
#   4097, 2^20     tiles 100, spectrum 256 fail, planes
#   1021, 2^20 - 1 blocks 2 * 159 fail, pairs
#   4033, 2^24     carry 2 * 1551 fail, spectrum 256
#   2047, 2^24     carry: one of two tables of 400 fits, which leaves the spectrum 160 and that table
@pytest.mark.parametrize("A,N,left,methods", [
    (4097, 1 << 20, 64, ["tiles", "spectrum", "planes"]),
    (1021, (1 << 20) - 1, 64, ["blocks", "pairs"]),
    (4033, 1 << 24, 512, ["carry", "spectrum", "planes"]),
    (2047, 1 << 24, 560, ["carry", "spectrum", "planes"]),
])
def test_tables_that_do_not_fit(A, N, left, methods):
    torch = pytest.importorskip("torch")
    assert pairs_methods(A, N) == methods
    with cra.Context(0) as ctx:
        ctx.an_pairs_auto(58659, 256)
        held = [torch.empty(1, dtype=torch.uint8, device="cuda:0")]
        while (more := ctx.device_memory()[0] - left * MiB) > 8 * MiB:
            held.append(torch.empty(more // (2 * MiB) * 2 * MiB, dtype=torch.uint8, device="cuda:0"))
        try:
            assert ctx.device_memory()[0] <= (left + 8) * MiB
            got, _ = ctx.an_pairs_auto(A, N)
            again, _ = ctx.an_pairs_auto(A, N)
        finally:
            del held
            torch.cuda.empty_cache()
        want, _ = ctx.an_pairs_auto(A, N)  # with its tables
        assert got == want and again == want
        if N < 1 << 24:
            assert ctx.an_pairs(A, N)[0] == want


@pytest.mark.parametrize("buffer", ["DeviceBuffer", "HostBuffer"])
def test_refused_allocation_leaves_no_error_behind(buffer):
    # the runtime's last error is what the next launch would report
    import ctypes as C
    from coding_reliability_amd._lib import lib
    with cra.Context(0):
        reserve = getattr(lib(), f"_ZN2cr{len(buffer)}{buffer}7reserveEm")
        reserve.argtypes, reserve.restype = [C.c_void_p, C.c_size_t], C.c_int
        empty = (C.c_uint64 * 2)()  # ptr, bytes
        assert lib().hipGetLastError() == 0
        assert reserve(empty, 1 << 60) == 4 and list(empty) == [0, 0]
        assert lib().hipGetLastError() == 0
