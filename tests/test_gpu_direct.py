"""One-launch calls after one that did not come to its end: what that call left in
the context's shared histogram copies, queue heads or tickets is cleared."""
import ctypes as C

import pytest

import coding_reliability_amd as cra
from coding_reliability_amd._lib import check, lib
from oracle import oracle as O

pytestmark = pytest.mark.gpu


class DirectResult(C.Structure):  # cr::dev::DirectResult
    _fields_ = [("copies", C.c_void_p), ("queue", C.c_void_p), ("tickets", C.c_void_p), ("host", C.c_void_p)]


def _begin_and_leave(ctx):
    """Begins a one-launch call, adds to its counters and queue heads as launches
    before a refused one may, and leaves."""
    begin = lib()._ZN2cr13direct_resultEP10cr_contextPNS_3dev12DirectResultE
    begin.argtypes, begin.restype = [C.c_void_p, C.c_void_p], C.c_int
    r = DirectResult()
    check(begin(ctx.handle, C.byref(r)))
    copy = lib().hipMemcpy
    copy.argtypes, copy.restype = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int], C.c_int
    counts = (C.c_uint64 * 64)(*range(1, 65))
    assert lib().hipDeviceSynchronize() == 0
    assert copy(r.copies, counts, C.sizeof(counts), 1) == 0
    assert copy(r.queue, (C.c_uint64 * 1)(3), 8, 1) == 0


def _calls():
    words = [(i * 0x9E3779B97F4A7C15) & 0xFFFFFFFF for i in range(5000)]
    return {
        "short": lambda c: (c.an_pairs_auto(58659, 5000)[0], O.an_pairs_raw(58659, 5000, 30)),
        "sliced": lambda c: (c.an_pairs_auto(58659, 1 << 14)[0], c.an_pairs(58659, 1 << 14)[0]),
        "carry": lambda c: (c.an_pairs_auto(61, 1 << 18)[0], c.an_pairs(61, 1 << 18)[0]),
        "ragged": lambda c: (c.an_pairs_auto(61, 100003)[0], c.an_pairs(61, 100003)[0]),
        "hamming": lambda c: (c.hamming_weights(32, cra.HAM_LIST, words=words)[0], O.hamming_weights_list(32, words)),
        "samples": lambda c: (c.an_mc(61, 12, 100, seed=3)[0], O.an_mc(61, 12, 100, 3)),
        "grid": lambda c: (c.an_grid_ref(1, 20, 100, 0, 61)[0], O.an_grid_ref(1, 20, 100, 0, 61)[0]),
        "rectangle": lambda c: (c.an_grid_ref(2, 20, 100, 100, 61)[0], O.an_grid_ref(2, 20, 100, 100, 61)[0]),
    }


@pytest.mark.parametrize("kind", list(_calls()))
def test_call_after_one_that_ended_early(kind):
    call = _calls()[kind]
    with cra.Context(0) as ctx:
        for _ in range(2):
            _begin_and_leave(ctx)
            got, want = call(ctx)
            n = max(len(got), len(want))
            assert got + [0] * (n - len(got)) == want + [0] * (n - len(want))
