"""Batches of short items (several work-queue heads) with the number of waves that
the caller asks for: fewer than heads, as many and more, in calls and in plans."""
import ctypes as C

import numpy as np
import pytest

import coding_reliability_amd as cra
from coding_reliability_amd._lib import check, cr_pair_tuning, lib
from oracle import oracle as O

pytestmark = pytest.mark.gpu

CODES = [(61 + 2 * i, 700 + i) for i in range(12)] + [((1 << 40) + 3, 500), (58659, 1 << 12)]


@pytest.fixture(scope="module")
def ctx():
    c = cra.Context(0)
    yield c
    c.close()


def _u64p(a):
    return a.ctypes.data_as(C.POINTER(C.c_uint64))


@pytest.mark.parametrize("rows", [0, 2, 8])
@pytest.mark.parametrize("waves", [1, 3, 4, 7, 8, 9, 100])
def test_every_item_is_counted(ctx, waves, rows):
    stride = max(cra.an_bins(A, N) for A, N in CODES)
    want = np.array([O.an_pairs_raw(A, N, stride) for A, N in CODES], dtype=np.uint64)
    tuning = cr_pair_tuning(rows, 0, waves, 0)
    out, ms = np.zeros_like(want), C.c_double(0)
    codes = cra.Context._codes(CODES)
    check(lib().cr_an_batch(ctx.handle, codes, len(CODES), _u64p(out), stride, C.byref(tuning), C.byref(ms)))
    assert (out == want).all()
    plan = C.c_void_p()
    check(lib().cr_batch_plan_create(ctx.handle, codes, len(CODES), stride, C.byref(tuning), C.byref(plan)))
    try:
        for _ in range(3):
            out[:] = 0
            check(lib().cr_batch_plan_run(plan, _u64p(out), C.byref(ms)))
            assert (out == want).all()
            ctx.an_pairs_auto(641, 1 << 13)
    finally:
        lib().cr_batch_plan_destroy(plan)
