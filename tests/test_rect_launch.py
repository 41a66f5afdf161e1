"""The rectangle launch refuses what it would not run: its callers wait for the
results of a kernel."""
import ctypes as C

from coding_reliability_amd._lib import lib


def test_empty_rectangle_is_refused():
    launch = lib()._ZN2cr11launch_rectERKNS_10RectLaunchERKNS_3dev12DirectResultEP12ihipStream_ti
    launch.argtypes, launch.restype = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_int], C.c_int
    zeros = (C.c_uint64 * 32)()  # no rows, no columns
    assert launch(zeros, zeros, None, 256) != 0
