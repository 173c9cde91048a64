"""Arguments of the per-box calls that the host refuses before any device
work; the arrays' pointers are never touched."""
import ctypes as C

from ilbmrex_amd import native

INVALID = 1


def _fab(ncomp):
    f = native.Fab()
    f.p = C.c_void_p(0x1000)
    f.lo, f.hi, f.ncomp = native.I3(0, 0, 0), native.I3(7, 7, 7), ncomp
    return f


def test_box_sums_refuses_components_beyond_the_array():
    L = native.load()
    lo, hi = native.I3(0, 0, 0), native.I3(7, 7, 7)
    out = (C.c_double * 64)()
    for comp, ncomp in ((0, 4), (3, 1), (2, 2), (2 ** 31 - 1, 1), (2 ** 31 - 40, 64), (-1, 1), (0, 0)):
        rc = L.ilbm_box_sums(C.byref(_fab(3)), comp, ncomp, lo, hi, C.c_void_p(0x1000), 1 << 20, out, None)
        assert rc == INVALID, (comp, ncomp)


def test_box_sums_workspace_of_any_extent():
    L = native.load()
    n = C.c_int64(0)
    assert L.ilbm_box_sums_workspace(native.I3(-2 ** 31, 0, 0), native.I3(2 ** 31 - 1, 0, 0), 2, C.byref(n)) == 0
    assert n.value == 8 * 2 * (2 ** 32 // 256 + 1)
