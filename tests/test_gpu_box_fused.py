"""The per-box calls that run several stages in one pass against the
separate stage calls (which the oracle tests pin): the same bits on every
cell of the arrays, over boundary kinds, lattices, strides, component counts
and a box inside the domain."""
import ctypes as C

import numpy as np
import pytest

from ilbmrex_amd import config as cf

pytestmark = pytest.mark.gpu

WALL = ((1.0, 0.01, 0.02, 0.03), (0.99, 0.03, -0.01, 0.02), (1.01, -0.02, 0.01, 0.0))
KINDS = {"periodic": None, "channel": (cf.EXT_DIR, cf.FOEXTRAP), "mirror": (cf.USER_2, cf.USER_2),
         "bounce": (cf.USER_1, cf.USER_1), "open": (cf.FOEXTRAP, cf.FOEXTRAP), "mixed": (cf.USER_2, cf.EXT_DIR)}


def _case(lattice, n, kinds):
    per = tuple(int(k == "periodic") for k in kinds) + (1,) * (3 - len(kinds))
    lo = tuple(cf.INT_DIR if KINDS[k] is None else KINDS[k][0] for k in kinds) + (0,) * (3 - len(kinds))
    hi = tuple(cf.INT_DIR if KINDS[k] is None else KINDS[k][1] for k in kinds) + (0,) * (3 - len(kinds))
    return cf.Case(lattice=lattice, n=n, nu=0.03, periodic=per, bc_lo=lo, bc_hi=hi, bc_lo_val=WALL, bc_hi_val=WALL[::-1])


def _cases():
    D2, D3 = cf.D2Q9, cf.D3Q19
    out = [(D2, (70, 9, 1), (a, b)) for a in KINDS for b in KINDS]
    out += [(D3, (11, 5, 7), k) for k in (("channel", "periodic", "periodic"), ("periodic", "mirror", "mirror"),
                                         ("open", "channel", "periodic"), ("bounce", "mixed", "open"),
                                         ("mixed", "bounce", "mirror"), ("open", "open", "open"))]
    out += [(cf.D3Q27, (6, 8, 5), ("periodic", "periodic", "periodic")), (cf.D3Q27, (3, 3, 3), ("channel", "mixed", "open"))]
    return out


class _Box:
    """arrays of one box with random contents"""

    def __init__(self, case, vlo, vhi, pad, seed):
        from ilbmrex_amd import native
        from ilbmrex_amd.boxpath import NG, _Arr
        self.L, self.check = native.load(), native._check
        self.desc = native.to_desc(case)
        self.d = C.byref(self.desc)
        self.q = case.lattice.q
        g = [NG if e < case.dim else 0 for e in range(3)]
        self.lo, self.hi = (C.c_int * 3)(*vlo), (C.c_int * 3)(*vhi)
        rng = np.random.default_rng(seed)
        box = (tuple(vlo[e] - g[e] for e in range(3)), tuple(vhi[e] + g[e] for e in range(3)))
        self.arr = lambda nc: _Arr(nc, box[0], box[1], pad)
        shape = tuple(box[1][e] - box[0][e] + 1 for e in (2, 1, 0))
        w = np.array(case.lattice.w).reshape(-1, 1, 1, 1)
        self.f, self.m, self.F = self.arr(self.q), self.arr(6), self.arr(3)
        self.f.upload(w * (1 + 0.1 * rng.uniform(-1, 1, (self.q,) + shape)))
        m = 0.05 * rng.uniform(-1, 1, (6,) + shape)
        m[0] += 1.0
        self.m.upload(m)
        self.F.upload(1e-3 * rng.uniform(-1, 1, (3,) + shape) * (rng.uniform(0, 1, shape) < 0.7))

    def call(self, name, *a):
        self.check(getattr(self.L, "ilbm_" + name)(*a), name)


def _same(a, b, what):
    x, y = a.download(), b.download()
    assert np.array_equal(x, y), f"{what}: {np.count_nonzero(x != y)} of {x.size} differ"


@pytest.mark.parametrize("pad", [False, True])
@pytest.mark.parametrize("lattice,n,kinds", _cases(), ids=lambda v: getattr(v, "name", None) or str(v))
def test_fill_patch_and_fill_collide_equal_the_stages(lattice, n, kinds, pad):
    case = _case(lattice, n, kinds)
    whole = ((0, 0, 0), tuple(x - 1 for x in n))
    inner = (tuple(1 if e < case.dim else 0 for e in range(3)), tuple(n[e] - 2 if e < case.dim else 0 for e in range(3)))
    print(f"[box] {lattice.name} {n} {kinds} pad={pad}", flush=True)
    for vlo, vhi in (whole, inner):
        b = _Box(case, vlo, vhi, pad, 3)
        d, lo, hi = b.d, b.lo, b.hi
        for src, meso, nc in ((b.f, 1, b.q), (b.m, 0, 6), (b.m, 0, 4)):
            one, ref = b.arr(nc), b.arr(nc)
            b.call("box_setval", one.ref(), 7.0, None)
            b.call("box_copy", src.ref(), ref.ref(), lo, hi, nc, None)
            b.call("box_fill_periodic", d, ref.ref(), lo, hi, None)
            b.call("box_fill_physical", d, ref.ref(), meso, None)
            b.call("box_fill_patch", d, src.ref(), one.ref(), meso, lo, hi, None)
            _same(one, ref, f"fill_patch {nc} components")
        for force in (None, b.F.ref()):
            one, ref, val = b.arr(b.q), b.arr(b.q), b.arr(b.q)
            b.call("box_copy", b.f.ref(), ref.ref(), lo, hi, b.q, None)
            b.call("box_fill_periodic", d, ref.ref(), lo, hi, None)
            b.call("box_fill_physical", d, ref.ref(), 1, None)
            b.call("box_copy", ref.ref(), val.ref(), b_lo(ref), b_hi(ref), b.q, None)
            b.call("box_collide", d, ref.ref(), b.m.ref(), force, lo, hi, None)
            b.call("box_collide", d, val.ref(), b.m.ref(), force, lo, hi, None)
            b.call("box_fill_periodic", d, ref.ref(), lo, hi, None)
            b.call("box_setval", one.ref(), 7.0, None)
            b.call("box_fill_collide", d, b.f.ref(), one.ref(), b.m.ref(), force, 1, lo, hi, None)
            _same(one, ref, "fill_collide")
            # ghosts = 0 leaves the ghost cells as they are
            b.call("box_copy", val.ref(), one.ref(), b_lo(one), b_hi(one), b.q, None)
            b.call("box_copy", b.f.ref(), one.ref(), lo, hi, b.q, None)
            b.call("box_fill_collide", d, b.f.ref(), one.ref(), b.m.ref(), force, 0, lo, hi, None)
            _same(one, val, "fill_collide without ghosts")


def b_lo(a):
    return (C.c_int * 3)(*a.lo)


def b_hi(a):
    return (C.c_int * 3)(*a.hi)


@pytest.mark.parametrize("pad", [False, True])
def test_cf_fill_patch_and_sums_equal_the_stages(pad):
    case = _case(cf.D3Q19, (16, 18, 20), ("channel", "periodic", "periodic"))
    fine = case.replace(n=(32, 36, 40), dx=(0.5, 0.5, 0.5))
    c0, c1 = _Box(case, (0, 0, 0), (15, 17, 19), pad, 1), _Box(case, (0, 0, 0), (15, 17, 19), pad, 2)
    b = _Box(fine, (8, 10, 12), (21, 25, 29), pad, 3)
    d, lo, hi = b.d, b.lo, b.hi
    for nc in (4, 6):
        f1, f2, m1, m2 = b.arr(b.q), b.arr(b.q), b.arr(nc), b.arr(nc)
        b.call("box_copy", b.m.ref(), m2.ref(), lo, hi, nc, None)
        b.call("box_cf_fill", d, c0.m.ref(), c1.m.ref(), 0.0, 1.0, 0.5, f2.ref(), m2.ref(), nc, lo, hi, None)
        b.call("box_cf_fill_patch", d, c0.m.ref(), c1.m.ref(), 0.0, 1.0, 0.5, f1.ref(), m1.ref(), b.m.ref(), nc, lo, hi,
               None)
        _same(f1, f2, "f")
        _same(m1, m2, "macros")
    from ilbmrex_amd import native
    n = C.c_int64(0)
    b.call("box_sums_workspace", lo, hi, 3, C.byref(n))
    work = native.DeviceArray((n.value // 8,))
    got, one = (C.c_double * 3)(), C.c_double(0.0)
    b.call("box_sums", b.F.ref(), 0, 3, lo, hi, work.ptr, n.value, got, None)
    for k in range(3):
        b.call("box_sum", b.F.ref(), k, lo, hi, C.byref(one), None)
        assert got[k] == one.value
    # too small a workspace, components out of range
    assert b.L.ilbm_box_sums(b.F.ref(), 0, 3, lo, hi, work.ptr, n.value - 8, got, None) != 0
    assert b.L.ilbm_box_sums(b.F.ref(), 1, 3, lo, hi, work.ptr, n.value, got, None) != 0
