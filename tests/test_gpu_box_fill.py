"""BoxLevel.fill_patch: the arrays a step starts from, against the separate
stages."""
import numpy as np
import pytest

from ilbmrex_amd import config as cf

pytestmark = pytest.mark.gpu


def test_one_level():
    from ilbmrex_amd.boxpath import BoxLevel
    c = cf.cylinder_2d(nx=40, ny=24, D=6.0, xc=14.0, yc=12.0)
    b = BoxLevel(c, cf.random_init(c, seed=4))
    b.advance(2)
    b.fill_patch(b.t_new)
    for src, dst, meso in ((b.f_old, b.sfS, 1), (b.m_old, b.smS, 0)):
        got = dst.download().copy()
        b._check(b.L.ilbm_box_setval(dst.ref(), 0.0, None), "box_setval")
        b._check(b.L.ilbm_box_copy(src.ref(), dst.ref(), b._lo, b._hi, dst.ncomp, None), "box_copy")
        b._check(b.L.ilbm_box_fill_periodic(b._d, dst.ref(), b._lo, b._hi, None), "box_fill_periodic")
        b._check(b.L.ilbm_box_fill_physical(b._d, dst.ref(), meso, None), "box_fill_physical")
        assert np.array_equal(got, dst.download())
