"""Coarse-fine fills and marker kinematics launched with the stream-collide
kernels before them, against launches of their own (ILBM_AMR_RIDE_CELLS=0):
the same bits."""
import numpy as np
import pytest

from ilbmrex_amd import config as cf

pytestmark = pytest.mark.gpu

BOXES = {2: [((24, 28, 0), (71, 67, 0))], 3: [((16, 16, 0), (79, 79, 0)), ((48, 48, 0), (127, 127, 0))]}


def _fields(case, boxes, regrid):
    from ilbmrex_amd.native import AmrHierarchy
    h = AmrHierarchy(case, boxes, 2, (1.0, case.U0, 0.0, 0.0))
    if regrid:
        h.set_regrid(threshold_ratio=(0.85, 0.90, 0.90), blocking_factor=8)
    h.advance(3)
    h.advance(4, want_state=True)
    return [a for l in range(h.nlev) for a in (h.f(l), h.macro(l))] + [h.force_history(), h.mass_history()]


@pytest.mark.parametrize("storage", ["f64", "f32", "f16s"])
@pytest.mark.parametrize("levels,moving,regrid", [(2, False, False), (3, False, True), (2, True, True), (3, True, False),
                                                  (3, True, True)])
def test_fills_with_the_step_before(monkeypatch, levels, moving, regrid, storage):
    st = cf.STORAGE_NAMES[storage]
    if moving:
        c, boxes = cf.pitching_naca_amr(storage=st)
        boxes = boxes[:levels - 1]
    else:
        # 70 wide: level blocks of 128 x 2, refined ones of other shapes
        c = cf.cylinder_2d(nx=70, ny=48, D=8.0, xc=20.0, yc=24.0, U=0.05, Re=40.0, storage=st)
        boxes = BOXES[levels]
    print(f"[ride] {c.name} levels={levels} regrid={regrid} {storage}", flush=True)
    one = _fields(c, boxes, regrid)
    monkeypatch.setenv("ILBM_AMR_RIDE_CELLS", "0")
    two = _fields(c, boxes, regrid)
    assert all(np.array_equal(a, b) for a, b in zip(one, two))
