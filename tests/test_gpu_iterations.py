"""Several forcing iterations of a fixed body with the sums, the correction
and the record in the launches beside them, against launches of their own
(ILBM_IB_FUSED=0): the same bits."""
import numpy as np
import pytest

from ilbmrex_amd import config as cf

pytestmark = pytest.mark.gpu


def _case(dim, loops, storage, near_wall):
    st = cf.STORAGE_NAMES[storage]
    if dim == 2:
        c = cf.cylinder_2d(nx=150, ny=64, D=9.0, xc=40.0, yc=8.0 if near_wall else 31.3, storage=st)
    else:
        c = cf.sphere_3d(nx=70, ny=34, nz=36, D=8.0, center=(20.0, 7.0 if near_wall else 17.2, 18.0), storage=st)
    return c.replace(loop_ns=loops)


def _level(c):
    from ilbmrex_amd.native import Level
    with Level(c, cf.uniform_init(c, u=(c.U0, 0.0, 0.0))) as lev:
        lev.advance(4)
        lev.advance(3, want_state=True)
        return (lev.f(), lev.macro(), *lev.markers(), lev.force_history(), lev.mass_history())


@pytest.mark.parametrize("storage", ["f64", "f32", "f16s"])
@pytest.mark.parametrize("near_wall", [False, True])
@pytest.mark.parametrize("loops", [2, 3])
@pytest.mark.parametrize("dim,overlap", [(2, False), (3, False), (3, True)])
def test_level(monkeypatch, dim, overlap, loops, near_wall, storage):
    c = _case(dim, loops, storage, near_wall)
    print(f"[iterations] {c.name} {dim}D loops={loops} wall={near_wall} overlap={overlap} {storage}", flush=True)
    monkeypatch.setenv("ILBM_BODY_TILES", "0")
    if overlap:
        monkeypatch.setenv("ILBM_OVERLAP_BYTES", "0")
    one = _level(c)
    monkeypatch.setenv("ILBM_IB_FUSED", "0")
    two = _level(c)
    assert all(np.array_equal(a, b) for a, b in zip(one, two))


@pytest.mark.parametrize("loops", [1, 2])
@pytest.mark.parametrize("dim", [2, 3])
def test_boxes(monkeypatch, dim, loops):
    from ilbmrex_amd.boxpath import BoxLevel
    c = _case(dim, loops, "f64", False)

    def run():
        b = BoxLevel(c, cf.uniform_init(c, u=(c.U0, 0.0, 0.0)))
        b.advance(4)
        return [b.f(), b.macro(), b.forcing(), np.array(b.record)]
    print(f"[iterations] boxes {dim}D loops={loops}", flush=True)
    one = run()
    monkeypatch.setenv("ILBM_IB_FUSED", "0")
    two = run()
    assert all(np.array_equal(a, b) for a, b in zip(one, two))


@pytest.mark.parametrize("storage", ["f64", "f32"])
def test_refined(monkeypatch, storage):
    from ilbmrex_amd.native import AmrHierarchy
    c = cf.cylinder_2d(nx=64, ny=48, D=8.0, xc=20.0, yc=24.0, U=0.05, Re=40.0,
                       storage=cf.STORAGE_NAMES[storage]).replace(loop_ns=2)

    def run():
        h = AmrHierarchy(c, [((24, 28, 0), (71, 67, 0))], 2, (1.0, c.U0, 0.0, 0.0))
        h.advance(5, want_state=True)
        return [h.f(1), h.macro(0), h.force_history(), h.mass_history()]
    print(f"[iterations] refined {storage}", flush=True)
    one = run()
    monkeypatch.setenv("ILBM_IB_FUSED", "0")
    two = run()
    assert all(np.array_equal(a, b) for a, b in zip(one, two))
