"""The overlapped step in every mode, where the size rules would keep these
levels on one stream or on body tiles, against the single-stream step: the
same populations, macros, marker forces and force records; Sum(Rho) is summed
in another order.  Each run says which path its steps took."""
import numpy as np
import pytest

from ilbmrex_amd import config as cf

pytestmark = pytest.mark.gpu

SWITCHES = ("ILBM_OVERLAP_TWO_REGIONS", "ILBM_FAR_AFTER", "ILBM_FAR_BLOCKS_PER_CU", "ILBM_GHOST_SEPARATE",
            "ILBM_RING_STREAM", "ILBM_STEP_LINEAR", "ILBM_IB_FUSED", "ILBM_XEV_FENCE")


@pytest.fixture(autouse=True)
def _forced(monkeypatch):
    for v in SWITCHES:
        monkeypatch.delenv(v, raising=False)
    monkeypatch.setenv("ILBM_OVERLAP_BYTES", "0")
    monkeypatch.setenv("ILBM_BODY_TILES", "0")


def _run(case, parts, overlap, path):
    from ilbmrex_amd.native import Level
    with Level(case, cf.uniform_init(case, u=(case.U0, 0.0, 0.0))) as lev:
        lev.set_overlap(overlap)
        for n in parts:
            lev.advance(n, want_state=True)
            assert lev.step_path() == path
        return [lev.f(), lev.macro(), *lev.markers(), lev.force_history()], lev.mass_history()


def _compare(case, parts, path="three regions"):
    print(f"[overlap] {case.name} {case.n} {case.lattice.name} {parts} steps, {path}", flush=True)
    got, mass = _run(case, parts, True, path)
    ref, mass0 = _run(case, [sum(parts)], False, "one stream")
    assert all(np.array_equal(a, b) for a, b in zip(got, ref))
    assert len(mass) == len(mass0) == sum(parts)
    np.testing.assert_allclose(mass, mass0, rtol=1e-12)   # of up to 10^6 terms of one sign


def _sphere(storage, lattice=cf.D3Q19, **kw):
    s = dict(nx=128, ny=96, nz=96, D=10.0, center=(48.0, 47.6, 48.3))
    s.update(kw)
    return cf.sphere_3d(**s, storage=cf.STORAGE_NAMES[storage]).replace(lattice=lattice)


@pytest.mark.parametrize("storage", ["f64", "f32"])
def test_cylinder(storage):
    _compare(cf.cylinder_2d(nx=1024, ny=1024, D=24.0, xc=200.0, yc=512.0, storage=cf.STORAGE_NAMES[storage]), [40])


def test_band_across_the_periodic_boundary():
    _compare(cf.cylinder_2d(nx=1024, ny=1024, D=10.0, xc=30.0, yc=2.0, Re=60.0), [20])


def test_sphere_at_the_inflow():
    # the near box is clipped at the face: two regions
    _compare(_sphere("f32", D=8.0, center=(6.0, 48.0, 48.0)), [20], "two regions")


@pytest.mark.parametrize("storage", ["f64", "f16s"])
def test_advance_in_parts(storage):
    _compare(_sphere(storage), [7, 1, 6])


@pytest.mark.parametrize("linear", ["0", "1"])
@pytest.mark.parametrize("mode", [
    {}, {"ILBM_OVERLAP_TWO_REGIONS": "1"}, {"ILBM_FAR_AFTER": "interp"}, {"ILBM_FAR_AFTER": "export"},
    {"ILBM_FAR_BLOCKS_PER_CU": "4"}, {"ILBM_GHOST_SEPARATE": "1"}, {"ILBM_RING_STREAM": "far"},
    {"ILBM_RING_STREAM": "own"}, {"ILBM_RING_STREAM": "own", "ILBM_FAR_AFTER": "interp"}], ids=str)
def test_modes_over_both_halves_of_the_mass_ring(monkeypatch, mode, linear):
    monkeypatch.setenv("ILBM_STEP_LINEAR", linear)   # rows, or linear blocks for the far cells
    for k, v in mode.items():
        monkeypatch.setenv(k, v)
    _compare(_sphere("f32", nx=150, ny=88, nz=82, center=(48.0, 43.6, 41.3)), [70],
             "two regions" if "ILBM_OVERLAP_TWO_REGIONS" in mode else "three regions")


@pytest.mark.parametrize("fused", ["0", "1"])
@pytest.mark.parametrize("near_wall", [False, True])
@pytest.mark.parametrize("lattice,storage,loops", [(cf.D3Q19, "f64", 2), (cf.D3Q19, "f32", 3), (cf.D3Q27, "f16s", 2)],
                         ids=lambda v: getattr(v, "name", str(v)))
def test_several_forcing_iterations(monkeypatch, lattice, storage, loops, near_wall, fused):
    monkeypatch.setenv("ILBM_IB_FUSED", fused)
    c = _sphere(storage, lattice, **(dict(D=8.0, center=(6.0, 48.0, 48.0)) if near_wall else {}))
    _compare(c.replace(loop_ns=loops), [4, 3], "two regions" if near_wall else "three regions")
