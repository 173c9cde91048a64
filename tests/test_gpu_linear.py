"""The stream-collide kernel in linear blocks against the row tiling (which
the oracle tests pin): the same bits of state and forces on every row width
class, alone, with the force record in the launch, and overlapped."""
import numpy as np
import pytest

from ilbmrex_amd import config as cf

pytestmark = pytest.mark.gpu

CASES = {
    "duct24": cf.square_duct().replace(n=(24, 20, 18)),
    "periodic32": cf.periodic_box(cf.D3Q19, (32, 5, 7), nu=0.04, force=(1e-5, 0.0, 2e-6)),
    "periodic1": cf.periodic_box(cf.D3Q19, (1, 9, 3), nu=0.04),
    "periodic33": cf.periodic_box(cf.D3Q27, (33, 6, 1), nu=0.04),
    "sphere90": cf.sphere_3d(nx=90, ny=40, nz=33, D=9.0, center=(30.0, 20.0, 16.5), Re=40.0),
    "sphere161": cf.sphere_3d(nx=161, ny=33, nz=40, D=9.0, center=(40.0, 16.5, 20.0), Re=40.0, loop_ns=2),
    "sphere64": cf.sphere_3d(nx=64, ny=40, nz=40, D=9.0, center=(25.0, 20.0, 20.0), Re=40.0),
    "overlapped": cf.sphere_3d(nx=150, ny=92, nz=90, D=12.0, center=(50.0, 46.0, 45.0), Re=50.0),
}


def _run(case, n):
    from ilbmrex_amd.native import Level
    m = cf.uniform_init(case, u=(case.bc_lo_val[0][1], 0.0, 0.0))
    m[1:4] += 0.002 * np.random.default_rng(4).uniform(-1.0, 1.0, (3, case.ncells))
    with Level(case, m) as lev:
        lev.advance(n)
        lev.advance(2, want_state=True)
        return {"f": lev.f(), "macro": lev.macro(), "history": lev.force_history()}, lev.mass_history()


@pytest.mark.parametrize("storage", ["f64", "f32", "f16s"])
@pytest.mark.parametrize("name", list(CASES))
def test_linear_blocks_equal_rows(monkeypatch, name, storage):
    case = CASES[name].replace(storage=cf.STORAGE_NAMES[storage])
    print(f"[linear] {name} {storage}", flush=True)
    monkeypatch.setenv("ILBM_OVERLAP_BYTES", "0")
    monkeypatch.setenv("ILBM_STEP_LINEAR", "0")
    ref, mass0 = _run(case, 4)
    monkeypatch.setenv("ILBM_STEP_LINEAR", "1")
    got, mass1 = _run(case, 4)
    for k, v in ref.items():
        assert np.array_equal(got[k], v), k
    assert np.abs(mass1 - mass0).max() <= 1e-13 * mass0[0]   # other block sums
