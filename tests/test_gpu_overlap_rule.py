"""Which immersed-boundary levels overlap their far cells: on both sides of
every line of the rule, by the population bytes of a step."""
import pytest

from ilbmrex_amd import config as cf

pytestmark = pytest.mark.gpu

Q19, Q27 = cf.D3Q19, cf.D3Q27
# lattice, extents, storage, forcing iterations, overlapped
SPHERES = [
    (Q19, (128, 120, 120), "f32", 1, False), (Q19, (256, 104, 104), "f32", 1, True),        # 280, 421 MB
    (Q19, (192, 104, 104), "f32", 1, False), (Q19, (150, 120, 120), "f32", 1, True),        # blocks of 192: 316, 328
    (Q27, (192, 88, 88), "f32", 1, False), (Q27, (150, 104, 104), "f32", 1, True),          # 321, 350
    (Q19, (128, 96, 96), "f64", 1, False), (Q19, (128, 120, 120), "f64", 1, True),          # 359, 560
    (Q19, (256, 120, 120), "f16s", 1, False), (Q19, (160, 144, 144), "f16s", 1, False),     # 280, linear 252
    (Q19, (192, 104, 104), "f16s", 1, False), (Q19, (192, 144, 144), "f16s", 1, True),      # blocks of 192: 158, 303
    (Q27, (192, 88, 88), "f16s", 1, False), (Q27, (180, 104, 104), "f16s", 1, True),        # 161, 210
    (Q19, (320, 80, 80), "f16s", 1, False), (Q19, (320, 104, 104), "f16s", 1, True),        # two blocks a row: 156, 263
    (Q19, (160, 104, 104), "f16s", 2, False), (Q19, (160, 120, 120), "f16s", 2, True),      # linear: 132, 175
    (Q19, (192, 144, 144), "f16s", 2, False), (Q27, (160, 104, 104), "f16s", 2, True),      # rows 303; D3Q27 187
    (Q27, (128, 104, 104), "f16s", 2, False), (Q19, (150, 120, 120), "f32", 2, False),      # 150; 328
]
IVC_SPHERES = [(Q19, (192, 144, 144), "f16s", False), (Q19, (160, 128, 128), "f16s", False),                # 303, linear 199
               (Q19, (160, 144, 144), "f16s", True), (Q27, (256, 104, 104), "f16s", True),                  # 252, 299
               (Q19, (150, 120, 120), "f32", False)]                                                        # 328
CYLINDERS = [((2000, 2000), "f16s", False), ((3000, 2000), "f16s", True), ((2400, 1250), "f32", False),
             ((2000, 2000), "f32", True), ((2000, 1200), "f64", False), ((2400, 1250), "f64", True)]


def _path(case):
    from ilbmrex_amd.native import Level
    with Level(case, cf.uniform_init(case, u=(case.U0, 0.0, 0.0))) as lev:
        lev.advance(2)
        return lev.step_path()


@pytest.fixture(autouse=True)
def _rule(monkeypatch):
    monkeypatch.delenv("ILBM_OVERLAP_BYTES", raising=False)
    monkeypatch.setenv("ILBM_BODY_TILES", "0")


@pytest.mark.parametrize("lattice,n,storage,loops,overlapped", SPHERES, ids=lambda v: getattr(v, "name", str(v)))
def test_spheres(lattice, n, storage, loops, overlapped):
    c = cf.sphere_3d(nx=n[0], ny=n[1], nz=n[2], D=10.0, center=(40.0, n[1] / 2, n[2] / 2 + 0.3), loop_ns=loops,
                     storage=cf.STORAGE_NAMES[storage]).replace(lattice=lattice)
    print(f"[overlap] {lattice.name} {n} {storage} {loops} iterations", flush=True)
    assert _path(c) == ("three regions" if overlapped else "one stream")


@pytest.mark.parametrize("lattice,n,storage,overlapped", IVC_SPHERES, ids=lambda v: getattr(v, "name", str(v)))
def test_ivc_spheres(lattice, n, storage, overlapped):
    c = cf.sphere_3d(nx=n[0], ny=n[1], nz=n[2], D=8.0, center=(40.0, n[1] / 2, n[2] / 2 + 0.3),
                     coupling=cf.COUPLING_IVC, storage=cf.STORAGE_NAMES[storage]).replace(lattice=lattice)
    print(f"[overlap] IVC {lattice.name} {n} {storage}", flush=True)
    assert _path(c) == ("three regions" if overlapped else "one stream")


@pytest.mark.parametrize("n,storage,overlapped", CYLINDERS)
def test_cylinders(n, storage, overlapped):
    c = cf.cylinder_2d(nx=n[0], ny=n[1], D=40.0, xc=0.3 * n[0], yc=0.5 * n[1], storage=cf.STORAGE_NAMES[storage])
    print(f"[overlap] cylinder {n} {storage}", flush=True)
    assert _path(c) == ("three regions" if overlapped else "one stream")


@pytest.mark.parametrize("D,overlapped", [(12, True), (36, False)])
def test_a_wide_body_waits_for_larger_levels(D, overlapped):
    c = cf.sphere_3d(nx=150, ny=120, nz=120, D=float(D), center=(60.0, 60.0, 60.3), storage=cf.STORE_F32)
    print(f"[overlap] D={D}", flush=True)
    assert _path(c) == ("three regions" if overlapped else "one stream")
