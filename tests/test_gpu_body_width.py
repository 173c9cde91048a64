"""Body tiles against the width of the body: a wide body on a small level keeps
the separate forcing kernels, a narrow one and a wide one on a large level
take tiles, with the same bits on both paths."""
import numpy as np
import pytest

from ilbmrex_amd import config as cf

pytestmark = pytest.mark.gpu

# size, diameter, what the step takes in FP64 and in reduced storage
CASES = [((500, 400), 60, "body tiles", "body tiles"), ((500, 400), 90, "body tiles", "body tiles"),
         ((500, 400), 150, "one stream", "one stream"), ((500, 400), 275, "one stream", "one stream"),
         ((300, 260), 200, "one stream", "one stream"), ((1000, 1000), 120, "body tiles", "body tiles"),
         ((1000, 1000), 150, "body tiles", "one stream"), ((1000, 1000), 220, "one stream", "one stream")]


def _run(case):
    from ilbmrex_amd.native import Level
    with Level(case, cf.uniform_init(case, u=(case.U0, 0.0, 0.0))) as lev:
        lev.advance(2)
        lev.advance(5, want_state=True)
        return lev.step_path(), [lev.f(), lev.macro(), *lev.markers(), lev.force_history(), lev.mass_history()]


@pytest.mark.parametrize("storage", ["f64", "f32", "f16s"])
@pytest.mark.parametrize("n,D,f64,reduced", CASES)
def test_path_and_results(monkeypatch, n, D, f64, reduced, storage):
    c = cf.cylinder_2d(nx=n[0], ny=n[1], D=float(D), xc=0.45 * n[0], yc=0.5 * n[1] + 0.3, U=0.02, Re=40.0,
                       storage=cf.STORAGE_NAMES[storage])
    print(f"[body] {n} D={D} {storage}", flush=True)
    monkeypatch.delenv("ILBM_BODY_TILES", raising=False)
    path, got = _run(c)
    assert path == (f64 if storage == "f64" else reduced)
    monkeypatch.setenv("ILBM_BODY_TILES", "0" if path == "body tiles" else "1")
    other, ref = _run(c)
    assert {path, other} == {"body tiles", "one stream"}
    assert all(np.array_equal(a, b) for a, b in zip(got, ref))


def test_a_refused_body_does_not_pay_for_the_tables(monkeypatch):
    """Markers too dense for a tile's lists are refused at the first tile: the
    first advance takes no longer than without tiles by a millisecond (the
    tables of all 20,000 markers take four)."""
    import time

    from ilbmrex_amd.native import Level
    c = cf.cylinder_2d(nx=300, ny=150, D=60.0, xc=100.0, yc=75.0).replace(n_marker=20000)
    init = cf.uniform_init(c, u=(c.U0, 0.0, 0.0))
    best = {}
    for tiles in ("0", "1") * 4:
        monkeypatch.setenv("ILBM_BODY_TILES", tiles)
        with Level(c, init) as lev:
            t = time.perf_counter()
            lev.advance(1)
            best[tiles] = min(best.get(tiles, 1.0), time.perf_counter() - t)
            assert lev.step_path() == "one stream"
    print(f"[body] first advance {best}", flush=True)
    assert best["1"] - best["0"] < 1e-3
