"""Body tiles (a 2D body's forcing inside the stream-collide launch)
against the separate forcing kernels, which the oracle tests pin:
the same sums in the same order, so every result is the same bits.  FP64 and
reduced storage, every
coupling, one and more iterations, bodies across a periodic boundary and at
walls, and an advance split into parts."""
import numpy as np
import pytest

from ilbmrex_amd import config as cf

pytestmark = pytest.mark.gpu

CHANNEL = dict(nx=96, ny=64, D=16.0, xc=32.0, yc=31.7, U=0.05, Re=80.0)
CASES = {
    "explicit": cf.cylinder_2d(**CHANNEL),
    "delta3_loop3": cf.cylinder_2d(**CHANNEL, loop_ns=3, delta_type=3),
    "loop2_wide": cf.cylinder_2d(nx=391, ny=203, D=25.0, xc=105.0, yc=101.5, loop_ns=2, delta_type=3),
    "ivc": cf.cylinder_2d(**CHANNEL, coupling=cf.COUPLING_IVC),
    "diag": cf.cylinder_2d(**CHANNEL, coupling=cf.COUPLING_EXPLICIT_DIAG).replace(mdf_relax=0.5),
    "renorm": cf.cylinder_2d(**CHANNEL).replace(renormalize_delta=1),
    "spinning": cf.cylinder_2d(**CHANNEL).replace(ub=(0.001, 0.002, 0.003), om=(0.0, 0.0, 0.002)),
    # stencils across the periodic boundary, on a row width that is no multiple of 64
    "periodic_edge": cf.cylinder_2d(nx=150, ny=40, D=12.0, xc=40.0, yc=2.0, U=0.05, Re=50.0),
    # one stencil column on the inflow face
    "at_inflow": cf.cylinder_2d(nx=64, ny=40, D=8.0, xc=6.5, yc=20.0, U=0.05, Re=40.0),
    "cavity": cf.cavity_ibm_box(),
    # a row of 192 threads per block, many tiles
    "wide": cf.cylinder_2d(nx=190, ny=150, D=60.0, xc=70.0, yc=75.0, U=0.05, Re=100.0),
    # many entries per cell: the most markers a tile's LDS holds, and more
    "dense": cf.cylinder_2d(**CHANNEL).replace(n_marker=120),
    "too_dense": cf.cylinder_2d(**CHANNEL).replace(n_marker=400),
    # more iterations than body tiles take
    "loop4": cf.cylinder_2d(**CHANNEL, loop_ns=4),
}


# forcing that diverges: every value that is not finite stays where it was
UNSTABLE = cf.cylinder_2d(nx=130, ny=68, D=9.0, xc=35.0, yc=34.0, U=0.05, Re=75.0, loop_ns=2, delta_type=3)


def _run(case, parts):
    from ilbmrex_amd.native import Level
    m = cf.uniform_init(case, u=(case.bc_lo_val[0][1], 0.0, 0.0))
    m[1] += 0.002 * np.random.default_rng(5).uniform(-1.0, 1.0, case.ncells)
    with Level(case, m) as lev:
        for n in parts:
            lev.advance(n, want_state=True)
        xyz, uvw, fxyz = lev.markers()
        return {"f": lev.f(), "macro": lev.macro(), "forcing": lev.forcing(), "uvw": uvw, "fxyz": fxyz,
                "history": lev.force_history(), "sum": lev.last_marker_force_sum(), "torque": lev.torque(),
                "checkpoint": np.frombuffer(lev.checkpoint(), dtype=np.uint8), "mass": lev.mass_history()}


@pytest.mark.parametrize("storage", ["f64", "f32", "f16s"])
@pytest.mark.parametrize("name", list(CASES))
def test_body_tiles_equal_separate_kernels(monkeypatch, name, storage):
    case = CASES[name].replace(storage=cf.STORAGE_NAMES[storage])
    print(f"[body] {name} {storage}", flush=True)
    one = _run(case, [13])
    split = _run(case, [1, 4, 8])
    monkeypatch.setenv("ILBM_BODY_TILES", "0")
    ref = _run(case, [13])
    for got in (one, split):
        for k, v in ref.items():
            assert np.array_equal(got[k], v), k


@pytest.mark.parametrize("storage", ["f64", "f32", "f16s"])
def test_body_tiles_equal_separate_kernels_when_diverging(monkeypatch, storage):
    case = UNSTABLE.replace(storage=cf.STORAGE_NAMES[storage])
    print(f"[body] diverging {storage}", flush=True)
    one = _run(case, [140])
    monkeypatch.setenv("ILBM_BODY_TILES", "0")
    ref = _run(case, [140])
    del one["checkpoint"], ref["checkpoint"]   # the bits of a NaN are not compared
    assert not np.isfinite(ref["history"]).all()
    for k, v in ref.items():
        assert np.array_equal(one[k], v, equal_nan=True), k


def test_record_beside_a_step_of_192_thread_blocks():
    """The force record rides in the stream-collide launch of a hierarchy's
    finest level, whose blocks hold 192 threads when its box is 129 to 192
    cells wide; more markers than that."""
    import refcpu
    from ilbmrex_amd.native import AmrHierarchy
    c = cf.cylinder_2d(nx=110, ny=56, D=12.0, xc=50.0, yc=28.0, U=0.05, Re=60.0).replace(n_marker=230)
    boxes = [((20, 20, 0), (179, 91, 0))]
    print("[body] hierarchy with a finest level 160 cells wide", flush=True)
    state = (1.0, 0.05, 0.0, 0.0)
    with AmrHierarchy(c, boxes, 2, state) as h:
        h.advance(3, want_state=True)
        o = refcpu.AmrOracle(c, boxes, 2, cf.uniform_init(c, u=(0.05, 0.0, 0.0)))
        o.advance(3)
        assert np.array_equal(h.macro(1), o.macro(1))
        rec, got = o.force_record(), h.force_history()[-1]
    floor = 1e-10 * np.abs(rec).max()
    assert np.all(np.abs(got - rec) <= 1e-12 * np.abs(rec) + floor), (got, rec)
