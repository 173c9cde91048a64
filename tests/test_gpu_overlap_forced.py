"""The overlapped IB step on levels that by their size step on one stream
(ILBM_OVERLAP_BYTES=0): the same results."""
import numpy as np
import pytest

from ilbmrex_amd import config as cf

pytestmark = pytest.mark.gpu


def _run(case, n):
    from ilbmrex_amd.native import Level
    with Level(case, cf.uniform_init(case, u=(case.U0, 0.0, 0.0))) as lev:
        lev.advance(n, want_state=True)
        return lev.f(), lev.force_history(), lev.mass_history()


@pytest.mark.parametrize("storage", ["f32", "f16s"])
@pytest.mark.parametrize("n", [(128, 96, 96), (161, 97, 83)])
def test_overlap_below_its_size(monkeypatch, n, storage):
    c = cf.sphere_3d(nx=n[0], ny=n[1], nz=n[2], D=16.0, center=(40.0, 48.0, 40.0), storage=cf.STORAGE_NAMES[storage])
    print(f"[overlap] sphere {n} {storage}", flush=True)
    one = _run(c, 9)
    monkeypatch.setenv("ILBM_OVERLAP_BYTES", "0")
    two = _run(c, 9)
    assert np.array_equal(one[0], two[0]) and np.array_equal(one[1], two[1])
    assert np.abs(one[2] - two[2]).max() <= 1e-12 * one[2][0]
