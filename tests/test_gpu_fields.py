"""Whole fields to the host: copies below, at and above the size from which
several threads share one, with and without a partial last slice, and more
slices than threads."""
import numpy as np
import pytest

from ilbmrex_amd import config as cf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1024, 1023, 1), (1024, 1024, 1), (1025, 1024, 1), (1200, 1100, 1), (112, 98, 97)])
def test_fields_arrive_whole(n):
    from ilbmrex_amd.native import Level
    lat = cf.D2Q9 if n[2] == 1 else cf.D3Q19
    c = cf.periodic_box(lat, n, nu=0.05)
    m = cf.random_init(c, seed=3)
    print(f"[fields] {lat.name} {n}", flush=True)
    with Level(c, m) as lev:
        assert np.array_equal(lev.macro(), m)      # the initial state as given
        lev.advance(2, want_state=True)
        f, mac = lev.f(), lev.macro()
        again = lev.macro()
    assert np.array_equal(mac, again)
    rho = np.zeros(c.ncells)
    for q in range(lat.q):                          # the kernel's order
        rho += f[q]
    assert np.array_equal(rho, mac[0])
