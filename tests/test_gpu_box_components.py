"""ilbm_box_fill_patch (mesoscopic) of arrays with more components than
populations against the separate stages: the same bits in every component of
every cell, over the boundary kinds."""
import itertools

import numpy as np
import pytest

from ilbmrex_amd import config as cf
from test_gpu_box_fused import KINDS, _Box, _case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lattice,n,dim", [(cf.D2Q9, (12, 9, 1), 2), (cf.D3Q19, (7, 5, 6), 3)],
                         ids=lambda v: getattr(v, "name", None))
def test_components_beyond_the_populations(lattice, n, dim):
    kinds = list(itertools.product(KINDS, repeat=2))
    rng = np.random.default_rng(11)
    for k in kinds:
        k = k + ("open",) * (dim - 2)
        b = _Box(_case(lattice, n, k), (0, 0, 0), tuple(x - 1 for x in n), False, 3)
        nc = b.q + 3
        print(f"[box] {lattice.name} {k} {nc} components", flush=True)
        src, one, ref = b.arr(nc), b.arr(nc), b.arr(nc)
        src.upload(1.0 + 0.1 * rng.uniform(-1, 1, src.download().shape))
        b.call("box_copy", src.ref(), ref.ref(), b.lo, b.hi, nc, None)
        b.call("box_fill_periodic", b.d, ref.ref(), b.lo, b.hi, None)
        b.call("box_fill_physical", b.d, ref.ref(), 1, None)
        b.call("box_setval", one.ref(), 7.0, None)
        b.call("box_fill_patch", b.d, src.ref(), one.ref(), 1, b.lo, b.hi, None)
        x, y = one.download(), ref.download()
        assert np.array_equal(x, y), f"{k}: {np.count_nonzero(x != y)} of {x.size} differ"
