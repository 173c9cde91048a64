"""Device memory that runs out while an advance sets up what only its fast path
needs: the advance takes the other path, or fails and can be called again,
with the results of an undisturbed run.  A library loaded before the
framework's in a process of its own refuses one allocation."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

REFUSE = r"""
#include <dlfcn.h>
#include <cstddef>
static int left = 0;
extern "C" void refuse(int k) { left = k; }           // the k-th allocation from now
extern "C" int pending() { return left; }
extern "C" int hipMalloc(void** p, size_t n) {
  static void* hip = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_NOLOAD);   // as the framework loaded it
  if (!hip) return 2;
  static auto real = (int (*)(void**, size_t))dlsym(hip, "hipMalloc");
  return real(p, left > 0 && --left == 0 ? (size_t)1 << 60 : n);   // more than there is
}
"""

PROGRAM = """
import ctypes, sys
lib = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
from ilbmrex_amd import config as cf
from ilbmrex_amd.native import Level

def results(case, first, last, must_succeed):
    # an advance for each allocation refused, first to last
    init = cf.uniform_init(case, u=(case.U0, 0.0, 0.0))
    with Level(case, init) as lev:
        lev.advance(1)
        lev.advance(8, want_state=True)
        ref = lev.f(), lev.force_history()
    for k in range(first, last + 1):
        print("refusing allocation", k, "of the first advance", flush=True)
        with Level(case, init) as lev:
            lib.refuse(k)
            try:
                lev.advance(1)
            except RuntimeError:
                assert not must_succeed, k
                lev.advance(1)
            assert lib.pending() == 0, "the advance allocates less than that"
            lev.advance(8, want_state=True)
            got = lev.f(), lev.force_history()
        assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1]), k
"""


def _child(tmp_path, body, **env):
    (tmp_path / "refuse.cpp").write_text(REFUSE)
    (tmp_path / "program.py").write_text(PROGRAM + body)
    lib = str(tmp_path / "librefuse.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-o", lib, str(tmp_path / "refuse.cpp"), "-ldl"], check=True)
    r = subprocess.run([sys.executable, "-u", str(tmp_path / "program.py"), lib], cwd=ROOT, timeout=100,
                       env={**os.environ, "PYTHONPATH": ROOT, **env}, capture_output=True, text=True)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0


def test_body_tiles_without_memory_for_their_tables(tmp_path):
    # the first six allocations of the advance are the tiles'; the seventh,
    # the Sum(Rho) ring, may fail it
    _child(tmp_path, """
case = cf.cylinder_2d(nx=96, ny=64, D=16.0, xc=32.0, yc=32.0)
results(case, 1, 6, True)
results(case, 7, 7, False)
results(case.replace(loop_ns=2), 1, 7, True)
""")


def test_overlapped_step_without_memory_for_its_record_slots(tmp_path):
    # six slots of the record, then the Sum(Rho) rings of the three regions
    _child(tmp_path, """
case = cf.sphere_3d(nx=128, ny=96, nz=96, D=10.0, center=(48.0, 47.6, 48.3), storage=cf.STORE_F32)
results(case, 1, 9, False)
""", ILBM_OVERLAP_BYTES="0")


def test_a_setting_that_is_not_used_takes_no_memory():
    # IVC forces once whatever loop_ns says; three doubles per marker and
    # iteration would be 10^12 bytes here
    import numpy as np
    from ilbmrex_amd import config as cf
    from ilbmrex_amd.native import Level
    case = cf.cylinder_2d(nx=96, ny=64, D=16.0, xc=32.0, yc=32.0, coupling=cf.COUPLING_IVC)
    out = []
    for loops in (1, 2 ** 31 - 1):
        with Level(case.replace(loop_ns=loops), cf.uniform_init(case, u=(case.U0, 0.0, 0.0))) as lev:
            lev.advance(5, want_state=True)
            out.append((lev.f(), lev.force_history()))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
