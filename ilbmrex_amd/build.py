"""Builds libilbm_hip.so in-tree for gfx950 with hipcc."""
from __future__ import annotations

import os
import subprocess
import sys

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG_DIR)
CSRC = os.path.join(PKG_DIR, "csrc")
OUT = os.path.join(PKG_DIR, "_lib", "libilbm_hip.so")

SOURCES = ["ilbm_level.hip"]
# headers the one translation unit includes
HEADERS = ["ilbm_host_copy.h", "ilbm_lattice.h", "ilbm_lbm_kernels.h", "ilbm_ib_kernels.h",
           "ilbm_amr_kernels.h", "ilbm_batch_impl.h", "ilbm_box_impl.h", "ilbm_box_ib_impl.h", "ilbm_amr_impl.h"]

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    # no fused multiply-add contraction: FP64 results follow the reference's
    # separate multiply and add roundings
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def build(verbose: bool = False) -> str:
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    cmd = [hipcc, *HIPCC_FLAGS, "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
           "-o", OUT + ".tmp"] + [os.path.join(CSRC, s) for s in SOURCES]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("hipcc failed building libilbm_hip.so")
    os.replace(OUT + ".tmp", OUT)
    if verbose:
        print("built", OUT)
    return OUT


if __name__ == "__main__":
    build(verbose=True)
