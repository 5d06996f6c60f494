"""Build libtm.so (HIP, gfx950) in-tree with hipcc.

    python -m trophic_maelstorm_amd.build      # or trophic_maelstorm_amd.build.build()

The FP64 kernels are compiled with -ffp-contract=off so their arithmetic rounds
exactly like the CPU restatement; all HIP code disables packed FP32 ops.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
INCLUDE = os.path.join(ROOT, "include")
BUILD = os.path.join(PKG, "_build")
LIB = os.path.join(PKG, "libtm.so")

ARCH = "gfx950"
COMMON = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-I", INCLUDE, "-I", CSRC,
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wall", "-Wno-unused-function"]
# The FP64 kernels hold some two hundred 64-bit literals (their polynomials).  Hoisted
# out of the cell loops they overflow the SGPRs and every use reads one back from a
# VGPR lane (450 SGPR spills in the two-pass DP step, 134 VGPRs); left in place they
# cost scalar moves beside the FP64 work (71 spills, 91 VGPRs).  The FP32 kernels'
# literals are instruction operands: the same flag measured nothing there.
NO_LICM = ["-mllvm", "-disable-machine-licm"]
UNITS = {
    "tm_kernels_f64.hip": ["-ffp-contract=off", *NO_LICM],
    "tm_kernels_f32.hip": ["-ffp-contract=fast"],
    "tm_ensemble.hip": ["-ffp-contract=off"],
    "tm_frames.hip": ["-ffp-contract=off"],
    "tm_consumers.hip": ["-ffp-contract=off", *NO_LICM],
    "tm_movement.hip": ["-ffp-contract=off", *NO_LICM],
    "tm_api.cpp": ["-ffp-contract=off"],
    "tm_io.cpp": ["-ffp-contract=off"],
    "tm_hostcopy.hip": [],
    "tm_groups.hip": [],
}


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found: the HIP toolchain is required to build libtm")


def _compile(src: str, extra: list[str]) -> str:
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    cmd = [hipcc(), *COMMON, *extra, "-c", os.path.join(CSRC, src), "-o", obj]
    if src.endswith(".cpp"):
        cmd[1:1] = ["-x", "hip"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr}")
    return obj


def build(verbose: bool = False) -> str:
    """Compile every HIP unit for gfx950 and link libtm.so next to this file."""
    os.makedirs(BUILD, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=len(UNITS)) as ex:
        objs = list(ex.map(lambda kv: _compile(*kv), UNITS.items()))
    tmp = LIB + ".tmp"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
