"""Build librtm_hip.so (all HIP sources under csrc/) for gfx950 with hipcc.

Run as ``python -m elastic_amd.build``. The library is built in-tree next to
this file so that it travels with the repository snapshot.
"""
from __future__ import annotations

import concurrent.futures
import glob
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "librtm_hip.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

# Kernel arguments are preloaded into scalar registers while a launch is being
# dispatched, instead of being loaded by each wave first: 0.3 to 0.5 us of a 4
# to 9 us step launch on small grids.
# Packed-FP32 VALU forms are disabled for all device code; the compiler still
# vectorises ordinary float code with the other instructions.
HIP_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
    "-Wall", "-Wno-unused-function", "-Wno-unused-result",
]


def build(verbose: bool = False) -> str:
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    objdir = os.path.join(HERE, "_build")
    os.makedirs(objdir, exist_ok=True)
    objs = [os.path.join(objdir, os.path.basename(src) + ".o") for src in srcs]
    cmds = [[HIPCC, *HIP_FLAGS, "-c", src, "-o", obj] for src, obj in zip(srcs, objs)]
    # one hipcc per source, in parallel (each is single-threaded)
    jobs = max(1, min(len(cmds), int(os.environ.get("MAX_JOBS", os.cpu_count() or 1))))
    with concurrent.futures.ThreadPoolExecutor(jobs) as pool:
        for cmd in cmds:
            if verbose:
                print(" ".join(cmd), flush=True)
        for r in pool.map(lambda c: subprocess.run(c, capture_output=True, text=True), cmds):
            sys.stderr.write(r.stderr)
            if r.returncode != 0:
                raise subprocess.CalledProcessError(r.returncode, r.args, r.stdout, r.stderr)
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    os.replace(tmp, LIB)
    shutil.rmtree(objdir, ignore_errors=True)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
