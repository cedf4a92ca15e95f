"""Build the HIP engine in-tree: gmes_amd/lib/libgmes_engine.so (gfx950).

FMA contraction is off so that FP64 runs keep the reference's operation
order; packed-FP32 instructions are disabled for the device code.
"""

import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.dirname(HERE)
LIB = os.path.join(PKG, "lib", "libgmes_engine.so")
# (file, extra flags): the kernel files but step3d.hip are compiled once per storage type
SOURCES = [("engine.hip", []), ("step3d.hip", [])] + [
    (src, ["-DGMES_TYPE=%d" % t])
    for src, n in (("kernels.hip", 4), ("step1d.hip", 4), ("step2d.hip", 4), ("stepfix.hip", 3)) for t in range(n)]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("GMES_OFFLOAD_ARCH", "gfx950")

FLAGS = ["-O3", "-std=c++17", "-fPIC", "-shared", "--offload-arch=" + ARCH,
         "-ffp-contract=off", "-fno-fast-math",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-Wno-unused-result", "-Wno-unused-command-line-argument", "-Wno-inline-asm"]


def build(verbose=True):
    """Compile the sources side by side, then link them."""
    os.makedirs(os.path.dirname(LIB), exist_ok=True)
    tmp = LIB + ".tmp"
    with tempfile.TemporaryDirectory() as d:
        jobs = []
        for n, (src, extra) in enumerate(SOURCES):
            obj = os.path.join(d, "%d.o" % n)
            cmd = [HIPCC] + [f for f in FLAGS if f != "-shared"] + extra + ["-c", "-o", obj, os.path.join(HERE, src)]
            if verbose:
                print(" ".join(cmd), flush=True)
            jobs.append((cmd, obj, subprocess.Popen(cmd)))
        for cmd, _, p in jobs:
            if p.wait() != 0:
                raise subprocess.CalledProcessError(p.returncode, cmd)
        cmd = [HIPCC, "-shared", "-fPIC", "--offload-arch=" + ARCH, "-o", tmp] + [o for _, o, _ in jobs]
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.run(cmd, check=True)
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    build()
    sys.exit(0)
