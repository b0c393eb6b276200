"""Build libpetite_hip.so for gfx950 with hipcc (in-tree, next to this file).

    python -m petite_amd.build
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(HERE, "libpetite_hip.so")
SOURCES = [os.path.join(HERE, "csrc", "petite_hip.hip")]
HEADERS = ["philox.h", "physics.h", "transport.h", "sweep.h", "tail.h", "quad.h", "dark.h"]

FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    # packed-FP32 (v_pk_*_f32) generation off for every device function
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # float64 constants stay in the loops that use them: hoisted into scalar
    # registers they spill to vector lanes and come back by v_readlane (k_tail
    # 341 scalar and 22 vector spills -> 113 and none, k_transport 121 -> 78
    # vector registers; walk, draws and yields 2-5 % faster)
    "-mllvm", "-disable-machine-licm",
    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(HERE, "csrc"),
]


def build(verbose=True):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    tmp = LIB + ".tmp"
    cmd = [hipcc] + FLAGS + SOURCES + ["-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    build()
    sys.exit(0)
