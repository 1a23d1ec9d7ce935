"""Build libgodar_amd.so (hand-written HIP for gfx950) in-tree."""
from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libgodar_amd.so")
PLACE_LIB = os.path.join(HERE, "libgodar_place.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("GODAR_ARCH", "gfx950")

# -ffp-contract=off keeps FP64 rounding identical to the reference (no fused
# multiply-adds); packed FP32 instructions are disabled on this target.
# -disable-machine-licm keeps the compiler from hoisting the physics' FP64
# constants out of the kernels' work loops: it held hundreds of them in scalar
# registers, spilled to vector registers and those to scratch (k_contact FP64
# 476 scalar spills and 160 B of scratch -> 26 and 40 B, k_repair 711 -> 7 and
# 140 -> 98 VGPRs, k_walls 155 -> 120), though each costs one move where used
# (262,144 floes FP64: contacts 0.038 -> 0.031 ms, fix-up 0.047 -> 0.032).
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-shared",
    "-ffp-contract=off", "-mllvm", "-disable-machine-licm",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def build_place(verbose: bool = False) -> str:
    """Host-only placement helper of the workload generators (gcc)."""
    tmp = PLACE_LIB + ".tmp"
    cmd = ["gcc", "-O2", "-fPIC", "-shared", "-std=c11", "-o", tmp,
           os.path.join(CSRC, "place.c"), "-lm"]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    os.replace(tmp, PLACE_LIB)
    return PLACE_LIB


def build(verbose: bool = False) -> str:
    build_place(verbose)
    src = os.path.join(CSRC, "godar_lib.hip")
    tmp = LIB + ".tmp"
    cmd = [HIPCC, *FLAGS, "-I", os.path.join(ROOT, "include"), "-I", CSRC, "-o", tmp, src]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in r.stdout.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed:\n{out}")
    if verbose and out.strip():
        print(out)
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
