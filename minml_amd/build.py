"""Builds libminml_hip.so (the C-ABI HIP backend for gfx950) in-tree with hipcc.

One translation unit per source under csrc/; objects go to csrc/build/, the library next to this file. hipcc
cross-compiles for gfx950 without a GPU present, so this runs anywhere the ROCm toolchain is installed.
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(CSRC, "build")
LIB = os.path.join(HERE, "libminml_hip.so")

SOURCES = ["runtime.hip", "winograd.hip", "gemm.hip", "gemm_tiles.hip", "conv.hip", "quantized.hip", "elementwise.hip", "heads.hip", "attention.hip", "moe.hip", "cuda_stubs.cpp"]
# packed fp32 VALU forms are switched off for all device code; the host pass does not know the feature and says so (harmless)
COMMON = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function",
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
# the leading kernel arguments arrive in scalar registers with the wavefront instead of being loaded by it (0.25 us from a workgroup's start until
# they are there): 20 x 256 channels, us per layer of two launches, 1 position 9.1 -> 8.9, 16 14.8 -> 14.6, 32 19.5 -> 19.2; fp32 128 channels 10.7 -> 10.4.
# The launch itself waits for them, up to 0.15 us, so that kernels of a few instructions are behind: element-wise calls on one or 16 boards take as much longer
# (us, without / with: conversion of 225 x 256 elements 1.68 / 1.84, sum of two tensors 1.79 / 1.94, bias and ReLU 2.16 / 2.25), on 256 they gain less (256
# channels 15.8 / 15.4, 11.0 / 11.1, 11.1 / 11.2). Gathers and products of the same length do too (1.81 / 1.88), but their files' longer kernels gain more (routing
# 2 to 7 %, products of the networks 1 %)
PRELOAD = ["-mllvm", "-amdgpu-kernarg-preload-count=16"]
WITHOUT_PRELOAD = {"elementwise.hip"}
# the transforms reproduce the reference's expression trees exactly: no contraction beyond the explicit fma calls
PER_FILE = {"winograd.hip": ["-ffp-contract=off"]}


def hipcc():
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.isabs(cand) and os.path.exists(cand) or not os.path.isabs(cand)):
            return cand
    raise RuntimeError("hipcc not found")


def _run(cmd):
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in res.stdout.splitlines() if "not a recognized feature for this target" not in l)
    if res.returncode != 0:
        raise RuntimeError("command failed: %s\n%s" % (" ".join(cmd), out))
    return out


def build(verbose=False, jobs=None):
    os.makedirs(OBJ, exist_ok=True)
    cc = hipcc()
    jobs = jobs or min(8, os.cpu_count() or 1)

    def compile_one(src):
        obj = os.path.join(OBJ, os.path.splitext(src)[0] + ".o")
        cmd = [cc] + COMMON + ([] if src in WITHOUT_PRELOAD else PRELOAD) + PER_FILE.get(src, []) + ["-c", os.path.join(CSRC, src), "-o", obj]
        if src.endswith(".cpp"):
            cmd = [cc, "-O2", "-std=c++17", "-fPIC", "-Wall", "-x", "c++", "-c", os.path.join(CSRC, src), "-o", obj]
        out = _run(cmd)
        if verbose and out.strip():
            print(out)
        return obj

    with ThreadPoolExecutor(max_workers=jobs) as pool:
        objs = list(pool.map(compile_one, SOURCES))
    _run([cc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB] + objs)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
