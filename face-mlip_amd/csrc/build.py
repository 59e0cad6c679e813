"""Compile the HIP sources of this directory into face_amd/libface_hip.so (gfx950).

Usage: python face-mlip_amd/csrc/build.py [--jobs N]
Each .hip file is compiled to an object in parallel, then linked into one shared library.
"""
import argparse
import concurrent.futures as cf
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "face_amd")
OUT = os.path.join(PKG, "libface_hip.so")
BUILD = os.path.join(HERE, "_build")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("FACE_OFFLOAD_ARCH", "gfx950")
# Packed FP32 instructions are disabled for every kernel; no fast-math (the pair test needs IEEE fp64).
FLAGS = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-Xclang", "-target-feature", "-Xclang",
         "-packed-fp32-ops", "-Wall"]
# graph.hip evaluates the pair-acceptance test in fp64 with a fixed operation order: no contraction.
SOURCES = {"capi.hip": "fast", "density.hip": "fast", "cprad.hip": "fast", "densfac.hip": "fast", "node.hip": "fast",
           "edge.hip": "fast", "graph.hip": "off",
           "transport.hip": "fast", "radial.hip": "fast", "linear.hip": "fast",
           "gemm.hip": "fast", "gemm_xs.hip": "fast", "gemm_split.hip": "fast", "gemm_op.hip": "fast", "densmix.hip": "fast"}


def compile_one(src):
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC, *FLAGS, f"-ffp-contract={SOURCES[src]}", "-c", os.path.join(HERE, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr}")
    return obj, r.stderr


def stale(src):
    """True when the object of src is missing or older than src or a header it includes."""
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    if not os.path.exists(obj):
        return True
    t = os.path.getmtime(obj)
    return any(os.path.getmtime(os.path.join(HERE, f)) > t
               for f in (src, "common.h", "edges.h", "densfac.h", "rows_gemm.h", "../../include/face_hip.h"))


def build(jobs=None, verbose=False, changed_only=False):
    os.makedirs(BUILD, exist_ok=True)
    todo = [s for s in SOURCES if stale(s)] if changed_only else list(SOURCES)
    with cf.ThreadPoolExecutor(max_workers=jobs or min(8, max(1, len(todo)))) as ex:
        results = list(ex.map(compile_one, todo))
    objs = [os.path.join(BUILD, os.path.splitext(s)[0] + ".o") for s in SOURCES]
    if verbose:
        for _, err in results:
            if err.strip():
                print(err, file=sys.stderr)
    tmp = OUT + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, OUT)
    return OUT


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=None)
    ap.add_argument("-v", action="store_true")
    ap.add_argument("--changed", action="store_true", help="recompile only sources newer than their objects")
    a = ap.parse_args()
    print(build(a.jobs, a.v, a.changed))
