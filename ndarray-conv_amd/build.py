"""Builds libndconv.so for gfx950 in-tree (ndarray-conv_amd/lib/).

    python ndarray-conv_amd/build.py [--jobs N]

Every translation unit is compiled with hipcc for gfx950 only; packed FP32
instructions are disabled (-packed-fp32-ops) for all device code.  The atomic
optimizer is off: it rewrites a single lane's fetch-and-add (the batch
work-queue pop) into a wave-wide broadcast that waits for the atomic's return
at once, instead of where the popped index is first used.
"""
import argparse
import concurrent.futures as cf
import os
import subprocess
import sys

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
BUILD = os.path.join(PKG, "_build")
LIBDIR = os.path.join(PKG, "lib")
LIB = os.path.join(LIBDIR, "libndconv.so")

SOURCES = ["plan.cpp", "capi.cpp", "batch.cpp", "direct_conv.hip", "fft_conv.hip", "mfma_conv.hip",
           "batch_conv.hip", "noalloc.hip", "tile_plan.cpp", "tile_conv.hip", "tile_conv_f64.hip",
           "matrix_conv.hip", "batch_tile.hip"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
CFLAGS = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
          "-mllvm", "-amdgpu-atomic-optimizer-strategy=None",
          "-Wall", "-Wno-unused-function", "-Wno-unused-result",
          f"-I{os.path.join(ROOT, 'include')}", f"-I{CSRC}"]


def _compile(src):
    path = os.path.join(CSRC, src)
    obj = os.path.join(BUILD, src + ".o")
    cmd = [HIPCC, "-x", "hip", "-c", path, "-o", obj] + CFLAGS
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    return obj, r.stderr


def build(jobs=None, verbose=False):
    os.makedirs(BUILD, exist_ok=True)
    os.makedirs(LIBDIR, exist_ok=True)
    jobs = jobs or min(len(SOURCES), os.cpu_count() or 4)
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        results = list(ex.map(_compile, SOURCES))
    if verbose:
        for _, warn in results:
            if warn.strip():
                print(warn, file=sys.stderr)
    objs = [o for o, _ in results]
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=None)
    ap.add_argument("-v", "--verbose", action="store_true")
    args = ap.parse_args()
    print(build(args.jobs, args.verbose))
