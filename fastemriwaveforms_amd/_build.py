"""Builds libfew_rocm.so (the HIP kernels + C ABI) in-tree with hipcc for gfx950.

Run ``python -m fastemriwaveforms_amd._build`` or call :func:`build`.
"""

from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG_DIR)
CSRC = os.path.join(PKG_DIR, "csrc")
INCLUDE = os.path.join(ROOT, "include")
BUILD_DIR = os.path.join(PKG_DIR, "_build")
LIB_NAME = "libfew_rocm.so"
LIB_PATH = os.path.join(PKG_DIR, LIB_NAME)
ARCH = os.environ.get("FEW_ROCM_ARCH", "gfx950")

SOURCES = ["capi.hip", "spline.hip", "modesum_direct.hip", "modesum_fact.hip", "modesum_fact16.hip", "batch.hip",
           "cells.hip",
           "adjoint.hip", "adjoint16.hip", "adjoint64.hip",
           "eval.hip", "fd.hip", "amp2d.hip",
           "aak.hip"]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found: the ROCm toolchain is required to build libfew_rocm.so")


def compile_flags() -> list[str]:
    return [
        "-O3",
        "-fPIC",
        "-std=c++17",
        f"--offload-arch={ARCH}",
        # packed FP32 VALU forms are kept out of every kernel
        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
        "-I", CSRC,
        "-I", INCLUDE,
    ]


# Per-source scheduler choice: the factorised sums are bound by instruction issue,
# and the iterative ILP strategy's instruction order measured faster than the
# default (same instructions, same results): 1.5-2 % on the split-FP16 sum of the
# 256-waveform batch, 3.4 % on the FP64-MFMA sum of full1.
_ILP = ["-mllvm", "-amdgpu-sched-strategy=iterative-ilp"]
# The frequency-domain sum's loop holds ~150 FP64 literals (log, exp, atan2, the
# series): hoisted out of it they fill the registers and are spilled lane by lane
# (213 VGPRs and 210 spilled SGPRs against 129 and 25 where they stay).
_NO_LICM = ["-mllvm", "-disable-machine-licm"]
SOURCE_FLAGS = {"modesum_fact16.hip": _ILP, "modesum_fact.hip": _ILP, "fd.hip": _NO_LICM}


def _compile(src: str, verbose: bool) -> str:
    obj = os.path.join(BUILD_DIR, os.path.splitext(src)[0] + ".o")
    base = [hipcc(), *compile_flags()]
    tail = ["-c", os.path.join(CSRC, src), "-o", obj]
    extra = SOURCE_FLAGS.get(src, [])
    cmd = [*base, *extra, *tail]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0 and extra:
        # the scheduler option is a tuning choice: a compiler that rejects it
        # (or fails with it) builds the source with its default schedule
        print(f"note: {src}: {' '.join(extra)} failed, building with the default schedule",
              file=sys.stderr, flush=True)
        r = subprocess.run([*base, *tail], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stderr}")
    return obj


def build(verbose: bool = False) -> str:
    """Compile every HIP source for gfx950 and link libfew_rocm.so (always rebuilds)."""
    os.makedirs(BUILD_DIR, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=min(len(SOURCES), 8)) as ex:
        objs = list(ex.map(lambda s: _compile(s, verbose), SOURCES))
    tmp = LIB_PATH + ".tmp"
    cmd = [hipcc(), "-shared", "-fPIC", f"--offload-arch={ARCH}", *objs, "-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link of {LIB_NAME} failed:\n{r.stderr}")
    os.replace(tmp, LIB_PATH)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
