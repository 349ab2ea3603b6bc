"""Builds libkukan_hip.so (gfx950) in-tree with hipcc, one object per source in parallel."""
from __future__ import annotations

import concurrent.futures as cf
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "_obj")
LIB = os.path.join(HERE, "libkukan_hip.so")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
HIPCC = os.path.join(ROCM, "bin", "hipcc")
ARCH = "gfx950"
SOURCES = ["common.hip", "kernels.hip", "gemm_mixed.hip", "gemm_f64.hip", "hartree_cg.hip", "seqcg.hip", "solvers.hip", "batch.hip", "abi.hip",
           "noalloc.hip", "bloch.hip", "abi_bloch.hip", "transfer.hip", "abi_trans.hip", "checkpoint.hip", "projector.hip",
           "force.hip"]
CFLAGS = ["-O3", "-fPIC", "-std=c++17", f"--offload-arch={ARCH}", "-Wall", "-Wno-unused-result",
          # packed FP32 instructions stay off (see the design notes on gfx950 hazards)
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
          "-I", os.path.join(os.path.dirname(HERE), "include")]
LDFLAGS = ["-shared", f"--offload-arch={ARCH}", "-L", os.path.join(ROCM, "lib"), "-lrocblas",
           "-lrocsolver", "-lrocprofiler-sdk-roctx", f"-Wl,-rpath,{os.path.join(ROCM, 'lib')}"]


def _compile(src):
    out = os.path.join(OBJ, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC, *CFLAGS, "-c", os.path.join(CSRC, src), "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stderr[-6000:]}")
    return out


def build(verbose=False):
    os.makedirs(OBJ, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=len(SOURCES)) as ex:
        objs = list(ex.map(_compile, SOURCES))
    tmp = LIB + ".tmp"
    r = subprocess.run([HIPCC, *LDFLAGS, *objs, "-o", tmp], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr[-6000:]}")
    os.replace(tmp, LIB)
    if verbose:
        print("built", LIB)
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
