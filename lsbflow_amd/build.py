"""Build recipe for the gfx950 library ``lsbflow_amd/liblsbflow_amd.so``.

Every source under ``csrc/`` is compiled by hipcc as HIP for gfx950 only, with
packed-FP32 instruction selection switched off, and linked into one shared
library with a plain C ABI (``include/lsbflow.h``).  Objects go to
``lsbflow_amd/_build/``; the library is written next to this file.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "liblsbflow_amd.so")
SOURCES = ["setup.cpp", "capi.cpp", "fft.hip", "fft_fast.hip", "fft_mixed_x64.hip", "fft_mixed_y64.hip",
           "fft_mixed_x32.hip", "fft_mixed_y32.hip", "fft_mixed_r32.hip", "fft_mixed_r64.hip", "fft_mixed_b64.hip", "zops.hip", "spectral.hip", "physical.hip",
           "step.hip", "dealias.hip", "iodiag.hip", "temperature.hip", "noalloc.hip", "dynamic.hip", "helmrefine.hip",
           "ensemble.hip"]
ARCH = "gfx950"
CFLAGS = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-Wall", "-Wno-unused-function",
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (ROCm is required to build lsbflow_amd)")


def _compile(src: str) -> str:
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    cmd = [hipcc(), "-x", "hip", *CFLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    return obj


def build(jobs: int | None = None, verbose: bool = False) -> str:
    """Compile all sources and link ``liblsbflow_amd.so``; returns its path."""
    os.makedirs(BUILD, exist_ok=True)
    jobs = jobs or min(8, os.cpu_count() or 4)
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(_compile, SOURCES))
    tmp = LIB + ".tmp"
    cmd = [hipcc(), "-shared", f"--offload-arch={ARCH}", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
