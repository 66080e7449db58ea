"""Build libamaterasu_amd.so in-tree with hipcc for gfx950.

``python -m amaterasu_amd.build`` compiles every source under ``csrc/`` (in parallel) and
links the shared library next to this file, where ``amaterasu_amd._lib`` loads it.
"""

from __future__ import annotations

import concurrent.futures
import os
import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent
CSRC = HERE / "csrc"
OUT = HERE / "libamaterasu_amd.so"
BUILD = HERE / "_build"
ARCH = os.environ.get("AMT_OFFLOAD_ARCH", "gfx950")

SOURCES = ["abi.cpp", "fft.hip", "fft_fast.hip", "fft_fast_a.hip", "fft_fast_b.hip", "fft_fast_c.hip",
           "fft_fast_d.hip", "gemm.hip", "dav.hip", "mlp.hip", "eig.hip", "chol.hip", "xc.hip",
           "noalloc.hip"]
LIBS: list = []
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
# Packed-FP32 instructions are disabled on purpose: plain float code only.
DEVICE_FLAGS = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
COMMON = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-Wall", "-Wno-unused-result"]


def _compile(src: str) -> Path:
    obj = BUILD / (Path(src).stem + ".o")
    cmd = [HIPCC, *COMMON, *DEVICE_FLAGS, "-I", str(HERE.parent / "include"), "-c", str(CSRC / src), "-o", str(obj)]
    if src.endswith(".cpp"):
        cmd = [HIPCC, "-O3", "-std=c++17", "-fPIC", "-Wall", "-I", str(HERE.parent / "include"), "-c",
               str(CSRC / src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{res.stdout}\n{res.stderr}")
    return obj


def build(verbose: bool = False) -> Path:
    BUILD.mkdir(exist_ok=True)
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, len(SOURCES))) as pool:
        objs = list(pool.map(_compile, SOURCES))
    tmp = OUT.with_suffix(".so.tmp")
    cmd = [HIPCC, "-shared", f"--offload-arch={ARCH}", "-o", str(tmp), *map(str, objs), *LIBS]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, OUT)
    if verbose:
        print(f"built {OUT}")
    return OUT


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
