"""Compile the HIP library for gfx950 in-tree (``_lib/liblbm_paged_attn.so``), and the Python extension module of the
host side of its attention calls (``_lib/lbm_host.so``).

hipcc cross-compiles without a GPU.  The packed-FP32 VALU forms are switched off for all
device code; the host pass prints a harmless "not a recognized feature" note for that flag.
"""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "csrc")
LIB_DIR = os.path.join(HERE, "_lib")
LIB_PATH = os.path.join(LIB_DIR, "liblbm_paged_attn.so")
HOST_PATH = os.path.join(LIB_DIR, "lbm_host.so")
SOURCES = ["c_abi.hip", "tables_gfx950.hip", "append_gfx950.hip", "qkv_prepare_gfx950.hip", "residual_norm_gfx950.hip", "frame_gfx950.hip", "linear_gfx950.hip",
           "paged_attn_gfx950.hip", "paged_attn_f32_gfx950.hip"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # no NaN-quieting moves around the row-maximum chains of the attention kernel; the
    # only NaN test in the library (fp32 -> bf16 append) is done on the integer bits
    "-fno-honor-nans",
]


def _build_host() -> None:
    """The extension module: against torch's headers and the library just built."""
    from torch.utils.cpp_extension import ROCM_HOME, include_paths, library_paths
    rocm = ROCM_HOME or "/opt/rocm"
    # NDEBUG: without it pybind11's headers bring a thread-local counter.  glibc up to 2.38 takes the slow way to every
    # thread-local of a process once a library with any of its own has been loaded whose thread-locals nobody touches: 10 %
    # on everything Python and torch do (an eager aggregator of 36 blocks on a small image 1,790 us a frame instead of 1,670).
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-DNDEBUG", "-std=c++17", "-fPIC", "-shared", "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__=1",
           *[f"-I{p}" for p in (*include_paths(), sysconfig.get_paths()["include"], os.path.join(rocm, "include"))],
           os.path.join(CSRC, "host_calls.cpp"), "-o", HOST_PATH, *[f"-L{p}" for p in (*library_paths(), LIB_DIR)],
           "-ltorch_python", "-ltorch_cpu", "-ltorch", "-lc10", "-lc10_hip", "-llbm_paged_attn", "-Wl,-rpath,$ORIGIN"]
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed ({proc.returncode}):\n{' '.join(cmd)}\n{proc.stdout}")


def build(verbose: bool = False) -> str:
    os.makedirs(LIB_DIR, exist_ok=True)
    if os.path.exists(HOST_PATH):      # (built last: no old one is left beside a new library)
        os.remove(HOST_PATH)
    cmd = [HIPCC, *FLAGS, "-o", LIB_PATH, *[os.path.join(CSRC, s) for s in SOURCES]]
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in proc.stdout.splitlines() if "not a recognized feature" not in l)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed ({proc.returncode}):\n{' '.join(cmd)}\n{out}")
    if verbose and out.strip():
        print(out, file=sys.stderr)
    _build_host()
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose=True))
