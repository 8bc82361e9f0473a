"""Build ``libkda_hip.so`` (the gfx950 KDA kernels + C ABI) in-tree with hipcc.

Usage: ``python -kimi-linear-_amd/build.py`` or ``build_native()`` from Python.
The library lands next to this file, where ``_native.py`` loads it from.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
REPO_DIR = PKG_DIR.parent
CSRC = PKG_DIR / "csrc"
INCLUDE = REPO_DIR / "include"
LIB_PATH = PKG_DIR / "libkda_hip.so"
HOST_PATH = PKG_DIR / "_kda_host.so"
BUILD_DIR = PKG_DIR / "_build"

SOURCES = ["kda_api.hip", "kda_recurrent.hip", "kda_chunkwise.hip", "kda_chunkwise_bwd.hip", "kda_layer_ops.hip",
           "kda_layer_bwd.hip", "kda_long.hip", "kda_ckpt_fp32.hip", "kda_linear.hip"]

# -packed-fp32-ops: no v_pk_{add,mul,fma}_f32 in the device code.
HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(exe).exists():
        raise RuntimeError("hipcc not found: a ROCm toolchain is required to build libkda_hip.so")
    return exe


def _run(cmd: list[str]) -> None:
    proc = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(line for line in proc.stderr.splitlines() if noise not in line)
    if proc.returncode != 0:
        raise RuntimeError(f"command failed ({proc.returncode}): {' '.join(cmd)}\n{proc.stdout}\n{err}")
    if err.strip():
        print(err, file=sys.stderr)


def build_host(verbose: bool = False) -> Path:
    """Compile the wrapper's native side (host code only) against torch."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths, library_paths
    tmp = HOST_PATH.with_suffix(".so.tmp")
    cmd = [shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f'-DKDA_TORCH_VERSION="{torch.__version__}"',
           *(x for p in include_paths() for x in ("-isystem", p)), f"-I{sysconfig.get_paths()['include']}",
           f"-I{INCLUDE}", str(CSRC / "host_binding.cpp"), "-o", str(tmp),
           *(f"-L{p}" for p in library_paths()), "-lc10", "-ltorch_cpu", "-ltorch", "-ltorch_python"]
    if verbose:
        print(" ".join(cmd))
    _run(cmd)
    os.replace(tmp, HOST_PATH)
    return HOST_PATH


def build_native(verbose: bool = False) -> Path:
    """Compile every source for gfx950, link the shared library and build the wrapper's native side."""
    hipcc = _hipcc()
    BUILD_DIR.mkdir(exist_ok=True)
    incs = [f"-I{INCLUDE}", f"-I{CSRC}"]

    def compile_one(src: str) -> Path:
        obj = BUILD_DIR / (Path(src).stem + ".o")
        cmd = [hipcc, *HIPCC_FLAGS, *incs, "-c", str(CSRC / src), "-o", str(obj)]
        if verbose:
            print(" ".join(cmd))
        _run(cmd)
        return obj

    workers = max(1, min(len(SOURCES), int(os.environ.get("MAX_JOBS", "4"))))
    with ThreadPoolExecutor(max_workers=workers) as pool:
        host = pool.submit(build_host, verbose)
        objs = list(pool.map(compile_one, SOURCES))
        host.result()
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)]
    if verbose:
        print(" ".join(cmd))
    _run(cmd)
    os.replace(tmp, LIB_PATH)
    return LIB_PATH


if __name__ == "__main__":
    print(build_native(verbose="-v" in sys.argv))
