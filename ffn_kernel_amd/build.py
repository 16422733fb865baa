"""Build libffnk.so (the HIP kernels + C ABI) for gfx950 with hipcc, and _call.so, Python's way into it, with g++.

    python -m ffn_kernel_amd.build            # compile every csrc/*.hip and link; compile csrc/call.cpp

hipcc cross-compiles without a GPU.  The library is written next to this file so that it
travels with the source tree; nothing is installed outside the tree.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
OBJ_DIR = CSRC / "build"
LIB_PATH = PKG_DIR / "libffnk.so"
CALL_PATH = PKG_DIR / "_call.so"

ARCH = "gfx950"
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fvisibility=hidden",
    "-Wall",
    "-Wno-unused-function",
    # scalar fp32 code only: keep the compiler from forming packed-fp32 instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(exe).exists():
        raise RuntimeError("hipcc not found; libffnk.so cannot be built")
    return exe


def _compile(src: Path) -> Path:
    obj = OBJ_DIR / (src.stem + ".o")
    cmd = [_hipcc(), *HIPCC_FLAGS, "-c", str(src), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in proc.stderr.splitlines() if noise not in l)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def call_command(src: Path, out: Path) -> list:
    """g++ on a CPython extension over torch's headers (host code only)."""
    import torch
    from torch.utils.cpp_extension import include_paths, library_paths

    cmd = [shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-I{sysconfig.get_paths()['include']}"]
    cmd += [flag for p in include_paths("cuda") for flag in ("-isystem", p)] + [str(src), "-o", str(out)]
    return cmd + [f"-L{p}" for p in library_paths()] + ["-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"]


def _compile_call() -> Path:
    """csrc/call.cpp -> _call.so."""
    tmp = CALL_PATH.with_suffix(".so.tmp")
    proc = subprocess.run(call_command(CSRC / "call.cpp", tmp), capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"g++ failed on call.cpp:\n{proc.stderr}")
    if proc.stderr.strip():
        sys.stderr.write(proc.stderr + "\n")
    os.replace(tmp, CALL_PATH)
    return CALL_PATH


def build_library(jobs: int | None = None, verbose: bool = True) -> Path:
    """Compile csrc/*.hip and link libffnk.so; compile _call.so beside them.  Always recompiles."""
    OBJ_DIR.mkdir(parents=True, exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    if not sources:
        raise RuntimeError(f"no .hip sources under {CSRC}")
    jobs = jobs or min(len(sources), os.cpu_count() or 4, 16)
    if verbose:
        print(f"[ffn_kernel_amd.build] hipcc {ARCH}: {len(sources)} files, {jobs} jobs", flush=True)
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        call = pool.submit(_compile_call)
        objs = list(pool.map(_compile, sources))
        call.result()
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{proc.stderr}")
    os.replace(tmp, LIB_PATH)
    if verbose:
        print(f"[ffn_kernel_amd.build] wrote {LIB_PATH} ({LIB_PATH.stat().st_size >> 10} KiB)", flush=True)
    return LIB_PATH


if __name__ == "__main__":
    build_library()
