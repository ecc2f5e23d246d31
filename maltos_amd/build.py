"""Build libmaltos_hip.so (gfx950) from maltos_amd/csrc/*.hip with hipcc, and the torch extension _torch_ops.so over it
from maltos_amd/csrc/torch/*.cpp with the host compiler.

    python -m maltos_amd.build            # compile every source and link, in-tree

The library is a plain C-ABI shared object (see include/maltos_hip.h); it links only against the
HIP runtime, not against torch, so C/C++ hosts can bind it as well.
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
LIB_PATH = PKG_DIR / "libmaltos_hip.so"
EXT_SRC = CSRC / "torch"
EXT_PATH = PKG_DIR / "_torch_ops.so"
OBJ_DIR = PKG_DIR / "csrc" / "build"

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-math-errno",
    # packed fp32 VALU forms are kept off for every kernel in this library
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _hipcc() -> str:
    found = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(found):
        raise RuntimeError("hipcc not found; the HIP kernels cannot be built")
    return found


def _compile_one(src: Path, verbose: bool) -> Path:
    obj = OBJ_DIR / (src.stem + ".o")
    cmd = [_hipcc(), *HIPCC_FLAGS, "-c", str(src), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{proc.stderr}")
    if verbose:
        print(f"[maltos_amd.build] compiled {src.name}", flush=True)
    return obj


def _torch_dir() -> Path:
    import torch

    return Path(torch.__file__).resolve().parent


def _run(cmd: list[str], what: str) -> None:
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{proc.stderr}")


def _compile_ext(src: Path, verbose: bool) -> Path:
    obj = OBJ_DIR / (src.stem + ".ext.o")
    inc = _torch_dir() / "include"
    rocm = Path(_hipcc()).resolve().parents[1] / "include"
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_EXTENSION_NAME=_torch_ops",
          "-DTORCH_API_INCLUDE_EXTENSION_H", f"-I{inc}", f"-I{inc}/torch/csrc/api/include", "-isystem", str(rocm), f"-I{sysconfig.get_paths()['include']}",
          "-c", str(src), "-o", str(obj)], f"compiling {src.name}")
    if verbose:
        print(f"[maltos_amd.build] compiled torch/{src.name}", flush=True)
    return obj


def build(verbose: bool = True, jobs: int | None = None) -> Path:
    """Compile every source and link the library and the torch extension; always rebuilds."""
    OBJ_DIR.mkdir(parents=True, exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    if not sources:
        raise RuntimeError(f"no .hip sources under {CSRC}")
    ext_sources = sorted(EXT_SRC.glob("*.cpp"))
    jobs = jobs or min(8, len(sources) + len(ext_sources), os.cpu_count() or 1)
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        ext_objs = pool.map(lambda s: _compile_ext(s, verbose), ext_sources)
        objs = list(pool.map(lambda s: _compile_one(s, verbose), sources))
        ext_objs = list(ext_objs)
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    _run(cmd, "linking the library")
    os.replace(tmp, LIB_PATH)
    tmp = EXT_PATH.with_suffix(".so.tmp")
    libs = _torch_dir() / "lib"
    _run(["g++", "-shared", "-fPIC", "-o", str(tmp), *map(str, ext_objs), f"-L{PKG_DIR}", "-l:libmaltos_hip.so", "-Wl,-rpath,$ORIGIN", f"-L{libs}",
          f"-Wl,-rpath,{libs}", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip"], "linking the torch extension")
    os.replace(tmp, EXT_PATH)
    if verbose:
        print(f"[maltos_amd.build] linked {LIB_PATH} and {EXT_PATH.name}", flush=True)
    return LIB_PATH


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
