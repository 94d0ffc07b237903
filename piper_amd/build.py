"""Build libpiper_amd.so (gfx950 HIP kernels + C ABI) with hipcc and _pk_host.so (the native host path
of the torch operators, linked against it) with g++, both in-tree.

Usage: ``python -m piper_amd.build`` or ``piper_amd.build.build_library()``.
The libraries are written next to this file so that they travel with the source tree.
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
LIB_PATH = PKG_DIR / "libpiper_amd.so"
HOST_PATH = PKG_DIR / "_pk_host.so"
SOURCES = ["bucket.hip", "route.hip", "permute.hip", "grouped_gemm.hip", "decode.hip", "timing.hip"]

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fvisibility=hidden",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; cannot build libpiper_amd.so")
    return exe


def _run(cmd: list[str]) -> None:
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    # hipcc's host pass warns that it does not know the packed-fp32-ops feature; harmless.
    out = "\n".join(l for l in proc.stdout.splitlines() if "packed-fp32-ops" not in l)
    if proc.returncode != 0:
        raise RuntimeError(f"command failed ({proc.returncode}): {' '.join(cmd)}\n{out}")
    if out.strip():
        print(out, file=sys.stderr)


def _host_commands(obj: Path, out: Path) -> tuple[list[str], list[str]]:
    """Compile and link commands of the torch extension module (no device code in it)."""
    import torch

    root = Path(torch.__file__).resolve().parent
    inc = [root / "include", root / "include" / "torch" / "csrc" / "api" / "include", Path("/opt/rocm/include"),
           Path(sysconfig.get_paths()["include"])]
    cxx = shutil.which("g++") or "g++"
    compile_cmd = [cxx, "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Wall", "-Wno-unused-function", "-D__HIP_PLATFORM_AMD__=1",
                   "-DUSE_ROCM=1", "-DTORCH_EXTENSION_NAME=_pk_host", "-DTORCH_API_INCLUDE_EXTENSION_H",
                   f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *[f"-isystem{i}" for i in inc],
                   "-c", str(CSRC / "host.cpp"), "-o", str(obj)]
    link_cmd = [cxx, "-shared", "-o", str(out), str(obj), f"-L{root / 'lib'}", "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch",
                "-ltorch_python", f"-L{PKG_DIR}", "-l:libpiper_amd.so", "-Wl,-rpath,$ORIGIN"]
    return compile_cmd, link_cmd


def build_library(verbose: bool = False) -> Path:
    """Compile every source and link both shared libraries.  Always rebuilds."""
    hipcc = _hipcc()
    obj_dir = PKG_DIR / "build"
    obj_dir.mkdir(exist_ok=True)
    objs = []
    cmds = []
    for src in SOURCES:
        obj = obj_dir / (src.replace(".hip", ".o"))
        objs.append(str(obj))
        cmds.append([hipcc, *HIPCC_FLAGS, "-c", str(CSRC / src), "-o", str(obj)])
    host_obj, host_tmp = obj_dir / "host.o", HOST_PATH.with_suffix(".so.tmp")
    host_compile, host_link = _host_commands(host_obj, host_tmp)
    cmds.append(host_compile)
    if verbose:
        for c in cmds:
            print(" ".join(c))
    with ThreadPoolExecutor(max_workers=min(6, len(cmds))) as pool:
        list(pool.map(_run, cmds))
    tmp = LIB_PATH.with_suffix(".so.tmp")
    _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(tmp), *objs])
    os.replace(tmp, LIB_PATH)
    _run(host_link)
    os.replace(host_tmp, HOST_PATH)
    return LIB_PATH


if __name__ == "__main__":
    print(build_library(verbose=True))
