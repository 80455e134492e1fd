"""Compile the native code of this package: ``liblastkv_amd.so`` and the extension module ``_host.so``.

Every ``csrc/*.hip`` file is compiled with hipcc for gfx950 only, then linked into one shared
library exporting the C ABI declared in ``include/lastkv_amd.h``.  ``csrc/host.cpp`` (host code
only) becomes the module ``lastkv_amd._host`` against the installed torch.  Run as
``python -m lastkv_amd.build``.
"""

from __future__ import annotations

import concurrent.futures
import os
import pathlib
import shutil
import subprocess
import sys
import sysconfig

PKG_DIR = pathlib.Path(__file__).resolve().parent
REPO_DIR = PKG_DIR.parent
CSRC = PKG_DIR / "csrc"
LIB_NAME = "liblastkv_amd.so"
LIB_PATH = PKG_DIR / LIB_NAME
HOST_PATH = PKG_DIR / "_host.so"
OBJ_DIR = PKG_DIR / "_build"

ARCH = "gfx950"
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Wno-unused-function",
    # packed fp32 arithmetic stays disabled: it has produced silent miscomputations on this pool
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{REPO_DIR / 'include'}",
]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; the ROCm toolchain is required to build lastkv_amd")
    return exe


def _compile(src: pathlib.Path, verbose: bool) -> pathlib.Path:
    obj = OBJ_DIR / (src.stem + ".o")
    cmd = [_hipcc(), *HIPCC_FLAGS, "-c", str(src), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    noise = "not a recognized feature for this target"
    log = "\n".join(line for line in (proc.stdout + proc.stderr).splitlines() if noise not in line)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{log}")
    if verbose and log.strip():
        print(log, file=sys.stderr)
    return obj


def _build_host() -> None:
    import torch

    root = pathlib.Path(torch.__file__).resolve().parent
    includes = [root / "include", root / "include/torch/csrc/api/include", sysconfig.get_paths()["include"],
                pathlib.Path(_hipcc()).resolve().parents[1] / "include"]
    tmp = HOST_PATH.with_suffix(".so.tmp")
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *(x for i in includes for x in ("-isystem", str(i))), str(CSRC / "host.cpp"), "-o", str(tmp),
           f"-L{root / 'lib'}", "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"compiling host.cpp failed:\n{proc.stdout}{proc.stderr}")
    os.replace(tmp, HOST_PATH)


def build(verbose: bool = False) -> pathlib.Path:
    """Compile every HIP source and link ``liblastkv_amd.so``, and build ``_host.so``; returns the library's path."""

    OBJ_DIR.mkdir(exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    if not sources:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, len(sources) + 1)) as pool:
        host = pool.submit(_build_host)
        objs = list(pool.map(lambda s: _compile(s, verbose), sources))
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{proc.stdout}{proc.stderr}")
    os.replace(tmp, LIB_PATH)
    host.result()  # (after the link: the library is complete without the launch module)
    return LIB_PATH


if __name__ == "__main__":
    path = build(verbose=True)
    print(path)
