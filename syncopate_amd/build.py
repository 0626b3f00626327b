"""Build libsyncopate_hip.so (gfx950) in-tree with hipcc, and the _native extension with g++.

    python -m syncopate_amd.build            # compile every csrc/*.hip and link; compile csrc/launch.cpp

hipcc cross-compiles for gfx950 without a GPU.  The library is linked without
an rpath to a ROCm tree: at run time ``syncopate_amd._lib`` imports torch first,
so the HIP runtime torch already loaded (same soname) is the one the kernels
launch on and torch's stream handles are valid in it.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

CSRC = Path(__file__).resolve().parent / "csrc"
LIB_NAME = "libsyncopate_hip.so"
LIB_PATH = CSRC / LIB_NAME
NATIVE_PATH = CSRC.parent / "_native.so"
ARCH = "gfx950"

# -packed-fp32-ops is off: hipcc must not form v_pk_*_f32 from scalar float code.
DEVICE_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; cannot build libsyncopate_hip.so")
    return exe


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip"))


def _run(cmd: list[str]) -> None:
    proc = subprocess.run(cmd, capture_output=True, text=True)
    # the host pass of hipcc does not know the AMDGPU target feature and says so
    err = "\n".join(
        line for line in proc.stderr.splitlines() if "packed-fp32-ops" not in line
    )
    if proc.returncode != 0:
        raise RuntimeError(f"command failed ({proc.returncode}): {' '.join(cmd)}\n{proc.stdout}\n{err}")
    if err.strip():
        print(err, file=sys.stderr)


def build_native() -> Path:
    """Compile csrc/launch.cpp, host code against torch's headers, into the extension module syncopate_amd._native."""
    import torch

    home = Path(torch.__file__).resolve().parent
    tmp = NATIVE_PATH.with_suffix(".so.tmp")
    _run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-isystem{home / 'include'}",
          f"-isystem{home / 'include/torch/csrc/api/include'}", f"-isystem{Path(_hipcc()).resolve().parents[1] / 'include'}",
          f"-I{sysconfig.get_paths()['include']}", str(CSRC / "launch.cpp"), f"-L{home / 'lib'}", "-ltorch_python", "-ltorch_cpu",
          "-ltorch", "-lc10", "-lc10_hip", "-lamdhip64", "-o", str(tmp)])
    os.replace(tmp, NATIVE_PATH)
    return NATIVE_PATH


def build_library(jobs: int = 4, verbose: bool = True) -> Path:
    """Compile all HIP sources and link the shared library, and the extension beside it; always recompiles."""
    hipcc = _hipcc()
    obj_dir = CSRC / "build"
    obj_dir.mkdir(exist_ok=True)
    srcs = sources()
    if not srcs:
        raise RuntimeError(f"no .hip sources under {CSRC}")

    def compile_one(src: Path) -> Path:
        obj = obj_dir / (src.stem + ".o")
        _run([hipcc, *DEVICE_FLAGS, "-c", str(src), "-o", str(obj)])
        if verbose:
            print(f"[syncopate_amd.build] compiled {src.name}")
        return obj

    with ThreadPoolExecutor(max_workers=max(1, jobs)) as pool:
        native = pool.submit(build_native)
        objs = list(pool.map(compile_one, srcs))
        native.result()

    tmp = LIB_PATH.with_suffix(".so.tmp")
    _run([hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)])
    os.replace(tmp, LIB_PATH)
    if verbose:
        print(f"[syncopate_amd.build] linked {LIB_PATH}")
    return LIB_PATH


if __name__ == "__main__":
    build_library()
