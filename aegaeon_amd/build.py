"""Build libaegkv.so (HIP, gfx950, with hipcc) and _hostargs.so (host C++) in-tree.

The library is a plain C-ABI shared object; it links against the HIP
runtime by SONAME (libamdhip64.so.7), so inside a process that has already
imported torch it binds to the runtime torch loaded.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sysconfig
import warnings
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
REPO_DIR = PKG_DIR.parent
CSRC = PKG_DIR / "csrc"
LIB_PATH = PKG_DIR / "libaegkv.so"
HOSTARGS_PATH = PKG_DIR / "_hostargs.so"
ARCH = os.environ.get("AEGKV_OFFLOAD_ARCH", "gfx950")

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    # packed FP32 instructions stay disabled in every HIP build here
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found: the HIP toolchain is required to build libaegkv")


def build_hostargs(verbose: bool = False) -> Path:
    """Compile csrc/hostargs.cpp into aegaeon_amd/_hostargs.so (always
    rebuilds): a Python module over torch's C++ interface."""
    import torch
    from torch.utils.cpp_extension import include_paths, library_paths

    tmp = HOSTARGS_PATH.with_suffix(".so.tmp")
    cmd = [
        os.environ.get("CXX") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall",
        f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
        f'-DAEGKV_TORCH_VERSION="{torch.__version__}"',
        *[f"-isystem{p}" for p in (*include_paths(), sysconfig.get_paths()["include"])],
        str(CSRC / "hostargs.cpp"),
        *[f"-L{p}" for p in library_paths()],
        "-ltorch_python", "-ltorch_cpu", "-lc10",
        "-o", str(tmp),
    ]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed ({res.returncode}):\n{res.stderr}")
    os.replace(tmp, HOSTARGS_PATH)
    return HOSTARGS_PATH


def build(verbose: bool = False) -> Path:
    """Compile csrc/aegkv.hip, csrc/fence.hip and csrc/plan.cpp into
    aegaeon_amd/libaegkv.so, then csrc/hostargs.cpp (always rebuilds). The
    library needs neither g++ nor torch's headers; where those fail, the
    Python package reads its arguments without _hostargs.so."""
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [
        hipcc(),
        *HIPCC_FLAGS,
        f"-I{REPO_DIR / 'include'}",
        str(CSRC / "aegkv.hip"),
        str(CSRC / "fence.hip"),
        str(CSRC / "plan.cpp"),
        "-o",
        str(tmp),
    ]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed ({res.returncode}):\n{res.stderr}")
    os.replace(tmp, LIB_PATH)
    try:
        build_hostargs(verbose)
    except (ImportError, OSError, RuntimeError) as exc:
        HOSTARGS_PATH.unlink(missing_ok=True)  # no stale one beside a new library
        warnings.warn(f"aegaeon_amd/_hostargs.so was not built: {exc}", RuntimeWarning,
                      stacklevel=2)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose=True))
