"""Builds libember_ops.so (the gfx950 HIP kernels behind the C ABI in include/ember_ops.h) and
_fast.so (the ops' native host path, a CPython extension over torch's C++ API).

`python -m emberserve_amd.build` or `build()` compiles every `csrc/*.hip` with hipcc for
gfx950, in parallel, and links the shared library next to this file, where `_lib` loads it;
csrc/fast_ops.cpp is compiled by the host compiler beside them.
No GPU is needed: hipcc cross-compiles.
"""

from __future__ import annotations

import concurrent.futures
import os
import shutil
import subprocess
import sys
import sysconfig
import warnings
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
BUILD_DIR = PKG_DIR / "_build"
LIB_PATH = PKG_DIR / "libember_ops.so"
FAST_PATH = PKG_DIR / "_fast.so"
ARCH = "gfx950"

# -ffp-contract=off: a*b+c stays two rounded operations, as in the reference's separate
# element-wise tensor ops (the rope and norm parity depends on it).
# -packed-fp32-ops: keep hipcc from forming packed fp32 instructions.
# -amdgpu-mfma-vgpr-form: MFMA accumulators in ordinary VGPRs, so the decode kernel's
# online-softmax rescale of its accumulators needs no accvgpr copies.
HIP_FLAGS = [
    "-O3", f"--offload-arch={ARCH}", "-std=c++17", "-fPIC", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-mllvm", "-amdgpu-mfma-vgpr-form=1",
    "-Wall", "-Wno-unused-command-line-argument",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found (set HIPCC or install ROCm)")


def _compile(src: Path, obj: Path) -> None:
    cmd = [hipcc(), *HIP_FLAGS, "-c", str(src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{res.stderr}")


def _build_fast() -> None:
    """Compiles csrc/fast_ops.cpp into _fast.so. Where a C++ compiler or the headers are not
    installed there is no native host path (nor a stale one): the library does without it."""
    import torch

    cxx = os.environ.get("CXX") or shutil.which("g++") or shutil.which("c++")
    rocm = Path(hipcc()).resolve().parent.parent
    inc = Path(torch.__file__).resolve().parent / "include"
    lib = inc.parent / "lib"
    headers = [Path(sysconfig.get_paths()["include"]) / "Python.h", inc / "torch/csrc/autograd/python_variable.h"]
    missing = ["a C++ compiler (set CXX)"] * (cxx is None) + [str(h) for h in headers if not h.exists()]
    if missing:
        FAST_PATH.unlink(missing_ok=True)
        warnings.warn(f"emberserve_amd: _fast.so is not built, {' and '.join(missing)} not found", RuntimeWarning)
        return
    tmp = FAST_PATH.with_suffix(".so.tmp")
    cmd = [*cxx.split(), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-I{inc}",
           f"-I{inc / 'torch/csrc/api/include'}", f"-I{sysconfig.get_paths()['include']}", f"-I{rocm / 'include'}",
           str(CSRC / "fast_ops.cpp"), "-o", str(tmp), f"-L{lib}", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10",
           "-lc10_hip"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{cxx} failed on fast_ops.cpp:\n{res.stderr}")
    os.replace(tmp, FAST_PATH)


def build(verbose: bool = False) -> Path:
    """Compiles every kernel source, links `libember_ops.so` and builds `_fast.so`; returns
    the library's path."""
    BUILD_DIR.mkdir(exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    objs = [BUILD_DIR / (s.stem + ".o") for s in sources]
    workers = min(len(sources), int(os.environ.get("MAX_JOBS", os.cpu_count() or 4)), 16)
    with concurrent.futures.ThreadPoolExecutor(max_workers=max(1, workers)) as ex:
        futs = [ex.submit(_build_fast)] + [ex.submit(_compile, s, o) for s, o in zip(sources, objs)]
        for f in futs:
            f.result()
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, LIB_PATH)  # atomic: a process that already mapped the old file keeps it
    if verbose:
        print(f"built {LIB_PATH}", file=sys.stderr)
    return LIB_PATH


if __name__ == "__main__":
    build(verbose=True)
