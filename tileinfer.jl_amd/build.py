"""Build libtileinfer_hip.so for gfx950 from csrc/*.hip with hipcc, and the Python package's
native call path _calls.so from csrc/py_calls.cpp with g++ (no GPU needed). The library needs
hipcc only; _calls.so is left out where torch's headers are not there.

    python tileinfer.jl_amd/build.py

Each .hip file compiles to an object under _build/ in parallel, then links into
tileinfer_hip/libtileinfer_hip.so next to the Python host package, where the package,
the tests and bench.py load it.
"""
from __future__ import annotations

import concurrent.futures as cf
import glob
import os
import subprocess
import sys

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
OUT = os.path.join(PKG, "tileinfer_hip", "libtileinfer_hip.so")
CALLS = os.path.join(PKG, "tileinfer_hip", "_calls.so")
BUILD = os.path.join(ROOT, "_build")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # Packed FP32 (v_pk_*_f32) is off for every kernel: hipcc would otherwise form it.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", os.path.join(ROOT, "include"), "-I", CSRC,
    "-Wall", "-Wno-unused-function",
]


# MFMA accumulators in VGPRs (not AGPRs): no AGPR<->VGPR copies around the softmax
# rescale.
VGPR_FORM = ["-mllvm", "-amdgpu-mfma-vgpr-form"]


def _compile(src: str) -> str:
    obj = os.path.join(BUILD, os.path.basename(src).replace(".hip", ".o"))
    cmd = [HIPCC, *FLAGS, *VGPR_FORM, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError(f"hipcc failed on {src}")
    return obj


def _build_calls() -> bool:
    """_calls.so: a CPython module against torch's headers (host code only). False where a ROCm
    torch, its headers, Python's or g++ are not there: the package then calls the library through ctypes."""
    import shutil
    import sysconfig

    if os.path.exists(CALLS):
        os.remove(CALLS)   # never one of another torch
    try:
        import torch
    except ImportError:
        return False
    if not torch.version.hip:
        return False
    inc = os.path.join(os.path.dirname(torch.__file__), "include")
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    needed = (os.path.join(inc, "torch", "csrc", "autograd", "python_variable.h"),
              os.path.join(sysconfig.get_paths()["include"], "Python.h"))
    if not all(map(os.path.exists, needed)) or not shutil.which("g++"):
        return False
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           "-I", os.path.join(ROOT, "include"), "-isystem", inc,
           "-isystem", os.path.join(inc, "torch", "csrc", "api", "include"), "-isystem", sysconfig.get_paths()["include"],
           "-isystem", "/opt/rocm/include",
           f'-DBUILT_FOR="torch {torch.__version__}, Python {sys.version_info[0]}.{sys.version_info[1]}"',
           os.path.join(CSRC, "py_calls.cpp"), "-o", CALLS, "-L", lib,
           "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip", f"-Wl,-rpath,{lib}"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("g++ failed on py_calls.cpp")
    return True


def build(verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs) + 1)) as ex:
        calls = ex.submit(_build_calls)
        objs = list(ex.map(_compile, srcs))
        cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", OUT, *objs]
        subprocess.run(cmd, check=True)
    if not calls.result():
        sys.stderr.write("_calls.so not built (no torch with headers, Python headers or g++): ops go through ctypes\n")
    if verbose:
        print("built", OUT, CALLS if calls.result() else "")
    return OUT


if __name__ == "__main__":
    build(verbose=True)
