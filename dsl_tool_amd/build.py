"""Build ``dsl_tool_amd/_lib/libdsl_gemm.so`` for gfx950 with hipcc.

Usage: ``python -m dsl_tool_amd.build`` (compiles every ``csrc/*.hip``
translation unit in parallel, then links one shared library, and beside it
``dsl_fast.so``, the CPython extension that calls it on torch tensors).  The
build is in-tree so the libraries travel with the source tree.
"""
from __future__ import annotations

import concurrent.futures as cf
import glob
import os
import shutil
import subprocess
import sys
import sysconfig

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
OUT_DIR = os.path.join(PKG, "_lib")
OBJ_DIR = os.path.join(OUT_DIR, "obj")
LIB = os.path.join(OUT_DIR, "libdsl_gemm.so")
FAST_SRC = os.path.join(CSRC, "fastcall.cpp")
FAST = os.path.join(OUT_DIR, "dsl_fast.so")
ARCH = os.environ.get("DSL_OFFLOAD_ARCH", "gfx950")

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    # packed-FP32 VALU ops are kept out of the generated code on purpose
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
    "-Wall", "-Wno-unused-function",
]


def _compile(src: str) -> str:
    obj = os.path.join(OBJ_DIR, os.path.basename(src) + ".o")
    cmd = [HIPCC, *FLAGS, "-c", src, "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{res.stdout}\n{res.stderr}")
    return obj


def _run(cmd: list, what: str) -> None:
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{res.stdout}\n{res.stderr}")


def _compile_fast() -> str:
    """The host-only extension (no device code), against torch's headers."""
    import torch
    inc = os.path.join(os.path.dirname(torch.__file__), "include")
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(HIPCC)))
    obj = os.path.join(OBJ_DIR, "fastcall.cpp.o")
    _run([shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}", "-I" + os.path.join(ROOT, "include"),
          "-isystem", inc, "-isystem", os.path.join(inc, "torch", "csrc", "api", "include"),
          "-isystem", sysconfig.get_paths()["include"], "-isystem", os.path.join(rocm, "include"),
          "-isystem", "/opt/rocm/include", "-Wall", "-c", FAST_SRC, "-o", obj], "g++ fastcall.cpp")
    return obj


def _link_fast(obj: str) -> None:
    import torch
    tl = os.path.join(os.path.dirname(torch.__file__), "lib")
    tmp = FAST + ".tmp"
    _run([shutil.which("g++") or "g++", "-shared", obj, "-o", tmp, "-L" + OUT_DIR, "-l:libdsl_gemm.so",
          "-L" + tl, "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip",
          "-Wl,-rpath,$ORIGIN"], "link dsl_fast.so")
    os.replace(tmp, FAST)


def build(verbose: bool = True) -> str:
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    with cf.ThreadPoolExecutor(max_workers=min(len(srcs) + 1, os.cpu_count() or 4)) as ex:
        fast = ex.submit(_compile_fast)
        objs = list(ex.map(_compile, srcs))
        fast_obj = fast.result()
    tmp = LIB + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-Wl,-soname,libdsl_gemm.so", *objs, "-o", tmp]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, LIB)
    _link_fast(fast_obj)
    if verbose:
        print(f"built {LIB} and {FAST}")
    return LIB


if __name__ == "__main__":
    try:
        build()
    except RuntimeError as exc:
        print(exc, file=sys.stderr)
        sys.exit(1)
