"""Build libverl_amd.so (gfx950) from the HIP sources in this directory, and _torch_ops.so over it.

    python -m verl_amd.csrc.build        # or: python verl_amd/csrc/build.py

hipcc cross-compiles without a GPU.  The library links only the HIP runtime; it is loaded with
ctypes after ``import torch`` so that the runtime torch already mapped is the one it binds to.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.dirname(HERE)
LIB_DIR = os.path.join(PKG, "lib")
LIB_PATH = os.path.join(LIB_DIR, "libverl_amd.so")
OPS_PATH = os.path.join(LIB_DIR, "_torch_ops.so")
SOURCES = ["runtime.hip", "lce.hip", "policy_math.hip", "gae.hip", "returns_scan.hip", "otb.hip", "metrics.hip", "rollout_corr.hip", "response_window.hip", "cov_select.hip", "row_softmax.hip"]
HEADERS = ["common.h", "gemm_core.h", "rowchunk.h", os.path.join("..", "..", "include", "verl_amd.h")]

OPS_SOURCE = "torch_ops.cpp"   # host code only: torch's C++ interface over the C ABI

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-mcode-object-version=5",
    # keep the compiler from forming packed-fp32 VALU ops
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    # the LDS-direct loads set M0 from inline assembly and say so in the clobber list
    "-Wno-inline-asm",
]


def _compile(src: str) -> str:
    obj = os.path.join(HERE, "build", os.path.splitext(src)[0] + ".o")
    os.makedirs(os.path.dirname(obj), exist_ok=True)
    cmd = [HIPCC, *FLAGS, "-c", os.path.join(HERE, src), "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in res.stderr.splitlines() if noise not in l)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _compile_ops() -> str:
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    obj = os.path.join(HERE, "build", os.path.splitext(OPS_SOURCE)[0] + ".o")
    os.makedirs(os.path.dirname(obj), exist_ok=True)
    include = [*cpp_extension.include_paths("cuda"), sysconfig.get_paths()["include"]]
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-DUSE_ROCM=1", "-D__HIP_PLATFORM_AMD__=1",
           "-DTORCH_EXTENSION_NAME=_torch_ops", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *(arg for path in include for arg in ("-isystem", path)), "-c", os.path.join(HERE, OPS_SOURCE), "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed on {OPS_SOURCE}:\n{res.stderr}")
    return obj


def link_ops(obj: str) -> None:
    from torch.utils import cpp_extension

    lib_dirs = [*cpp_extension.library_paths(), LIB_DIR]
    cmd = [os.environ.get("CXX", "g++"), "-shared", "-fPIC", obj, *(f"-L{path}" for path in lib_dirs), "-lverl_amd",
           "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch", "-ltorch_python", "-lamdhip64",
           "-Wl,-rpath,$ORIGIN", "-o", OPS_PATH]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link of {os.path.basename(OPS_PATH)} failed:\n{res.stderr}")


def build(verbose: bool = True) -> str:
    """Compile every source and link the shared library; always recompiles."""
    with ThreadPoolExecutor(max_workers=min(5, len(SOURCES))) as pool:
        ops = pool.submit(_compile_ops)
        objs = list(pool.map(_compile, SOURCES))
        ops_obj = ops.result()
    os.makedirs(LIB_DIR, exist_ok=True)
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", LIB_PATH]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    link_ops(ops_obj)
    if verbose:
        for path in (LIB_PATH, OPS_PATH):
            print(f"built {path} ({os.path.getsize(path) >> 10} KiB)")
    return LIB_PATH


if __name__ == "__main__":
    build()
