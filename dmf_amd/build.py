"""Builds dmf_amd/libdmf_attn.so (gfx950) from dmf_amd/csrc with hipcc, and the native host path dmf_amd/_host*.so on top of it.

Run as ``python -m dmf_amd.build``.  Both are built in-tree next to this
file so that they travel with the source tree.
"""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libdmf_attn.so")
HOST = os.path.join(HERE, "_host" + sysconfig.get_config_var("EXT_SUFFIX"))
SOURCES = ["attn_fwd.hip", "attn_fwd_bf16.hip", "attn_fwd_small.hip", "attn_bwd.hip", "attn_bwd_bf16.hip", "dmf_attn_abi.hip", "block_ops.hip", "modulation.hip", "linear.hip"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden",
    # packed fp32 VALU ops are kept off for every HIP translation unit
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _compile(src: str, objdir: str) -> str:
    obj = os.path.join(objdir, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC, *FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{err}")
    if err.strip():
        print(err, file=sys.stderr)
    return obj


def _build_host(objdir: str) -> str:
    """The native host path: a CPython extension against the installed torch, linked to the kernel library beside it."""
    import torch

    root = os.path.dirname(torch.__file__)
    inc, lib = os.path.join(root, "include"), os.path.join(root, "lib")
    obj = os.path.join(objdir, "host.o")
    rocm = os.path.dirname(os.path.dirname(HIPCC))
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM",
           "-DTORCH_API_INCLUDE_EXTENSION_H", "-DTORCH_EXTENSION_NAME=_host",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-I" + os.path.join(CSRC, "stub"), "-I" + inc,
           "-I" + os.path.join(inc, "torch", "csrc", "api", "include"), "-I" + os.path.join(rocm, "include"),
           "-I" + sysconfig.get_path("include"), "-c", os.path.join(CSRC, "host.cpp"), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed for host.cpp:\n{r.stderr}")
    return obj


def _link_host(obj: str) -> str:
    import torch

    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    cmd = ["g++", "-shared", "-fPIC", "-o", HOST, obj, "-L" + lib, "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu", "-ltorch_hip",
           "-ltorch_python", "-L" + HERE, "-l:" + os.path.basename(LIB), "-Wl,-rpath,$ORIGIN", "-Wl,-rpath," + lib]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link of the host path failed:\n{r.stderr}")
    return HOST


def build(verbose: bool = True) -> str:
    objdir = os.path.join(HERE, "build")
    os.makedirs(objdir, exist_ok=True)
    with ThreadPoolExecutor(max_workers=len(SOURCES) + 1) as ex:
        host = ex.submit(_build_host, objdir)
        objs = list(ex.map(lambda s: _compile(s, objdir), SOURCES))
        host = host.result()
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-Wl,-soname," + os.path.basename(LIB), "-o", LIB, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    _link_host(host)
    if verbose:
        print(f"built {LIB} and {HOST}")
    return LIB


if __name__ == "__main__":
    build()
