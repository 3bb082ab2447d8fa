"""Builds liblookupffn_hip.so (the C-ABI kernel library) for gfx950 with hipcc, and _host.so (the layer's host path in C++,
csrc/host.cpp, against the installed torch) with g++.

Run as ``python -m lookupffn_amd._build``.  hipcc cross-compiles, so no GPU is
needed.  Both land next to this file so that they are found in-tree.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG_DIR, "csrc")
LIB_NAME = "liblookupffn_hip.so"
LIB_PATH = os.path.join(PKG_DIR, LIB_NAME)
HOST_PATH = os.path.join(PKG_DIR, "_host.so")
SOURCES = ["fht.hip", "code_score.hip", "gather.hip", "lookup_gather.hip", "lookup_gather_pair.hip", "lookup_gather_quad.hip", "lookup_scatter.hip", "lookup_scatter_sorted.hip", "lookup_inner.hip", "lookup_inner_quad.hip", "bh4_block.hip", "bh4_split.hip", "bh4_wgrad.hip", "fht_bwd.hip", "layer_norm.hip", "linear.hip", "attention.hip"]

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-munsafe-fp-atomics",
    # no packed-fp32 instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found: the kernel library can only be built in a ROCm image")
    return exe


def _build_host() -> None:
    import torch
    root = os.path.dirname(torch.__file__)
    includes = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
                "/opt/rocm/include", sysconfig.get_paths()["include"]]
    tmp = HOST_PATH + ".tmp"
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}", f'-DLFFN_TORCH_VERSION="{torch.__version__}"',
           *[a for d in includes for a in ("-isystem", d)], os.path.join(CSRC, "host.cpp"), "-o", tmp,
           "-L" + os.path.join(root, "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed on host.cpp:\n{res.stderr[-8000:]}")
    os.replace(tmp, HOST_PATH)


def build_library(verbose: bool = False) -> str:
    hipcc = _hipcc()
    objdir = os.path.join(CSRC, "build")
    os.makedirs(objdir, exist_ok=True)
    missing = [s for s in SOURCES if not os.path.exists(os.path.join(CSRC, s))]
    if missing:
        raise RuntimeError(f"kernel sources missing from {CSRC}: {', '.join(missing)}")
    srcs = list(SOURCES)

    def compile_one(src: str) -> str:
        obj = os.path.join(objdir, src.replace(".hip", ".o"))
        cmd = [hipcc, *HIPCC_FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
        res = subprocess.run(cmd, capture_output=True, text=True)
        err = "\n".join(l for l in res.stderr.splitlines() if "packed-fp32-ops" not in l)
        if res.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{err}")
        if verbose and err.strip():
            print(err, file=sys.stderr)
        return obj

    with ThreadPoolExecutor(max_workers=5) as ex:
        host = ex.submit(_build_host)
        objs = list(ex.map(compile_one, srcs))
        host.result()
    tmp = LIB_PATH + ".tmp"
    res = subprocess.run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", tmp],
                         capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, LIB_PATH)
    return LIB_PATH


if __name__ == "__main__":
    print(build_library(verbose=True))
