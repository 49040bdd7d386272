"""Builds libprime_moe_hip.so (the C-ABI library, hipcc for gfx950) and _torch_ops.so (the package's host side on
top of it: checks, allocation, op registration; plain C++ against torch's headers) in-tree.

Usage: ``python -m prime_moe.build`` (with ``prime-flash-moe_amd`` on ``sys.path``) or
``python prime-flash-moe_amd/prime_moe/build.py``.  Both land next to this file, where
``prime_moe`` finds them; nothing is installed outside the tree.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "csrc")
OBJ_DIR = os.path.join(CSRC, "build")
LIB_NAME = "libprime_moe_hip.so"
LIB_PATH = os.path.join(HERE, LIB_NAME)
SOURCES = ["api.hip", "moe_align.hip", "route.hip", "quantize_mx.hip", "fused_moe.hip", "fused_moe_bf16.hip"]
ARCH = "gfx950"
EXT_SOURCE = "torch_ops.cpp"
EXT_PATH = os.path.join(HERE, "_torch_ops.so")

# Packed-fp32 VALU forms are switched off for every device compile.
# Private arrays are never moved into LDS by the compiler: the kernels budget LDS themselves.
DEVICE_FLAGS = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                "-mllvm", "-disable-promote-alloca-to-lds"]


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; the prime_moe HIP library cannot be built")
    return exe


def _compile(src: str, verbose: bool) -> str:
    obj = os.path.join(OBJ_DIR, os.path.splitext(src)[0] + ".o")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-munsafe-fp-atomics",
           *DEVICE_FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{res.stdout}\n{res.stderr}")
    if verbose and res.stderr.strip():
        # the host pass reports the device-only target feature as unknown; harmless
        lines = [l for l in res.stderr.splitlines() if "packed-fp32-ops" not in l and l.strip()]
        if lines:
            print("\n".join(lines), flush=True)
    return obj


def _run(what: str, cmd: list, verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{res.stdout}\n{res.stderr}")


def _compile_extension(verbose: bool) -> str:
    import sysconfig

    import torch
    from torch.utils import cpp_extension
    obj = os.path.join(OBJ_DIR, os.path.splitext(EXT_SOURCE)[0] + ".o")
    rocm_include = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(hipcc()))), "include")
    includes = [f"-I{d}" for d in [*cpp_extension.include_paths(), sysconfig.get_paths()["include"], rocm_include]]
    _run(f"g++ on {EXT_SOURCE}",
         ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *includes,
          "-c", os.path.join(CSRC, EXT_SOURCE), "-o", obj], verbose)
    return obj


def _link_extension(obj: str, verbose: bool) -> None:
    from torch.utils import cpp_extension
    _run("link of the torch extension",
         ["g++", "-shared", "-fPIC", obj, "-o", EXT_PATH, f"-L{HERE}", "-l:" + LIB_NAME, "-Wl,-rpath,$ORIGIN",
          *[f"-L{d}" for d in cpp_extension.library_paths()], "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip"], verbose)


def build(verbose: bool = True) -> str:
    os.makedirs(OBJ_DIR, exist_ok=True)
    with ThreadPoolExecutor(max_workers=7) as pool:
        ext = pool.submit(_compile_extension, verbose)
        objs = list(pool.map(lambda s: _compile(s, verbose), SOURCES))
        ext_obj = ext.result()
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", LIB_PATH]
    _run("link", cmd, verbose)
    _link_extension(ext_obj, verbose)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose="-q" not in sys.argv))
