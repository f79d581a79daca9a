"""Builds librwkv6_amd.so (all HIP sources in csrc/) for gfx950 with hipcc.

and _native.so (csrc/autograd.cpp, the autograd functions over its C ABI) with the host compiler
against the installed torch.

Usage: python rwkv-megatron_amd/build.py   (also called by __graft_entry__.build()).
Both land next to this file so they travel with the source tree.
"""
import glob
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "librwkv6_amd.so")
NATIVE = os.path.join(HERE, "_native.so")
ARCH = os.environ.get("RWKV6_OFFLOAD_ARCH", "gfx950")

# Packed-FP32 instructions are disabled for all device code; hipcc's host pass
# warns that it does not know the feature, which is harmless.
FLAGS = [
    "-O3", "-std=c++17", "-fPIC", "-shared", f"--offload-arch={ARCH}",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-command-line-argument",
]


def sources():
    return sorted(glob.glob(os.path.join(HERE, "csrc", "*.hip")))


def build(verbose: bool = False) -> str:
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    tmp = LIB + ".tmp"
    cmd = [hipcc, *FLAGS, *sources(), "-o", tmp]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError("hipcc failed building librwkv6_amd.so")
    if verbose:
        msgs = [l for l in (res.stdout + res.stderr).splitlines() if "packed-fp32-ops" not in l]
        if msgs:
            print("\n".join(msgs))
    os.replace(tmp, LIB)
    return LIB


def build_native() -> str:
    """The torch extension; needs the HIP library (build()) to link against."""
    import torch
    from torch.utils import cpp_extension

    torch_lib = cpp_extension.library_paths()[0]
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    tmp = NATIVE + ".tmp"
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_EXTENSION_NAME=_native",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *(f"-isystem{p}" for p in cpp_extension.include_paths()),
           "-isystem" + sysconfig.get_paths()["include"], f"-isystem{rocm}/include",
           os.path.join(HERE, "csrc", "autograd.cpp"), "-o", tmp,
           f"-L{HERE}", "-l:librwkv6_amd.so", "-Wl,-rpath,$ORIGIN",
           f"-L{torch_lib}", "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError("the host compiler failed building _native.so")
    os.replace(tmp, NATIVE)
    return NATIVE


if __name__ == "__main__":
    print(build(verbose=True))
    print(build_native())
