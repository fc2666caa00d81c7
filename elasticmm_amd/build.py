"""In-tree build of libemm_kv.so with hipcc for gfx950, and of the native host side of the
appends (_emm_frontend, an extension module of the Python and the torch it is built with).

The shared object is written next to this file so that it travels with the
source tree; nothing is installed and no JIT cache is used.
"""
from __future__ import annotations

import importlib.util
import os
import shutil
import subprocess
import sysconfig

_PKG = os.path.dirname(os.path.abspath(__file__))
_ROOT = os.path.dirname(_PKG)
_SRC = os.path.join(_PKG, "csrc", "emm_kv.hip")
_INC = os.path.join(_ROOT, "include")
_OUT = os.path.join(_PKG, "libemm_kv.so")
_SRC_FRONTEND = os.path.join(_PKG, "csrc", "emm_frontend.cpp")
_OUT_FRONTEND = os.path.join(_PKG, "_emm_frontend" + sysconfig.get_config_var("EXT_SUFFIX"))
_OUT_HOOKS = os.path.join(_PKG, "libemm_kv_hooks.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    # bit-exact arithmetic: no fused multiply-add / fused multiply-convert (the fp8 rule is
    # "round the fp32 product, then round to 16 bits", two roundings)
    "-ffp-contract=off",
    # keep the compiler from forming packed-fp32 ops out of float code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # the leading scalar kernel arguments arrive in scalar registers when a wave starts (the
    # kernels order their parameters by first use for this): one memory round trip less per wave
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
]


def library_path() -> str:
    return _OUT


def hooks_library_path() -> str:
    return _OUT_HOOKS


def frontend_path() -> str:
    return _OUT_FRONTEND


def build_frontend(verbose: bool = False) -> str:
    """Compile csrc/emm_frontend.cpp -> _emm_frontend.<python tag>.so against the installed torch (always recompiles)."""
    import torch

    root = os.path.dirname(torch.__file__)
    inc, lib = os.path.join(root, "include"), os.path.join(root, "lib")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    cmd = [shutil.which("g++") or "c++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-I{_INC}",
           f"-I{sysconfig.get_paths()['include']}", f"-isystem{inc}", f"-isystem{os.path.join(inc, 'torch', 'csrc', 'api', 'include')}",
           f"-isystem{os.path.join(rocm, 'include')}", "-o", _OUT_FRONTEND, _SRC_FRONTEND, f"-L{lib}", f"-Wl,-rpath,{lib}",
           "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu", "-ltorch_python"]
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed ({proc.returncode}):\n{proc.stdout}")
    if verbose and proc.stdout:
        print(proc.stdout)
    return _OUT_FRONTEND


def build_library(verbose: bool = False, hooks: bool = False) -> str:
    """Compile csrc/emm_kv.hip (which includes the csrc/*.inc kernel files) -> libemm_kv.so (always recompiles). ``hooks=True`` builds
    libemm_kv_hooks.so instead: the same source with -DEMM_BENCH_HOOKS, which adds the launch-variant
    switch, the memory-system probes and the quotient sweep that bench.py and the GPU tests use
    (csrc/emm_kv_hooks.h, csrc/emm_kv_hooks.inc). The product library never contains them; with it the native host
    side of the appends (``build_frontend``) is built where torch is installed."""
    if not hooks and importlib.util.find_spec("torch") is not None:
        build_frontend(verbose)
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    out = _OUT_HOOKS if hooks else _OUT
    extra = ["-DEMM_BENCH_HOOKS", f"-I{os.path.join(_PKG, 'csrc')}"] if hooks else []
    cmd = [hipcc, *HIPCC_FLAGS, *extra, f"-I{_INC}", "-o", out, _SRC]
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed ({proc.returncode}):\n{proc.stdout}")
    if verbose and proc.stdout:
        print(proc.stdout)
    return out


if __name__ == "__main__":
    print(build_library(verbose=True))
    print(build_library(verbose=True, hooks=True))
