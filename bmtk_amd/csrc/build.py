"""Compile the HIP sources into ``bmtk_amd/libbmtk_amd.so`` for gfx950.

Run as ``python -m bmtk_amd.csrc.build``.  hipcc cross-compiles without a GPU.
Flags that matter for results:
  -ffp-contract=off      no fused multiply-add, so the fp32 update rounds like a
                         scalar evaluation of the same expressions;
  -munsafe-fp-atomics    fp32 atomicAdd becomes the hardware global atomic
                         instead of a compare-and-swap loop (device memory only);
  -packed-fp32-ops off   no packed fp32 instructions are generated.
"""
import os
import subprocess
import sys
import sysconfig
import warnings

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.dirname(HERE)
LIB = os.path.join(PKG, "libbmtk_amd.so")
PTR = os.path.join(PKG, "_ptr" + sysconfig.get_config_var("EXT_SUFFIX"))   # (names the Python it is for)
SOURCES = ["kernels.hip", "propagate_pull.hip", "simulate.hip", "simulate_fused.hip", "resident.hip", "resident_solo.hip", "resident_windows.hip", "resident_batch.hip", "backward.hip", "poisson.hip", "microbench.hip"]
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off",
         "-munsafe-fp-atomics", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-Wall", "-Wno-unused-function"]


def build(verbose=False, extra=()):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    cmd = [hipcc] + FLAGS + list(extra) + ["-o", LIB] + [os.path.join(HERE, s) for s in SOURCES]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in res.stdout.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError("hipcc failed:\n" + out)
    if verbose and out.strip():
        print(out)
    build_ptr(verbose)
    return LIB


def build_ptr(verbose=False):
    """The pointer checks of ``ops._p`` as a Python module (host code).  The package does the same in Python without it: what
    keeps it from being compiled (no C++ compiler, no headers) is a warning, and an older one is taken away."""
    import torch
    from torch.utils import cpp_extension
    lib_dir = os.path.join(os.path.dirname(torch.__file__), "lib")
    cmd = ([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-w",
            "-D_GLIBCXX_USE_CXX11_ABI={}".format(int(torch._C._GLIBCXX_USE_CXX11_ABI)), '-DBMTK_AMD_TORCH="{}"'.format(torch.__version__)]
           + ["-I" + d for d in cpp_extension.include_paths() + [sysconfig.get_paths()["include"]]]
           + ["-o", PTR, os.path.join(HERE, "ptr.cpp"), "-L" + lib_dir, "-ltorch_python", "-ltorch_cpu", "-lc10"])
    if verbose:
        print(" ".join(cmd), flush=True)
    try:
        res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        failed = res.stdout if res.returncode != 0 else None
    except OSError as exc:
        failed = str(exc)
    if failed is not None:
        if os.path.exists(PTR):
            os.remove(PTR)
        warnings.warn("ptr.cpp was not compiled, its checks are made in Python:\n" + failed)
        return None
    return PTR


if __name__ == "__main__":
    print(build(verbose=True, extra=sys.argv[1:]))
