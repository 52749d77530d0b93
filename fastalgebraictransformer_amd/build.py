"""Build libkat.so (the HIP kernels behind the C ABI in include/kat.h).

Compiles every csrc/*.hip file for gfx950 with hipcc, in parallel, into
objects under fastalgebraictransformer_amd/_build/ and links them into
fastalgebraictransformer_amd/libkat.so. The library records no RUNPATH to
ROCm: at load time its libamdhip64.so.7 dependency binds to the HIP runtime
the host process (PyTorch) already loaded, so one runtime serves both.

Beside it, csrc/torch_ops.cpp (host code: the autograd entry points over that
C ABI) becomes the extension module _katops.so, linked to libkat.so in the same
folder.
"""

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import sysconfig

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
INCLUDE = os.path.join(ROOT, "include")
BUILD = os.path.join(PKG, "_build")
LIB = os.path.join(PKG, "libkat.so")
OPS = os.path.join(PKG, "_katops.so")
ARCH = os.environ.get("KAT_OFFLOAD_ARCH", "gfx950")

HIPCC_FLAGS = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    "-I", INCLUDE, "-I", CSRC,
    # packed fp32 VALU ops are kept out of the generated code on purpose
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def hipcc():
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (ROCm is required to build libkat.so)")


def _compile(src, obj):
    cmd = [hipcc(), *HIPCC_FLAGS, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {os.path.basename(src)}:\n{r.stdout}\n{r.stderr}")
    return obj


def _run(cmd, what):
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{r.stdout}\n{r.stderr}")


def _compile_ops(obj):
    """torch_ops.cpp with the host compiler against torch's headers."""
    import torch
    tinc = os.path.join(os.path.dirname(torch.__file__), "include")
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(hipcc())))
    _run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-c",
          os.path.join(CSRC, "torch_ops.cpp"), "-o", obj,
          # what torch's ROCm headers and the HIP headers expect
          "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
          "-I", INCLUDE, "-I", tinc, "-I", os.path.join(tinc, "torch", "csrc", "api", "include"),
          "-I", os.path.join(rocm, "include"), "-I", sysconfig.get_paths()["include"]],
         "compiling torch_ops.cpp")
    return obj


def _link_ops(obj):
    import torch
    tlib = os.path.join(os.path.dirname(torch.__file__), "lib")
    tmp = OPS + ".tmp"
    _run([os.environ.get("CXX", "g++"), "-shared", "-fPIC", obj, "-o", tmp, "-L", tlib, "-ltorch",
          "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip", "-L", PKG, "-l:libkat.so",
          "-Wl,-rpath,$ORIGIN"], "linking _katops.so")
    os.replace(tmp, OPS)


def build(verbose=True, jobs=None):
    os.makedirs(BUILD, exist_ok=True)
    srcs = sorted(f for f in os.listdir(CSRC) if f.endswith(".hip"))
    objs = [os.path.join(BUILD, s[:-4] + ".o") for s in srcs]
    jobs = jobs or min(len(srcs), max(1, (os.cpu_count() or 4)))
    with cf.ThreadPoolExecutor(jobs) as ex:
        futs = [ex.submit(_compile, os.path.join(CSRC, s), o) for s, o in zip(srcs, objs)]
        futs.append(ex.submit(_compile_ops, os.path.join(BUILD, "torch_ops.o")))
        for f in futs:
            f.result()
    tmp = LIB + ".tmp"
    _run([hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs], "link")
    os.replace(tmp, LIB)
    _link_ops(os.path.join(BUILD, "torch_ops.o"))
    if verbose:
        print(f"built {LIB} and {OPS}", file=sys.stderr)
    return LIB


if __name__ == "__main__":
    build()
