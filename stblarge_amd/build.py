"""Builds libstbl_amd.so in-tree with hipcc for gfx950, and _bind.so, the torch-facing call path of
stblarge_amd.ops, with g++ (no JIT cache: the .so files travel with the tree).

Run: python -m stblarge_amd.build   (or __graft_entry__.build()).
"""

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libstbl_amd.so")
BIND = os.path.join(HERE, "_bind.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SOURCES = ["abi.hip", "quant.hip", "gemv.hip", "moe.hip", "gemm.hip", "expert_cache.hip", "gguf.hip", "calib.hip"]

FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    "-Wall",
    "-Wno-unused-function",
    # Packed fp32 VALU ops are kept out of the generated code (they are not needed here).
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # Products and sums written in the sources may fuse into FMAs (each kernel's exactness argument
    # allows for it), but not the multiply-subtract pairs inside the compiler's own expansions of
    # expf / log1pf: under -ffp-contract=fast the backend fuses the range reduction's x * log2(e) - n
    # into one FMA, which counts the product's rounding error twice (device expf off by up to 43 fp32
    # ulps at |x| ~ 70, 5 ulps within |x| < 10); fast-honor-pragmas leaves them as written.
    "-ffp-contract=fast-honor-pragmas",
]


def sources():
    return [os.path.join(CSRC, s) for s in SOURCES if os.path.exists(os.path.join(CSRC, s))]


def bind_command(out):
    """The g++ command for csrc/bind.cpp, against the torch and Python that run this. The HIP headers that
    torch's stream header includes ask the host compiler for their platform."""
    import sysconfig

    import torch

    from . import _lib

    t = os.path.join(os.path.dirname(torch.__file__))
    rocm = os.path.dirname(os.path.dirname(HIPCC))
    abi = int(torch._C._GLIBCXX_USE_CXX11_ABI)
    return ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Wno-missing-field-initializers", f"-D_GLIBCXX_USE_CXX11_ABI={abi}", "-DUSE_ROCM=1",
            "-D__HIP_PLATFORM_AMD__=1", f'-DSTBL_BUILT_FOR="{_lib.host_version()}"', "-isystem", os.path.join(t, "include"), "-isystem",
            sysconfig.get_paths()["include"], "-isystem", os.path.join(rocm, "include"),
            os.path.join(CSRC, "bind.cpp"), "-o", out, "-L" + os.path.join(t, "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu",
            "-ltorch_python"]


def build(verbose=False):
    """Compile every HIP source into one shared library, and the binding. Always recompiles."""
    lib = [HIPCC, *FLAGS, "-I", CSRC, "-I", os.path.join(os.path.dirname(HERE), "include"), *sources(), "-o", LIB + ".tmp"]
    jobs = []
    for cmd, out in ((lib, LIB), (bind_command(BIND + ".tmp"), BIND)):
        if verbose:
            print(" ".join(cmd), flush=True)
        jobs.append((subprocess.Popen(cmd), cmd, out))
    for job, cmd, out in jobs:
        if job.wait():
            raise subprocess.CalledProcessError(job.returncode, cmd)
        os.replace(out + ".tmp", out)
    return LIB


if __name__ == "__main__":
    build(verbose="-v" in sys.argv)
    print("built", LIB)
