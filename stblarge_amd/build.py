"""Builds libstbl_amd.so in-tree with hipcc for gfx950, and _bind.so, the torch-facing call path of
stblarge_amd.ops, with g++ (no JIT cache: the .so files travel with the tree).

Run: python -m stblarge_amd.build   (or __graft_entry__.build()).
"""

import os
import shutil
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


def rocm_home():
    """The ROCm tree that HIPCC (a path or a bare name) belongs to."""
    exe = shutil.which(HIPCC)
    homes = [os.environ.get("ROCM_PATH"), exe and os.path.dirname(os.path.dirname(os.path.realpath(exe))), "/opt/rocm"]
    return next((h for h in homes if h and os.path.isdir(os.path.join(h, "include", "hip"))), "/opt/rocm")


def bind_command(out):
    """The g++ command for csrc/bind.cpp, against the torch and Python that run this. The HIP headers that
    torch's stream header includes ask the host compiler for their platform."""
    import sysconfig

    import torch

    from . import _lib

    t = os.path.dirname(torch.__file__)
    abi = int(torch._C._GLIBCXX_USE_CXX11_ABI)
    return ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Wno-missing-field-initializers",
            f"-D_GLIBCXX_USE_CXX11_ABI={abi}", "-DUSE_ROCM=1", "-D__HIP_PLATFORM_AMD__=1",
            f'-DSTBL_BUILT_FOR="{_lib.host_version()}"', "-isystem", os.path.join(t, "include"), "-isystem",
            sysconfig.get_paths()["include"], "-isystem", os.path.join(rocm_home(), "include"),
            os.path.join(CSRC, "bind.cpp"), "-L" + os.path.join(t, "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu",
            "-ltorch_python", "-o", out]


def build_bind(verbose=False):
    """Compile the binding. The library works without it, so a failure (no g++, no torch headers) is only
    reported, and an older binding, which may not fit the library, is removed."""
    tmp = BIND + ".tmp"
    try:
        cmd = bind_command(tmp)
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.run(cmd, check=True)
        os.replace(tmp, BIND)
    except (ImportError, OSError, subprocess.CalledProcessError) as e:
        if os.path.exists(BIND):
            os.remove(BIND)
        print(f"{BIND} was not built ({e}): calls will take the slower Python path", file=sys.stderr)


def build(verbose=False):
    """Compile every HIP source into one shared library, and beside it the binding. Always recompiles."""
    tmp = LIB + ".tmp"
    cmd = [HIPCC, *FLAGS, "-I", CSRC, "-I", os.path.join(os.path.dirname(HERE), "include"), *sources(), "-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    with subprocess.Popen(cmd) as job:  # leaving waits for it
        build_bind(verbose)
    if job.returncode:
        raise subprocess.CalledProcessError(job.returncode, cmd)
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    build(verbose="-v" in sys.argv)
    print("built", LIB)
