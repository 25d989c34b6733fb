import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU and the built HIP library")


def has_gpu():
    try:
        import torch
        return torch.cuda.is_available()
    except Exception:
        return False


@pytest.fixture(scope="session")
def gpu():
    if not has_gpu():
        pytest.skip("no GPU")
    import torch
    return torch.device("cuda:0")


@pytest.fixture(scope="session")
def gemm_plan(tmp_path_factory):
    """(kernel, chained, steps of a group) of a GEMM call, from the rules the library is built with."""
    import ctypes
    import subprocess

    lib = str(tmp_path_factory.mktemp("plan") / "gemm_plan.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "stblarge_amd", "csrc"),
                    os.path.join(ROOT, "tests", "gemm_plan_check.cpp"), "-o", lib], check=True)
    fn = ctypes.CDLL(lib).gemm_plan_of
    kernels = ("split", "waves22", "waves24", "one32", "one64", "tile64", "tile128")

    def plan(fmt, m, n, k, aligned=True):
        out = (ctypes.c_int * 3)()
        fn(fmt, m, n, k, int(aligned), out)
        return kernels[out[0]], bool(out[1]), out[2]
    return plan
