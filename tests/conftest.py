import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP kernels)")


def gpu_available():
    try:
        import torch

        return torch.cuda.is_available()
    except Exception:
        return False


@pytest.fixture(scope="session")
def golden_dir():
    return os.path.join(ROOT, "tests", "golden")


@pytest.fixture(scope="session")
def lanes_lib(tmp_path_factory):
    """The device headers on emulated lanes (tests/host), built with the host compiler."""
    import ctypes
    import shutil
    import subprocess

    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    so = str(tmp_path_factory.mktemp("lanes") / "lanes.so")
    host = os.path.join(ROOT, "tests", "host")
    subprocess.run([gxx, "-O2", "-march=native", "-ffp-contract=off", "-std=c++17", "-w", "-shared", "-fPIC",
                    "-I", os.path.join(host, "lanes"), "-I", os.path.join(ROOT, "qex_amd", "csrc"),
                    os.path.join(host, "lanes_harness.cpp"), "-o", so],
                   check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    return ctypes.CDLL(so)
