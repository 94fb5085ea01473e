"""Run a piece of Python against libnekcem_hip.so on the stand-in runtime of
fake_hip.cpp, in a child interpreter (no GPU, no torch)."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

PRELUDE = """
import ctypes as C, sys
import numpy as np
fake = C.CDLL({lib!r}, mode=C.RTLD_GLOBAL)
fake.fake_log.restype = C.c_char_p
fake.fake_used.restype = C.c_size_t
fake.fake_set_capacity.argtypes = [C.c_int, C.c_size_t]
fake.fake_fail_launch.argtypes = [C.c_long]
def log():
    out = fake.fake_log().decode().splitlines()
    fake.fake_clear_log()
    return out
def launches(part=""):
    return [l for l in log() if l.startswith("launch") and part in l]
sys.path.insert(0, {root!r})
from nekcem_amd import _lib
from nekcem_amd.maxwell import BatchSolver, MaxwellSolver
from nekcem_amd.mesh import BoxMesh
def dev_array(n):
    p = C.c_void_p()
    assert fake.hipMalloc(C.byref(p), C.c_size_t(8 * n)) == 0
    return C.cast(p, C.POINTER(C.c_double))
"""

needs_gxx = pytest.mark.skipif(
    shutil.which("g++") is None or not os.path.exists(os.path.join(ROCM, "include", "hip", "hip_runtime_api.h")),
    reason="needs g++ and the HIP headers")


@pytest.fixture(scope="session")
def fake_hip(tmp_path_factory):
    """run(code): the code's assertions hold in a child on the stand-in runtime."""
    lib = str(tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROCM, "include"), "-o", lib,
                    os.path.join(HERE, "fake_hip.cpp")], check=True)

    def run(code):
        r = subprocess.run([sys.executable, "-c", PRELUDE.format(lib=lib, root=ROOT) + code], capture_output=True,
                           text=True, timeout=300)
        assert r.returncode == 0, (r.stdout + r.stderr)[-4000:]
        return r.stdout

    return run
