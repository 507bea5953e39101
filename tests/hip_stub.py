"""Runs a piece of test code on the library's host side without a GPU: a child
Python process loads tests/cpp/hip_host_stub.cpp (a HIP runtime on the host, whose
kernels do nothing) ahead of libljhip.so, so that sizes, routes, allocations and
captured graphs can be looked at, and allocations refused.

The code sees `ljamd`, `L` (ljamd._lib), `C` (ctypes), `np`, `stub` (the stub's
functions) and `kernels()`: the (name, grid) of the kernels launched or captured
since the last call."""
import os
import subprocess
import sys

TESTS = os.path.dirname(os.path.abspath(__file__))
PYTHON = os.path.join(os.path.dirname(TESTS), "lennard-jones-cuda_amd", "python")

PRELUDE = """
import ctypes as C, sys
import numpy as np
stub = C.CDLL({so!r}, mode=C.RTLD_GLOBAL)
sys.path.insert(0, {python!r})
import ljamd
from ljamd import _lib as L
stub.stub_refuse_above.argtypes = [C.c_size_t]
stub.stub_fail_in.argtypes = [C.c_long, C.c_int]
stub.stub_launch_name.argtypes = stub.stub_launch_grid.argtypes = [C.c_long]
stub.stub_launch_name.restype = C.c_char_p
stub.stub_launch_grid.restype = C.c_uint
stub.stub_live_bytes.restype = C.c_size_t
for f in ("mallocs", "refused", "instantiated", "graphs", "events", "live", "num_launches"):
    getattr(stub, "stub_" + f).restype = C.c_long

def kernels():
    out = [(stub.stub_launch_name(k).decode(), stub.stub_launch_grid(k))
           for k in range(stub.stub_num_launches())]
    stub.stub_clear_launches()
    return out

assert L.lib().lj_device_count() == 1  # the stub's device
"""


def build(tmp):
    so = os.path.join(str(tmp), "hip_host_stub.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", os.path.join(TESTS, "cpp", "hip_host_stub.cpp"), "-o", so],
                   check=True)
    return so


def run(so, code, env=None):
    """Runs `code`; its failed assertions fail the caller's test."""
    r = subprocess.run([sys.executable, "-c", PRELUDE.format(so=so, python=PYTHON) + code],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300,
                       env={**os.environ, **(env or {})})
    assert r.returncode == 0, r.stdout
    return r.stdout
