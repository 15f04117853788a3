"""Runs a test body against libsgpp_hip.so on host memory (host_hip.cpp), in a child process."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes, sys
sys.modules["torch"] = None  # (torch would bring its own HIP runtime)
hip = ctypes.CDLL(%r, ctypes.RTLD_GLOBAL)
hip.host_hip_fail_malloc.argtypes = [ctypes.c_long, ctypes.c_int]
hip.host_hip_allocated.restype = ctypes.c_size_t
hip.host_hip_launches.restype = ctypes.c_size_t
hip.host_hip_launches.argtypes = [ctypes.c_char_p, ctypes.c_size_t]
sys.path[:0] = [%r, %r]
import numpy as np
from sgpp_amd import capi, workloads

def launches():
    "the kernels launched since the last call: (mangled name, grid x, grid y, threads)"
    buf = ctypes.create_string_buffer(hip.host_hip_launches(None, 0))
    hip.host_hip_launches(buf, len(buf))
    hip.host_hip_clear()
    lines = [line.split() for line in buf.value.decode().splitlines()]
    return [(n, int(x), int(y), int(t)) for n, x, y, t in lines]
"""


@pytest.fixture(scope="session")
def on_host(tmp_path_factory):
    """on_host(body): body's output, run with `hip`, `capi` and `launches` at hand"""
    out = str(tmp_path_factory.mktemp("host_hip") / "host_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I" + os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"),
                    os.path.join(HERE, "host_hip.cpp"), "-o", out], check=True)

    def run(body):
        r = subprocess.run([sys.executable, "-c", PRELUDE % (out, ROOT, HERE) + textwrap.dedent(body)],
                           capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, (r.returncode, r.stdout[-2000:], r.stderr[-4000:])
        return r.stdout
    return run
