"""Runs a piece of Python with the engine's host code on host memory
(host_runtime.cpp), in a process of its own, without a GPU."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

HEAD = """
import ctypes, sys
sys.path.insert(0, %r)
rt = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)
rt.rt_fail_above.argtypes = rt.rt_alloc_us.argtypes = [ctypes.c_size_t]
rt.rt_live_bytes.restype = rt.rt_live.restype = ctypes.c_size_t
rt.rt_lds.restype = ctypes.c_size_t
rt.rt_stored.restype = ctypes.c_longlong
rt.rt_cost.argtypes = [ctypes.c_char_p, ctypes.c_double, ctypes.c_double,
                       ctypes.c_int]
import numpy as np
import mpci
from mpci import synth

def system(s, gauge="v"):
    E, D = synth.system_arrays(s, seed=3)
    return mpci.System(E, D, gauge=gauge)

def launches(name):
    return rt.rt_launched(name.encode())

def attempts():
    a = (ctypes.c_int * 4096)()
    return list(a[:rt.rt_attempts(a, 4096)])
"""


@pytest.fixture(scope="session")
def host_runtime(tmp_path_factory):
    """Runs code; np, mpci, synth, rt, system, launches, attempts are there."""
    if not os.path.isdir(os.path.join(ROCM, "include", "hip")):
        pytest.skip("no HIP headers")
    if not shutil.which("g++"):
        pytest.skip("no g++")
    so = str(tmp_path_factory.mktemp("rt") / "host_runtime.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-w",
                    "-D__HIP_PLATFORM_AMD__", "-I" + ROCM + "/include",
                    os.path.join(HERE, "host_runtime.cpp"), "-o", so,
                    "-pthread"], check=True, timeout=300)
    pkg = os.path.join(os.path.dirname(HERE), "mp-citdse_amd")

    def run(code):
        r = subprocess.run([sys.executable, "-c",
                            HEAD % (pkg, so) + textwrap.dedent(code)],
                           capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stderr[-3000:]
        return r.stdout

    return run
