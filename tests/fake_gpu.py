"""Runs a program against libwtc.so with fake_hip.c in the place of the HIP
runtime, in a process of its own, to see what the host code allocates, copies
and launches without a GPU."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "wedge-parallel-triangle-counting_amd")

_PRELUDE = """
import ctypes as C, sys
import numpy as np
fake = C.CDLL({so!r}, mode=C.RTLD_GLOBAL)
fake.fake_launch.restype = C.c_char_p
fake.fake_allocs.restype = fake.fake_copies.restype = C.c_uint64
sys.path.insert(0, {pkg!r})
import wtc
assert wtc.device_count() == 1


def launches(f):
    "Names of the kernels that f() launches, without their arguments."
    fake.fake_reset()
    f()
    return [fake.fake_launch(i).decode() for i in range(fake.fake_launches())]


def ran(names, kernel):
    return any(f"{{len(kernel)}}{{kernel}}" in x for x in names)
"""


def run(tmp_path, program, env=None):
    """Runs the program (source text) after the prelude above; fails with its
    output where it fails."""
    if shutil.which("gcc") is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime_api.h"):
        pytest.skip("needs gcc and the HIP headers")
    so = os.path.join(str(tmp_path), "libfakehip.so")
    subprocess.run(["gcc", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-shared", "-fPIC", "-o", so,
                    os.path.join(HERE, "fake_hip.c")], check=True, timeout=120)
    r = subprocess.run([sys.executable, "-c", _PRELUDE.format(so=so, pkg=PKG) + program], capture_output=True, text=True,
                       timeout=300, env=dict(os.environ, **(env or {})))
    assert r.returncode == 0, f"exit {r.returncode}\n{r.stdout}\n{r.stderr}"
    return r.stdout
