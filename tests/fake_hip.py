"""Runs a piece of Python against the built library on a HIP runtime without a
device (host/fake_hip.cpp), in a process of its own that never imports torch:
`lib` is the library, `fake` the runtime, `h` a handle."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(os.path.dirname(HERE), "gempy_amd", "libgkhip.so")

_HEAD = """
import ctypes as C, sys
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
fake.fake_name.restype = fake.fake_log.restype = C.c_char_p
lib = C.CDLL(sys.argv[2])
lib.gk_last_error.restype = C.c_char_p
h = C.c_void_p()
assert lib.gk_create(0, C.byref(h)) == 0
def i64(*v): return (C.c_int64 * len(v))(*v)
def f64(*v): return (C.c_double * len(v))(*v)
def device(n):
    p = C.c_void_p()
    assert fake.hipMalloc(C.byref(p), C.c_size_t(n)) == 0
    return p
def launched(): return [fake.fake_name(i).decode() for i in range(fake.fake_launches())]
"""


def build(directory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    so = os.path.join(str(directory), "libfakehip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-o", so, os.path.join(HERE, "host", "fake_hip.cpp")], check=True)
    return so


def run(so, body):
    r = subprocess.run([sys.executable, "-c", _HEAD + body, so, LIB], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
