"""The library's host code on a HIP runtime without a GPU (hip_stub.cpp): a
script runs in a process of its own, in which the library's HIP calls bind to
the stand-in, and returns what it leaves in `result`."""
import json
import os
import subprocess
import sys
import textwrap

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
PKG = os.path.join(ROOT, "j-pet-mlem-old_amd")

_PREAMBLE = """
import ctypes, json, sys
import numpy as np
stub = ctypes.CDLL({stub!r}, mode=ctypes.RTLD_GLOBAL)
stub.stub_fail_in.argtypes = [ctypes.c_long]
stub.stub_allocations.restype = stub.stub_live.restype = ctypes.c_long
stub.stub_launches.argtypes = [ctypes.c_char_p, ctypes.c_int,
                               ctypes.c_ulonglong]
stub.stub_launches.restype = ctypes.c_long
stub.stub_work_items.argtypes = [ctypes.c_char_p]
stub.stub_work_items.restype = ctypes.c_ulonglong
stub.stub_effect.argtypes = [ctypes.c_char_p, ctypes.c_int, ctypes.c_char_p,
                             ctypes.c_size_t]
sys.path.insert(0, {package!r})
import pystrip
result = None
"""


def compiler():
    return ["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__",
            "-I/opt/rocm/include", "-I" + os.path.join(PKG, "csrc"),
            "-I" + os.path.join(ROOT, "include")]


def build(directory) -> str:
    """Compiles the stand-in runtime; returns its path."""
    out = os.path.join(str(directory), "hip_stub.so")
    subprocess.run(compiler() + ["-shared", "-fPIC",
                                 os.path.join(HERE, "hip_stub.cpp"),
                                 "-o", out],
                   check=True, capture_output=True, text=True)
    return out


def run(directory, script):
    """Runs `script` on the stand-in; returns the value of its `result`."""
    code = _PREAMBLE.format(stub=build(directory), package=PKG) \
        + textwrap.dedent(script) + "\nprint(json.dumps(result))\n"
    p = subprocess.run([sys.executable, "-c", code], capture_output=True,
                       text=True, timeout=120)
    assert p.returncode == 0, p.stdout + p.stderr
    return json.loads(p.stdout.strip().splitlines()[-1])
