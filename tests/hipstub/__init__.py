"""Runs a piece of Python in a process of its own whose HIP runtime is hip_stub.cpp."""

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))

HEAD = """
import ctypes as C, sys
import numpy as np
sys.path[:0] = [{root!r}, {root!r} + "/tests"]
stub = C.CDLL({lib!r}, mode=C.RTLD_GLOBAL)
for f in ("stub_mallocs", "stub_events", "stub_news", "stub_launches"):
    getattr(stub, f).restype = C.c_long
stub.stub_launch.restype = C.c_char_p
stub.stub_launch.argtypes = stub.stub_malloc_ok.argtypes = stub.stub_new_fail.argtypes = [C.c_long]
from olam_amd import abi, cases, mesh as M
from olam_amd.gpu import Context, OlamGpuError, lib

def launches(since=0):
    return [stub.stub_launch(i).decode() for i in range(since, stub.stub_launches())]

def fails(f, *a, **k):
    try:
        f(*a, **k)
    except OlamGpuError as e:
        return str(e)
    return None
"""


def build(out):
    lib = os.path.join(str(out), "hip_stub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", lib, os.path.join(HERE, "hip_stub.cpp")],
                   check=True)
    return lib


def run(lib, body, timeout=300):
    """The process's output; asserts that it ended with status 0."""
    p = subprocess.run([sys.executable, "-c", HEAD.format(root=ROOT, lib=lib) + body], capture_output=True, text=True,
                       timeout=timeout)
    assert p.returncode == 0, f"status {p.returncode}\n{p.stdout[-2000:]}\n{p.stderr[-4000:]}"
    return p.stdout
