"""Runs a test body in a process of its own whose HIP runtime is fake_hip.cpp."""
import os
import subprocess
import sys
import textwrap

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))

PRELUDE = """
import ctypes, sys, threading, time
import numpy as np
sys.path.insert(0, {root!r})
fake = ctypes.CDLL({lib!r}, mode=ctypes.RTLD_GLOBAL)  # before the library: its calls end here
fake.fake_device_limit.argtypes = [ctypes.c_size_t]
fake.fake_device_used.restype = ctypes.c_size_t
from emptyroom_amd import api, synth
f = synth.small_framework(7, n_atoms=40, cell=(10.0, 11.0, 12.0, 85.0, 95.0, 100.0))
a = f.particles()
ARGS = (a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2)
"""


def build(folder) -> str:
    lib = os.path.join(str(folder), "libfake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-o", lib, os.path.join(HERE, "fake_hip.cpp")],
                   check=True)
    return lib


def run(lib: str, body: str, timeout: float = 60.0) -> str:
    code = PRELUDE.format(root=ROOT, lib=lib) + textwrap.dedent(body)
    p = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True,
                       timeout=timeout, env=dict(os.environ, OMP_NUM_THREADS="1",
                                                 OPENBLAS_NUM_THREADS="1"))
    assert p.returncode == 0, p.stdout[-2000:] + p.stderr[-4000:]
    return p.stdout
