"""Runs a piece of Python in a process whose HIP runtime is recording_hip.cpp: the built library's host code
plans, allocates and launches as on the device, and the launches are read back as text."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes, re, sys
import numpy as np
rec = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
rec.rec_launches.restype = ctypes.c_char_p
rec.rec_pinned_most.restype = ctypes.c_size_t
rec.rec_pinned_flags.restype = ctypes.c_uint
rec.rec_fail_pinned_from.argtypes = [ctypes.c_size_t]
import rbergomi_amd as rb

def launches(kernel=""):
    '''(name, fields) of the launches since the last call, of kernels whose name has `kernel`'''
    out = []
    for line in rec.rec_launches().decode().splitlines():
        w = line.split()
        if kernel not in w[0]:
            continue
        f = dict(grid=int(w[2]), grid_y=int(w[3]))
        f.update((w[i], int(w[i + 1])) for i in range(4, len(w), 2))
        out.append((w[0], f))
    rec.rec_clear()
    return out
"""


def build(folder):
    hipcc = next((c for c in ("/opt/rocm/bin/hipcc", shutil.which("hipcc")) if c and os.path.exists(c)), None)
    if hipcc is None:
        pytest.skip("hipcc not available")
    lib = str(folder / "librecording_hip.so")
    r = subprocess.run([hipcc, "-O1", "-std=c++17", "-fPIC", "-shared", "-x", "hip", "--cuda-host-only",
                        "-I" + os.path.join(ROOT, "rbergomi_amd", "csrc"), os.path.join(HERE, "recording_hip.cpp"), "-o", lib],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-3000:]
    return lib


def run(lib, code, env=None):
    r = subprocess.run([sys.executable, "-c", PRELUDE + code, lib], capture_output=True, text=True, timeout=600, cwd=ROOT,
                       env=dict(os.environ, **(env or {})))
    assert r.returncode == 0, (r.stdout + r.stderr)[-3000:]
    return r.stdout
