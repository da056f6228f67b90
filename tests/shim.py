"""Runs a piece of test code in a process of its own in which tests/hip_shim.cpp
stands between libtbtkx.so and the HIP runtime."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes, sys
sys.path.insert(0, {root!r})
shim = ctypes.CDLL({lib!r}, mode=ctypes.RTLD_GLOBAL)
import numpy as np
from tbtk_amd import engine as X
from tbtk_amd import lattice as L
value = lambda name: ctypes.c_int.in_dll(shim, name)
eng = X.Engine(0)
"""


def run_shimmed(tmp_path, code, timeout=100):
    """Runs `code` (with eng, X, L, np and value(name), an int of the shim)."""
    lib = str(tmp_path / "libhip_shim.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-o", lib,
                    os.path.join(ROOT, "tests", "hip_shim.cpp"), "-ldl"], check=True)
    text = PRELUDE.format(root=ROOT, lib=lib) + code + "\nprint('shimmed ok')\n"
    r = subprocess.run([sys.executable, "-u", "-c", text], capture_output=True, text=True,
                       timeout=timeout)
    assert r.returncode == 0 and r.stdout.endswith("shimmed ok\n"), r.stdout + r.stderr
    return r.stdout
