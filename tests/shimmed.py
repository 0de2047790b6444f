"""Runs a test's body in a Python process of its own whose liblbm.so calls the
runtime through tests/host/hip_shim.cpp, which fails chosen calls on request."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes, sys
sys.path[:0] = [{root!r} + "/d3q19-single-phase_amd", {root!r} + "/oracle"]
shim = ctypes.CDLL({shim!r}, mode=ctypes.RTLD_GLOBAL)
import numpy as np
import d3q19
from d3q19 import workloads
lib = d3q19.load_library()


def switch(name, value):
    ctypes.c_int.in_dll(shim, name).value = value


def bits(a):
    return np.ascontiguousarray(a).view(np.uint64)


def start(lx, ly, lz, prec="fp64", seed=6):
    ch = d3q19.Channel(lx, ly, lz, prec)
    u = workloads.laminar_parabola_noise(lx, ly, lz, seed=seed)
    ch.set_macros(ux=u[0], uy=u[1], uz=u[2])
    ch.FORCING()
    ch.initpop()
    return ch


"""


def run_shimmed(body, tmp_path, timeout=100):
    """Runs `body` after PRELUDE; it fails by raising."""
    shim = os.path.join(tmp_path, "hip_shim.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", os.path.join(ROOT, "tests", "host", "hip_shim.cpp"), "-o", shim,
                    "-ldl"], check=True, capture_output=True)
    r = subprocess.run([sys.executable, "-c", PRELUDE.format(root=ROOT, shim=str(shim)) + body + "\nprint('body done')\n"],
                       capture_output=True, text=True, timeout=timeout)
    assert r.returncode == 0 and "body done" in r.stdout, r.stdout + r.stderr
