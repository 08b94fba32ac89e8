"""The library's host side without a GPU: a program run in a process of its own
in which tests/cpp/host_hip.cpp stands in for the HIP runtime (memory is host
memory, kernels do nothing, launches are logged and take the time a test gives
them)."""
import os
import subprocess
import sys
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes, sys
sys.path.insert(0, %r)
H = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)  # before the library: its HIP calls bind to these
H.host_hip_used.restype = ctypes.c_size_t
H.host_hip_limit.argtypes = [ctypes.c_size_t]
H.host_hip_cost.argtypes = [ctypes.c_char_p, ctypes.c_uint, ctypes.c_uint, ctypes.c_double]
H.host_hip_launches.restype = H.host_hip_copies.restype = ctypes.c_char_p
import numpy as np
import asl_amd
from asl_amd import _lib


def launches(part="k_step"):
    # (grid, block) of the launches of kernels with `part` in their name since the last call
    out = [l.rsplit(" ", 2) for l in H.host_hip_launches().decode().splitlines()]
    H.host_hip_forget()
    return [(int(g), int(b)) for n, g, b in out if part in n]


DIRECT, TILE, RUN = b"6k_stepI", b"11k_step_tileI", b"10k_step_runI"


def cost(kernel, ms, block=0, below=0):
    # time of a launch per workgroup: of that size, in launches of fewer than `below` workgroups
    H.host_hip_cost(kernel, block, below, ms)


def copies():
    # (to, from, bytes) of the copies since the last call: d device, p pinned, h other host memory
    out = [l.split() for l in H.host_hip_copies().decode().splitlines()]
    H.host_hip_forget()
    return [(t, f, int(n)) for t, f, n in out]


def cavity(size, q=19, **k):
    L = asl_amd.Lattice(size, q, nu=0.05, **k)
    L.init_equilibrium()
    if not k.get("periodic"):
        for b in (L.add_slice_bc(_lib.BC_NOSLIP, 63),):
            L.execute_bc(b)
    return L
"""


_built = []  # the directory that holds the stand-in, built once a process


def run(program, timeout=300):
    """Runs the program (Python source) over the stand-in; returns what it printed."""
    if not _built:
        _built.append(tempfile.TemporaryDirectory())
        subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o",
                        os.path.join(_built[0].name, "libhosthip.so"),
                        os.path.join(ROOT, "tests", "cpp", "host_hip.cpp")], check=True)
    d = _built[0].name
    r = subprocess.run([sys.executable, "-c", PRELUDE % (ROOT, os.path.join(d, "libhosthip.so")) + program],
                       capture_output=True, text=True, timeout=timeout, cwd=d)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
