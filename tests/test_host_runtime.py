"""The library's host code over a HIP runtime without a GPU (host_hip.cpp): what it waits for and
what memory it gives back.  Kernels do nothing there, so no values are looked at; every check runs
in a process of its own."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "host_hip.cpp")

HEAD = """
import ctypes, sys
import numpy as np
H = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
H.host_hip_limit.argtypes = [ctypes.c_size_t]
H.host_hip_live.restype = ctypes.c_size_t
sys.path.insert(0, sys.argv[2])
from gnu_femlisp_amd import flgpu as F
from gnu_femlisp_amd import iteration as it
from gnu_femlisp_amd import lattice as lat
from gnu_femlisp_amd import matlisp as ml
L = F.lib()
MB = 1 << 20
"""


@pytest.fixture(scope="module")
def host_hip(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host_hip") / "host_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I/opt/rocm/include", SRC,
                    "-o", so], check=True)
    return so


def run(host_hip, body, *args):
    r = subprocess.run([sys.executable, "-c", HEAD + body, host_hip, ROOT, *map(str, args)],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


@pytest.mark.parametrize("dim,order,smoother", [(1, 1, "Jacobi"), (2, 1, "Jacobi"), (2, 1, "SOR"),
                                                (2, 2, "GeometricSSC"), (3, 1, "SOR"),
                                                (3, 2, "GeometricSSC"), (3, 2, "GeometricPSC")])
def test_captured_cycles_are_dropped_after_a_wait(host_hip, dim, order, smoother):
    """flgpu_mg_apply returns before its cycle has run: a reassembly, a change of a level's
    storage and the end of the hierarchy drop the captured cycle only once the stream is idle"""
    run(host_hip, """
dim, order, sm = int(sys.argv[3]), int(sys.argv[4]), sys.argv[5]
cs = it.GeometricCS(getattr(it, sm)(0.5), 1, 1, 0)
Hy = it.Hierarchy.lattice(cs, dim, order, 1, 3)
n = Hy.top_matrix().nrows
x, b, r = (ml.GpuVector(n) for _ in range(3))
kap = ml.GpuVector(4 ** dim)
def gone(): return H.host_hip_graphs_destroyed()
for k in range(2):  # the first may free forms of the levels, which waits by itself
    Hy.apply(x, b, r)
    g = gone()
    ml.check(L.flgpu_mg_reassemble(Hy.h, kap.h, 4))
    assert gone() == g + 1
    assert H.host_hip_destroyed_in_flight() == 0, "reassembly"
g = gone()
Hy.apply(x, b, r)
Hy.level_matrix(1).storage(0)
Hy.apply(x, b, r)
Hy.apply(x, b, r)
del Hy
assert gone() > g
assert H.host_hip_destroyed_in_flight() == 0
""", dim, order, smoother)
