"""The library's host code over a HIP runtime without a GPU (host_hip.cpp): what it waits for and
what memory it gives back.  Device memory reads as zero there, so no values are looked at; every
check runs in a process of its own."""
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


@pytest.mark.parametrize("kind", ["vector", "matrix", "hierarchy", "other context"])
def test_kept_blocks_are_given_back_to_any_allocation(host_hip, kind):
    """the blocks that a context keeps for its next setup do not make another allocation fail:
    of its own vectors, matrices and hierarchies, or of another context's"""
    run(host_hip, """
kind = sys.argv[3]
ctx = ml.default_context()
other = ml.Context(0)
before = H.host_hip_live()
A = lat.assemble(3, 2, 12, rhs=False)[0]
del A
kept = H.host_hip_live() - before  # the assembly's temporaries
assert kept > 8 * MB, kept
# what the allocation takes by itself, and then with no more memory than that
def get(c):
    if kind == "matrix":
        return lat.assemble(3, 1, 24, rhs=False, ctx=c)[0]
    if kind == "hierarchy":
        return it.Hierarchy.lattice(it.GeometricCS(it.Jacobi(0.5)), 3, 1, 3, 4, ctx=c)
    return ml.GpuVector(4 * kept // 5 // 8, ctx=c)
c = other if kind == "other context" else ctx
H.host_hip_limit(H.host_hip_live() + kept // 2)
try:
    v = get(c)
finally:
    H.host_hip_limit(1 << 60)
assert H.host_hip_live() < before + kept + kept // 2
del v
""", kind)


def test_kept_blocks_end_with_their_context(host_hip):
    """all memory is given back when the objects and their contexts are gone"""
    run(host_hip, """
start = H.host_hip_live()
c = ml.Context(0)
A = lat.assemble(3, 2, 6, ctx=c)
Hy = it.Hierarchy.lattice(it.GeometricCS(it.GeometricSSC(1.0)), 3, 2, 1, 3, ctx=c)
del A, Hy
assert H.host_hip_live() > start
ml.check(L.flgpu_ctx_destroy(c.h))
c.h = None
assert H.host_hip_live() == start
""")


@pytest.mark.parametrize("prec", ["F64", "F32"])
def test_a_hierarchy_keeps_no_larger_block_than_it_needs(host_hip, prec):
    """the memory that a hierarchy holds does not depend on the blocks that its context had kept
    from other work, and a reassembly leaves it as it is"""
    run(host_hip, """
prec = getattr(F, sys.argv[3])
def free_kept():  # an allocation that fails releases every kept block
    H.host_hip_limit(H.host_hip_live())
    try:
        ml.GpuVector(MB)
    except Exception:
        pass
    H.host_hip_limit(1 << 60)
def held(work):
    c = ml.Context(0)
    for n in work:
        del_me = lat.assemble(3, 2, n, rhs=False, prec=prec, ctx=c)[0]
        del del_me
    before = H.host_hip_live()
    Hy = it.Hierarchy.lattice(it.GeometricCS(it.Jacobi(0.5), prec=prec), 3, 1, 4, 2, ctx=c)
    out = []
    for k in range(3):
        free_kept()
        out.append(H.host_hip_live())
        ml.check(L.flgpu_mg_reassemble(Hy.h, None, 0))
    del Hy
    free_kept()
    out = [o - H.host_hip_live() for o in out]
    return out
alone = held([])
assert alone[0] == alone[1] == alone[2], alone
for work in ([3], [2, 3, 4], [3, 5, 6, 3]):
    assert held(work) == alone, (work, held(work), alone)
""", prec)


@pytest.mark.parametrize("cap,kernel", [("CELL", b"k_rap_q1"), ("STENCIL", b"k_rap_q1"),
                                        ("SELL", b"k_rap_entry")])
def test_galerkin_levels_of_a_lattice_take_a_lattice_product(host_hip, cap, kernel):
    """the Galerkin products of a reassembly compute their positions also where the levels'
    storage was capped; the product that searches the rows is for other matrices"""
    run(host_hip, """
cs = it.GeometricCS(it.Jacobi(0.5), transfer="blackbox")
Hy = it.Hierarchy.lattice(cs, 3, 1, 2, 3)
for l in range(3):
    Hy.level_matrix(l).storage(getattr(F, "STORAGE_" + sys.argv[3]))
kap = ml.GpuVector(8 ** 3)
count = lambda k: H.host_hip_launches(k)
a, b = count(sys.argv[4].encode()), count(b"k_rap")
ml.check(L.flgpu_mg_reassemble(Hy.h, kap.h, 8))
assert count(sys.argv[4].encode()) == a + 2
assert count(b"k_rap") == b + 2
del Hy
""", cap, kernel.decode())


@pytest.mark.parametrize("dim,order", [(3, 1), (3, 2), (2, 2)])
def test_a_storage_cap_reaches_the_interpolation(host_hip, dim, order):
    """capped to SELL, an interpolation, its transpose and its copies stream their stored values,
    and a captured cycle that had read the positions instead is dropped"""
    run(host_hip, """
dim, order = int(sys.argv[3]), int(sys.argv[4])
lattice_products = lambda: H.host_hip_launches(b"k_q2_") + H.host_hip_launches(b"k_tp_")
def products(P):
    c, f = ml.GpuVector(P.ncols, P.prec), ml.GpuVector(P.nrows, P.prec)
    n = lattice_products()
    ml.gemm(1.0, P, c, 0.0, f)
    ml.gemm(1.0, P, f, 0.0, c, job="tn")
    return lattice_products() - n
P = lat.interpolation(dim, order, 2)
own = 2 if dim == 3 else 0
assert products(P) == products(P.convert(F.F32)) == own
if order == 2:
    P.storage(F.STORAGE_STENCIL)
    assert products(P) == own
assert P.storage(F.STORAGE_SELL) == F.STORAGE_SELL
assert products(P) == products(P.convert(F.F32)) == 0
sm = it.Jacobi(0.5) if order == 1 else it.GeometricSSC(1.0)
Hy = it.Hierarchy.lattice(it.GeometricCS(sm), dim, order, 1, 3)
x, b, r = (ml.GpuVector(Hy.top_matrix().nrows) for _ in range(3))
n = lattice_products()
Hy.apply(x, b, r)
assert (lattice_products() > n) == (dim == 3)
for l in range(2):
    Hy.level_matrix(l, interp=True).storage(F.STORAGE_SELL)
g, n = H.host_hip_graphs_destroyed(), lattice_products()
Hy.apply(x, b, r)
assert lattice_products() == n
assert H.host_hip_graphs_destroyed() == g + (dim == 3)
del Hy
""", dim, order)


@pytest.mark.parametrize("dim,smoother", [(2, "GeometricSSC"), (3, "GeometricSSC"),
                                          (3, "GeometricPSC")])
def test_a_hierarchy_is_built_where_only_its_rows_fit(host_hip, dim, smoother):
    """with a coefficient finer than the lattice an order-2 hierarchy keeps its element matrices
    if there is memory for them; with no more than one per cell takes, it is built without them"""
    run(host_hip, """
dim, sm = int(sys.argv[3]), getattr(it, sys.argv[4])
cs = it.GeometricCS(sm(0.5), 1, 1, 0)
n = 24 if dim == 2 else 8
kaps = {nk: ml.GpuVector(nk ** dim) for nk in (n, 2 * n)}
start = H.host_hip_live()
def build(nk, room):
    H.host_hip_limit(start + room)
    try:
        return it.Hierarchy.lattice(cs, dim, 2, n // 4, 3, kappa=(kaps[nk], nk))
    finally:
        H.host_hip_limit(1 << 60)
def fits(nk, room):
    try:
        build(nk, room)
        return True
    except Exception:
        return False
def least(nk):  # memory, to 1 %
    lo, hi = 0, 1 << 32
    while hi > lo * 1.01 + 4096:
        mid = (lo + hi) // 2
        lo, hi = (lo, mid) if fits(nk, mid) else (mid, hi)
    return hi
room = 1.03 * least(n)  # one factor per cell on the top level
assert fits(2 * n, int(room))
def sweeps(Hy):
    x, b, r = (ml.GpuVector(Hy.top_matrix().nrows) for _ in range(3))
    k = [H.host_hip_launches(q) for q in (b"k_blk_cell", b"k_blk_sweep")]
    Hy.apply(x, b, r)
    return [H.host_hip_launches(q) > o for q, o in zip((b"k_blk_cell", b"k_blk_sweep"), k)]
assert sweeps(build(2 * n, int(room))) == [False, True]  # from the rows
assert sweeps(build(2 * n, 1 << 32)) == [True, False]  # from the element matrices
""", dim, smoother)


def test_geometric_interpolations_hold_no_value_planes(host_hip):
    """the planes that products of changed values read are made when the values change, not for
    the trilinear weights, which no product reads; a converted copy follows"""
    run(host_hip, """
fills = lambda: H.host_hip_launches(b"k_tp8_fill")
P = lat.interpolation(3, 1, 6)
Q = P.convert(F.F32)
Hy = it.Hierarchy.lattice(it.GeometricCS(it.Jacobi(0.5)), 3, 1, 1, 3)
assert fills() == 0
P.update_values(np.ones(P.nnz))
assert fills() == 1
R = P.convert(F.F32)
assert fills() == 2
del Hy
""")
