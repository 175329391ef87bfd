"""GPU tests of what follows a change of a matrix or hierarchy that is in use: new coefficients
while a cycle is queued, other values or another storage form, converted copies."""
import sys

import numpy as np
import pytest
import scipy.sparse as sp

from gnu_femlisp_amd import flgpu as F
from gnu_femlisp_amd import iteration as it
from gnu_femlisp_amd import lattice as lat
from gnu_femlisp_amd.flgpu import check, lib
from gnu_femlisp_amd.matlisp import GpuVector, compute_residual, gemm
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def relerr(x, y):
    d = np.linalg.norm(y)
    return np.linalg.norm(x - y) / (d if d > 0 else 1.0)


@pytest.mark.parametrize("dim,order,smoother", [(2, 1, it.Jacobi(0.6)), (2, 1, it.SOR(1.0)),
                                                (2, 2, it.GeometricSSC(1.0)),
                                                (3, 2, it.GeometricSSC(1.0))])
def test_reassembly_right_after_a_queued_cycle(dim, order, smoother):
    """a cycle, new coefficients and a cycle again, with no host read in between, equal the same
    cycles of hierarchies of their own (the later cycles replace captured ones)"""
    say(f"queued cycle, reassembly, cycle: dim={dim} order={order} {type(smoother).__name__}")
    m, levels = 3, 4 if dim == 2 else 2
    n = m << (levels - 1)
    rng = np.random.default_rng(dim + order)
    kaps = [np.exp(rng.normal(size=(n,) * dim)) for _ in range(3)]
    kvs = [GpuVector.from_array(k.ravel()) for k in kaps]
    cs = it.GeometricCS(smoother, 2, 2, 0)
    H = it.Hierarchy.lattice(cs, dim, order, m, levels, kappa=kaps[0])
    N = H.top_matrix().nrows
    bh = rng.uniform(-1, 1, N)
    x, b, r = (GpuVector.from_array(a) for a in (np.zeros(N), bh, bh))
    check(lib().flgpu_mg_apply(H.h, x.h, b.h, r.h))
    for kv in kvs[1:]:
        check(lib().flgpu_mg_reassemble(H.h, kv.h, n))
        compute_residual(H.top_matrix(), x, b, r)
        check(lib().flgpu_mg_apply(H.h, x.h, b.h, r.h))
    y, q = GpuVector.from_array(np.zeros(N)), GpuVector.from_array(bh)
    for k, kap in enumerate(kaps):
        G = it.Hierarchy.lattice(cs, dim, order, m, levels, kappa=kap)
        if k:
            compute_residual(G.top_matrix(), y, b, q)
        check(lib().flgpu_mg_apply(G.h, y.h, b.h, q.h))
        y.numpy()
    assert relerr(x.numpy(), y.numpy()) < 1e-13


@pytest.mark.parametrize("prec", [F.F64, F.F32])
@pytest.mark.parametrize("capped", ["levels", "interpolations"])
@pytest.mark.parametrize("m,levels", [(1, 4), (3, 3)])
def test_galerkin_levels_of_capped_hierarchies(m, levels, capped, prec):
    """reassembled black-box hierarchies hold the same level matrices, bit for bit, where the
    levels or their interpolations were capped to SELL and their products read the CSRs"""
    say(f"galerkin levels capped m={m} levels={levels} {capped} prec={prec}")
    n = m << (levels - 1)
    rng = np.random.default_rng(n)
    kap = [np.exp(rng.normal(size=(n,) * 3)) for _ in range(2)]
    vals = []
    for cap in (False, True):
        cs = it.GeometricCS(it.Jacobi(0.6), 1, 1, 0, prec=prec, transfer="blackbox")
        H = it.Hierarchy.lattice(cs, 3, 1, m, levels, kappa=kap[0])
        if cap:
            for l in range(levels - (capped == "interpolations")):
                M = H.level_matrix(l, interp=capped == "interpolations")
                assert M.storage(F.STORAGE_SELL) == F.STORAGE_SELL
        H.reassemble(kap[1])
        vals.append([H.level_matrix(l).csr()[2] for l in range(levels)])
    for a, b in zip(*vals):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("dim,m,levels", [(1, 2, 4), (2, 1, 4), (2, 3, 3), (3, 1, 3), (3, 2, 2)])
@pytest.mark.parametrize("smoother", ["ssc", "psc", "sor"])
@pytest.mark.parametrize("changed", [False, True])
def test_successive_cycles_start_their_levels_from_zero(dim, m, levels, smoother, changed):
    """three cycles in a row on one order-2 hierarchy, as assembled and with transfers whose
    values were stored anew (products from the CSR), equal the oracle's, each of which starts its
    coarse levels from zero: a cycle's rounding is 1e-12 of its correction, and there are three"""
    say(f"successive cycles dim={dim} m={m} levels={levels} {smoother} changed={changed}")
    n = m << (levels - 1)
    rng = np.random.default_rng(dim + m)
    kap = np.exp(rng.normal(size=(n,) * dim))
    sm, kind, omega = {"ssc": (it.GeometricSSC(1.0), po.SMOOTH_SSC, 1.0),
                       "psc": (it.GeometricPSC(0.2), po.SMOOTH_PSC, 0.2),
                       "sor": (it.SOR(1.0), po.SMOOTH_SOR, 1.0)}[smoother]
    cs = it.GeometricCS(sm, 1, 1, 0, symmetric=True)
    H = it.Hierarchy.lattice(cs, dim, 2, m, levels, kappa=kap)
    if changed:
        for l in range(levels - 1):
            P = H.level_matrix(l, interp=True)
            P.update_values(P.csr()[2])
    oh = po.Hierarchy(dim, 2, m, levels, kappa=kap)
    prm = po.params(smoother=kind, omega=omega, ordering=po.ORDER_COLOUR, pre_steps=1,
                    post_steps=1, base_level=0, symmetric=1, alias=0)
    A = H.top_matrix()
    b = rng.uniform(-1, 1, A.nrows)
    b[po.boundary(dim, 2, n)] = 0
    x, bv, r = (GpuVector.from_array(a) for a in (np.zeros(A.nrows), b, b))
    rp, ci, v = oh.matrix()
    S = sp.csr_matrix((v, ci, rp))
    y = np.zeros(A.nrows)
    for _ in range(3):
        H.apply(x, bv, r)
        compute_residual(A, x, bv, r)
        y = y + oh.apply(prm, b - S @ y)
        assert relerr(x.numpy(), y) < 3e-12


@pytest.mark.parametrize("prec", [F.F64, F.F32])
@pytest.mark.parametrize("order,nc", [(1, 1), (1, 6), (2, 1), (2, 4)])
def test_converted_interpolations_follow_changed_values(order, nc, prec):
    """copies in the other precision of a 3D interpolation, made before and after its values were
    changed, multiply with the values that it had (scipy, FP64)"""
    say(f"converted interpolations order={order} nc={nc} prec={prec}")
    other = F.F32 if prec == F.F64 else F.F64
    rng = np.random.default_rng(nc)
    P = lat.interpolation(3, order, nc, prec=prec)
    rp, ci, v = P.csr()
    copies = [(P.convert(other), v)]
    v = (v * rng.uniform(0.5, 1.5, v.size)).astype(np.float32).astype(float)
    P.update_values(v)
    copies.append((P.convert(other), v))
    copies.append((copies[-1][0].convert(prec), v))
    xc = rng.uniform(-1, 1, P.ncols).astype(np.float32).astype(float)
    yf = rng.uniform(-1, 1, P.nrows).astype(np.float32).astype(float)
    for Q, w in copies:
        S = sp.csr_matrix((w.astype(float), ci, rp), shape=(P.nrows, P.ncols))
        tol = 1e-14 if Q.prec == F.F64 else 2e-6
        f, c = GpuVector(P.nrows, Q.prec), GpuVector(P.ncols, Q.prec)
        gemm(1.0, Q, GpuVector.from_array(xc, Q.prec), 0.0, f)
        gemm(1.0, Q, GpuVector.from_array(yf, Q.prec), 0.0, c, job="tn")
        assert np.abs(f.numpy() - S @ xc).max() <= 8 * tol
        assert np.abs(c.numpy() - S.T @ yf).max() <= 64 * tol
