"""GPU tests of what follows a change of a matrix or hierarchy that is in use: new coefficients
while a cycle is queued, other values or another storage form, converted copies."""
import sys

import numpy as np
import pytest

from gnu_femlisp_amd import flgpu as F
from gnu_femlisp_amd import iteration as it
from gnu_femlisp_amd.flgpu import check, lib
from gnu_femlisp_amd.matlisp import GpuVector, compute_residual

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
