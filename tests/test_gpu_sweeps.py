"""GPU tests of the stencil-form <sor> sweep at the lattice sizes where its tiles change shape."""
import numpy as np
import pytest

from gnu_femlisp_amd import flgpu as F
from gnu_femlisp_amd import lattice as lat
from gnu_femlisp_amd.flgpu import check, lib
from gnu_femlisp_amd.matlisp import GpuVector

pytestmark = pytest.mark.gpu


def relerr(x, y):
    d = np.linalg.norm(y)
    return np.linalg.norm(x - y) / (d if d > 0 else 1.0)


@pytest.mark.parametrize("n,prec,sym", [(131, F.F64, True), (132, F.F64, False),
                                        (131, F.F32, False), (132, F.F32, True),
                                        (144, F.F32, True)])
def test_stencil_sor_taller_tiles(n, prec, sym):
    """tiles of 12 lines up to 132 nodes a side, above of 16 or, in FP32 where that leaves fewer
    idle lines in the last tile, of 20: equal to the SELL colour sweep, forwards and backwards;
    rounding as for the sweep's other shapes"""
    print(f"stencil sor tiles n={n} prec={prec} sym={sym}", flush=True)
    rng = np.random.default_rng(n)
    kap = np.exp(rng.normal(size=(n, n, n)))
    A, _ = lat.assemble(3, 1, n, kap, prec=prec)
    B, _ = lat.assemble(3, 1, n, kap, prec=prec)
    if not sym:
        v = A.csr()[2]
        v = v * (1.0 + 0.1 * rng.uniform(-1, 1, v.size))
        A.update_values(v)
        B.update_values(v)
    assert A.storage(F.STORAGE_STENCIL) == F.STORAGE_STENCIL
    assert B.storage(F.STORAGE_SELL) == F.STORAGE_SELL
    tol = 1e-13 if prec == F.F64 else 2e-6
    y, c = rng.uniform(-1, 1, A.nrows), rng.uniform(-1, 1, A.nrows)
    for bw in (0, 1):
        out = []
        for M in (A, B):
            x, r, b = (GpuVector.from_array(a, prec) for a in (y, c, c))
            check(lib().flgpu_sor_iterate(M.h, 1.1, bw, x.h, b.h, r.h))
            out.append((x.numpy(), r.numpy()))
        assert relerr(out[0][0], out[1][0]) < tol, bw
        assert relerr(out[0][1], out[1][1]) < 10 * tol, bw
