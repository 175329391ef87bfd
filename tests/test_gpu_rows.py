"""GPU tests of the products of a caller's matrices around the lines where their form changes:
SELL, or the CSR with four or eight lanes a row."""
import numpy as np
import pytest
import scipy.sparse as sp

from gnu_femlisp_amd import flgpu as F
from gnu_femlisp_amd.matlisp import GpuSparseMatrix, GpuVector, compute_residual, gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [F.F64, F.F32])
@pytest.mark.parametrize("rows,short,long", [(30001, 5, 13), (30001, 12, 20), (30001, 14, 22),
                                             (100000, 8, 14), (100001, 5, 9), (100001, 8, 14),
                                             (100001, 10, 22), (100001, 12, 18),
                                             (300001, 10, 14), (300001, 8, 16)])
def test_products_of_irregular_rows(rows, short, long, prec):
    """rows of `short` to `long` entries, a few empty ones: nn, tn and the residual against scipy;
    a sum of w products of values up to 1 rounds by at most w eps per term"""
    print(f"irregular rows {rows} of {short}..{long} prec={prec}", flush=True)
    rng = np.random.default_rng(rows + short)
    lens = rng.integers(short, long + 1, rows)
    lens[rng.integers(0, rows, 5)] = 0
    row = np.repeat(np.arange(rows), lens)
    col = np.clip(row + rng.integers(-900, 901, row.size), 0, rows - 1)
    S = sp.csr_matrix((rng.uniform(-1, 1, row.size), (row, col)), shape=(rows, rows))
    S.data = S.data.astype(np.float32).astype(float)
    S.sort_indices()
    A = GpuSparseMatrix.from_scipy(S, prec=prec)
    x, y = (rng.uniform(-1, 1, rows).astype(np.float32).astype(float) for _ in range(2))
    tol = 2 * (long + 1) ** 2 * (2.0 ** -53 if prec == F.F64 else 2.0 ** -24)
    xv, yv, r = GpuVector.from_array(x, prec), GpuVector.from_array(y, prec), GpuVector(rows, prec)
    compute_residual(A, xv, yv, r)
    assert np.abs(r.numpy() - (y - S @ x)).max() <= tol
    gemm(0.5, A, xv, 2.0, yv)
    assert np.abs(yv.numpy() - (0.5 * (S @ x) + 2.0 * y)).max() <= tol
    yv = GpuVector.from_array(y, prec)
    gemm(1.0, A, xv, 0.0, yv, job="tn")
    w = np.diff(S.tocsc().indptr).max()
    assert np.abs(yv.numpy() - S.T @ x).max() <= tol * max(1, w / long) ** 2
