"""GPU tests of the products of a caller's matrices around the lines where their form changes:
SELL, or the CSR with four or eight lanes a row."""
import numpy as np
import pytest
import scipy.sparse as sp

from gnu_femlisp_amd import flgpu as F
from gnu_femlisp_amd.flgpu import check, lib
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


@pytest.mark.parametrize("prec", [F.F64, F.F32])
@pytest.mark.parametrize("rows,mean,longest", [(70, 3, 40), (5000, 6, 9), (5000, 8, 60)])
def test_sweeps_of_irregular_rows_follow_changed_values(rows, mean, longest, prec):
    """colour sweeps read the values that the matrix has: after a change, and in a copy of the
    other precision, they equal those of a matrix built with these values, bit for bit"""
    print(f"irregular sweeps {rows} mean {mean} longest {longest} prec={prec}", flush=True)
    rng = np.random.default_rng(rows + mean)
    per = np.minimum(rng.geometric(2.0 / mean, rows), longest // 2)
    i = np.repeat(np.arange(rows), per)
    j = np.minimum(i + 1 + rng.integers(0, 60, i.size), rows - 1)
    S = sp.csr_matrix((np.ones(i.size), (i, j)), shape=(rows, rows))
    S = S + S.T + sp.eye(rows)
    S = S.tocsr()
    S.sort_indices()
    vals = []
    for _ in range(2):
        v = -rng.uniform(0.1, 1.0, S.nnz)
        v[S.indices == np.repeat(np.arange(rows), np.diff(S.indptr))] = 60.0
        vals.append(v)
    other = F.F32 if prec == F.F64 else F.F64
    A = GpuSparseMatrix.from_csr(S.indptr, S.indices, vals[0], prec=prec)
    A.colour_greedy()
    A.update_values(vals[1])
    B = GpuSparseMatrix.from_csr(S.indptr, S.indices, vals[1], prec=prec)
    B.colour_greedy()
    y, c = rng.uniform(-1, 1, rows), rng.uniform(-1, 1, rows)

    def sweep(M):
        x, b, r = (GpuVector.from_array(a, M.prec) for a in (y, c, c))
        for bw in (0, 1):
            check(lib().flgpu_sor_iterate(M.h, 1.1, bw, x.h, b.h, r.h))
        return x.numpy(), r.numpy()

    for P, Q in ((A, B), (A.convert(other), B.convert(other))):
        for p, q in zip(sweep(P), sweep(Q)):
            assert np.array_equal(p, q) and np.isfinite(p).all()
    if prec == F.F64:  # and the sweep is the sequential one in (colour, index) order
        x = y.copy()
        D = sp.csr_matrix((vals[1], S.indices, S.indptr))
        colour = np.full(rows, -1)
        for r in range(rows):
            used = set(colour[D.indices[D.indptr[r]:D.indptr[r + 1]]].tolist())
            k = 0
            while k in used:
                k += 1
            colour[r] = k
        for order in (np.argsort(colour, kind="stable"), np.argsort(-colour, kind="stable")):
            for r in order:
                s = slice(D.indptr[r], D.indptr[r + 1])
                x[r] += 1.1 * (c[r] - D.data[s] @ x[D.indices[s]]) / 60.0
        assert np.abs(sweep(A)[0] - x).max() < 1e-12
