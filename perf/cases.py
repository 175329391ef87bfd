"""The work that users of this library have it do, as cases to time.

A case is a dict of plain values.  Its "kind" is one of

- "solve":    a linear system -div(kappa grad u) = f on a uniformly refined cube, solved to
              1e-10 by a multigrid-preconditioned (flexible) CG (iteration.solve on a
              blackboard, as tests/test_gpu_configs.py and bench.py do), and the solution
              brought to the host.  With "renew" the coefficient is new in every pass: every
              level is assembled again first, as in a time step, a nonlinear iteration or an
              inverse problem.
- "csr":      a caller's own sparse matrix (irregular rows, no lattice): plain CG to 1e-10.
- "sweep":    Gauss-Seidel steps on a caller's own matrix, its residual and a transposed
              product (the matlisp generics gemm nn / tn), FP64 or FP32.
- "train":    loss and gradient of the learned correction's network on a batch.
- "forward":  the network's forward pass.

listed() holds the sizes of the reference configurations and of the tests, draw() gives others
of the same ranges.
"""
import math

import numpy as np
import torch

from gnu_femlisp_amd import flgpu as F
from gnu_femlisp_amd import iteration as it
from gnu_femlisp_amd import lattice as lat
from gnu_femlisp_amd import learned
from gnu_femlisp_amd import matlisp as ml
from gnu_femlisp_amd.fields import gaussian_log_field, inclusions

TOL = 1e-10


def _solve(name, dim, order, n0, levels, field, smoother, omega, steps, base, prec, transfer,
           renew):
    return {"name": name, "kind": "solve", "dim": dim, "order": order, "n0": n0,
            "levels": levels, "field": field, "smoother": smoother, "omega": omega,
            "steps": steps, "base": base, "prec": prec, "transfer": transfer, "renew": renew}


def listed():
    return [
        # the smallest solve: 2D Poisson, 32 x 32 cells, damped <jacobi>: launches and latency
        _solve("poisson2d_32", 2, 1, 1, 6, "one", "jacobi", 0.6, 2, 0, "f64", "geometric", False),
        # 2D Q2 with femlisp's default smoother for order 2, on a lattice of odd extent
        _solve("q2_2d_96", 2, 2, 3, 6, "lognormal", "ssc", 1.0, 1, 0, "f64", "geometric", False),
        # 3D Poisson with multicolour Gauss-Seidel, 64^3 cells
        _solve("poisson3d_64", 3, 1, 1, 7, "one", "sor", 1.0, 2, 0, "f64", "geometric", False),
        # variable coefficient, Q2, 48^3 cells, block smoother, FP32 cycle in FP64 flexible CG
        _solve("q2_48_mixed", 3, 2, 3, 5, "lognormal", "ssc", 1.0, 1, 0, "f32", "geometric",
               False),
        # two-phase material with contrast 1e4, 128^3 cells: the fastest configuration ...
        _solve("inclusions_128_mixed", 3, 1, 1, 8, "inclusions", "jacobi", 0.9, 2, 4, "f32",
               "blackbox", False),
        # ... and femlisp's own plain FP64 geometric multigrid on the same problem (the largest)
        _solve("inclusions_128_plain", 3, 1, 1, 8, "inclusions", "sor", 1.0, 2, 3, "f64",
               "geometric", False),
        # a new coefficient in every pass, Q1 on 96^3 cells: assembly, operator-dependent
        # transfers, Galerkin products, the coarse inverse, then the solve
        _solve("renew_q1_96", 3, 1, 3, 6, "inclusions", "jacobi", 0.9, 2, 2, "f32", "blackbox",
               True),
        # a new coefficient in every pass, Q2 on 24^3 cells, all in FP64
        _solve("renew_q2_24", 3, 2, 3, 4, "lognormal", "ssc", 1.0, 1, 0, "f64", "geometric",
               True),
        # a caller's own matrix: plain CG, and FP32 smoothing with nn and tn products
        {"name": "csr_cg", "kind": "csr", "rows": 300007, "degree": 18, "prec": "f64"},
        {"name": "csr_sweeps_f32", "kind": "sweep", "rows": 60001, "degree": 12, "steps": 8,
         "prec": "f32"},
        # the learned correction: a training batch as tests and bench.py train it, and one
        # sample's forward pass as the solver calls it
        {"name": "train_32x32", "kind": "train", "batch": 32, "n": 32},
        {"name": "forward_1x32", "kind": "forward", "batch": 1, "n": 32},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_solve(rng):
    dim = rng.choice([2, 3, 3])
    order = rng.choice([1, 1, 2])
    renew = rng.random() < 0.35
    n0 = rng.choice([1, 2, 3, 5])
    if dim == 2:
        cap = 512 if order == 1 else 160
    else:
        cap = 112 if order == 1 else 32
    top = int(math.log2(cap / n0))
    levels = rng.randint(3, max(3, top + 1))
    prec = rng.choice(["f64", "f32"])
    if dim == 3 and order == 1 and rng.random() < 0.5 and levels >= 4:
        # contrast 1e4 needs the operator-dependent transfers and a resolved coarse solve
        base = max(l for l in range(levels - 1) if l == 0 or (n0 << l) <= 12)
        return _solve("", 3, 1, n0, levels, "inclusions", "jacobi", 0.9, 2, base, prec,
                      "blackbox", renew)
    field = rng.choice(["one", "lognormal"]) if not renew else "lognormal"
    base = 1 if n0 == 1 and order == 1 else 0
    if order == 2:
        return _solve("", dim, 2, n0, levels, field, "ssc", 1.0, 1, base, prec, "geometric",
                      renew)
    sm, om = rng.choice([("jacobi", 0.6), ("sor", 1.0)])
    return _solve("", dim, 1, n0, levels, field, sm, om, 2, base, prec, "geometric", renew)


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "solve", "csr", "sweep", "train", "forward"])
    if kind == "solve":
        c = _draw_solve(rng)
    elif kind == "csr":
        c = {"kind": "csr", "rows": _log_int(rng, 2000, 400000), "degree": rng.randint(6, 24),
             "prec": "f64"}
    elif kind == "sweep":
        c = {"kind": "sweep", "rows": _log_int(rng, 2000, 100000), "degree": rng.randint(6, 24),
             "steps": rng.randint(2, 10), "prec": rng.choice(["f64", "f32"])}
    elif kind == "train":
        c = {"kind": "train", "batch": rng.randint(1, 24), "n": 4 * rng.randint(3, 8)}
    else:
        n = 4 * rng.randint(3, 16)
        c = {"kind": "forward", "batch": rng.randint(1, max(1, min(8, 100000 // n ** 3))), "n": n}
    c.pop("name", None)
    return c


# ---- inputs ---------------------------------------------------------------------------------


def _cells(c):
    return c["n0"] << (c["levels"] - 1)


def _field(c, seed):
    """the per-cell coefficient (nk = n cells per axis), None for kappa = 1"""
    n, dim = _cells(c), c["dim"]
    if c["field"] == "one":
        return None
    if c["field"] == "lognormal":
        return np.exp(np.random.default_rng(seed).normal(scale=1.5, size=(n,) * dim))
    r = max(1.5, 3.0 * n / 128)
    return inclusions(n, seed=seed, frac=0.30, rmin=r, rmax=r * 8 / 3, contrast=1e4)


def _rhs(c, seed):
    """U[-1, 1] per interior DOF, zero on the Dirichlet boundary"""
    M, dim = c["order"] * _cells(c) + 1, c["dim"]
    b = np.zeros((M,) * dim)
    inner = (slice(1, M - 1),) * dim
    b[inner] = np.random.default_rng(seed + 1).uniform(-1, 1, (M - 2,) * dim)
    return b.ravel()


def _graph(c, seed):
    """CSR of a weighted graph Laplacian plus a shift: neighbours near in the numbering, row
    lengths irregular, ascending columns"""
    n, deg = c["rows"], c["degree"]
    rng = np.random.default_rng(seed)
    w = 4 * int(math.sqrt(n)) + 2
    per = np.minimum(rng.geometric(2.0 / deg, n), 2 * deg)  # edges to later rows
    i = np.repeat(np.arange(n), per)
    j = i + 1 + (w * rng.random(i.size) ** 3).astype(np.int64)
    ok = j < n
    key = np.unique(i[ok] * n + j[ok])
    i, j = key // n, key % n
    v = -np.exp(rng.normal(scale=0.5, size=i.size))
    d = np.bincount(i, -v, n) + np.bincount(j, -v, n)
    d = d * 1.02 + 0.05
    k = np.arange(n)
    rows, cols = np.concatenate([i, j, k]), np.concatenate([j, i, k])
    vals = np.concatenate([v, v, d])
    o = np.argsort(rows * n + cols)
    ptr = np.zeros(n + 1, np.int64)
    ptr[1:] = np.cumsum(np.bincount(rows, minlength=n))
    return ptr.astype(np.int32), cols[o].astype(np.int32), vals[o], rng


# the network's layers: input channels, output channels, level
_CIN = [2, 16, 16, 32, 32, 64, 96, 48, 16]
_COUT = [16, 16, 32, 32, 64, 64, 32, 16, 1]


def _net_values(c, seed):
    """parameters (He-scaled), inputs [r / rms(r), log(kappa) / 4] and targets of a batch"""
    rng = np.random.default_rng(seed)
    th = []
    for l, (ci, co) in enumerate(zip(_CIN, _COUT)):
        s = math.sqrt(2.0 / (27 * ci)) * (0.1 if l == 8 else 1.0)
        th += [s * rng.normal(size=27 * ci * co), 0.05 * rng.normal(size=co)]
    theta = np.concatenate(th).astype(np.float32)
    B, n = c["batch"], c["n"]
    x = np.empty((B, n, n, n, 2), np.float32)
    x[..., 0] = rng.standard_normal((B, n, n, n), np.float32)
    for s in range(B):
        x[s, ..., 1] = np.log(gaussian_log_field(n, seed + 7 * s)) / 4
    t = rng.standard_normal((B, n, n, n), np.float32)
    for ax in (1, 2, 3):  # the error is smoother than the residual
        t = (t + np.roll(t, 1, ax) + np.roll(t, -1, ax)) / np.float32(math.sqrt(3.0))
    return theta, x, t.astype(np.float32)


def _prec(c):
    return F.F32 if c["prec"] == "f32" else F.F64


def prepare(case, seed):
    kind, st = case["kind"], {"case": case}
    if kind == "solve":
        n, prec = _cells(case), _prec(case)
        kap = _field(case, seed)
        sm = {"jacobi": it.Jacobi, "sor": it.SOR, "ssc": it.GeometricSSC}[case["smoother"]]
        cs = it.GeometricCS(sm(case["omega"]), case["steps"], case["steps"], case["base"],
                            symmetric=True, prec=prec, transfer=case["transfer"])
        kv = None if kap is None else (ml.GpuVector.from_array(kap.ravel()), n)
        mode = F.ASM_MFMA if prec == F.F32 else F.ASM_F64
        H = it.Hierarchy.lattice(cs, case["dim"], case["order"], case["n0"], case["levels"],
                                 kappa=kv, mode=mode)
        if prec == F.F32:
            A, _ = lat.assemble(case["dim"], case["order"], n, kv, prec=F.F64, rhs=False)
        else:
            A = H.top_matrix()
        outer = it.FCG(cs) if prec == F.F32 else it.CG(cs)
        st.update(H=H, A=A, kv=kv, b=ml.GpuVector.from_array(_rhs(case, seed)),
                  x=A.make_domain_vector(),
                  solver=it.LinearSolver(outer, success_if=("<", "reduction", TOL),
                                         failure_if=(">", "step", 600), true_residual=True))
    elif kind in ("csr", "sweep"):
        rp, ci, v, rng = _graph(case, seed)
        A = ml.GpuSparseMatrix.from_csr(rp, ci, v, prec=_prec(case))
        b = rng.uniform(-1, 1, case["rows"])
        st.update(A=A, b=ml.GpuVector.from_array(b, _prec(case)), x=A.make_domain_vector())
        if kind == "csr":
            st["solver"] = it.LinearSolver(it.CG(), success_if=("<", "reduction", TOL),
                                           failure_if=(">", "step", 600))
        else:
            A.colour_greedy()
            st["gs"] = it.make_iterator(it.GaussSeidel(), A, steps=case["steps"])
            st.update(r=A.make_image_vector(), y=A.make_domain_vector())
    else:
        theta, x, t = _net_values(case, seed)
        net = learned.UNet(cin=2, seed=0)
        net.set_params(theta)
        st.update(net=net, xv=ml.GpuVector.from_array(x, F.F32))
        if kind == "train":
            st["tv"] = ml.GpuVector.from_array(t, F.F32)
        else:
            st["yv"] = ml.GpuVector(case["batch"] * case["n"] ** 3, F.F32)
    return st


def run(st):
    c = st["case"]
    if c["kind"] == "solve":
        if c["renew"]:
            st["H"].reassemble(st["kv"])
            if c["prec"] == "f32":
                lat.reassemble(st["A"], st["kv"])
        it.solve(st["solver"], {"matrix": st["A"], "rhs": st["b"], "hierarchy": st["H"],
                                "solution": st["x"]})
        return {"solution": st["x"].numpy()}
    if c["kind"] == "csr":
        it.solve(st["solver"], {"matrix": st["A"], "rhs": st["b"], "solution": st["x"]})
        return {"solution": st["x"].numpy()}
    if c["kind"] == "sweep":
        A, x, b, r, y = (st[k] for k in ("A", "x", "b", "r", "y"))
        ml.x_lt_0(x)
        st["gs"].iterate(x, b, r)
        ml.compute_residual(A, x, b, r)
        ml.gemm(1.0, A, r, 0.0, y, "tn")
        out = {"x": x.numpy(), "residual": r.numpy(), "gradient": y.numpy()}
        return out if c["prec"] == "f64" else {k: v.astype(np.float32) for k, v in out.items()}
    if c["kind"] == "train":
        loss, g = st["net"].loss_grad(st["xv"], st["tv"], c["batch"], c["n"])
        return {"loss": np.float32(loss), "grad": g.astype(np.float32)}
    st["net"].forward(st["xv"], c["batch"], c["n"], st["yv"])
    return {"y": st["yv"].numpy().astype(np.float32)}


# ---- what a pass cannot do without ------------------------------------------------------------


def _solve_steps(c):
    """CG steps to 1e-10 (about what these configurations take)"""
    n = _cells(c)
    if c["field"] == "inclusions":
        return 2 * n if c["transfer"] == "geometric" else max(8, n // 2)
    if c["field"] == "lognormal":
        return 25
    return 9


def work(case):
    c = case
    if c["kind"] == "solve":
        dim, order, n = c["dim"], c["order"], _cells(c)
        N, cells = (order * n + 1) ** dim, n ** dim
        vb = 4 if c["prec"] == "f32" else 8
        row = (2 * order + 1) ** dim  # mean-size row of the operator
        all_levels = 1.0 / (1.0 - 0.5 ** dim)
        passes = 2 * c["steps"] + 1  # smoothing steps and the restricted residual
        blk = (2 * order - 1) ** dim if c["smoother"] == "ssc" else 0
        # per cycle: the cells' coefficients and x, b, x' per pass, twice the transfer
        cyc = all_levels * (passes * (cells * vb + 3 * N * vb) + 3 * N * vb)
        cfl = all_levels * (passes * 2 * row * N + (2 * c["steps"] * blk * 2 * N))
        # per CG step: A p, the updates of x, r, p and the dots, in FP64
        out = cells * 8 + 10 * N * 8
        s = _solve_steps(c)
        by, fl = s * (cyc + out) + 2 * N * 8, s * (cfl + 2 * row * N + 12 * N)
        if c["renew"]:  # the coefficient read, the matrix entries of all levels written
            nz = ((3 * n + 1) if order == 1 else (8 * n + 1)) ** dim
            by += cells * 8 + all_levels * nz * vb
            fl += all_levels * cells * 2 * (order + 1) ** (2 * dim) * (order + 1) ** dim
        return {"bytes": by, "flops": fl}
    if c["kind"] in ("csr", "sweep"):
        n, vb = c["rows"], 4 if c["prec"] == "f32" else 8
        nz = n * (c["degree"] + 1)
        mat, passes = nz * (vb + 4) + 4 * n, 60 if c["kind"] == "csr" else c["steps"] + 2
        vec = (10 if c["kind"] == "csr" else 3) * n * vb
        return {"bytes": passes * (mat + vec), "flops": passes * (2 * nz + 10 * n)}
    vox = [c["batch"] * (c["n"] >> l) ** 3 for l in (0, 0, 1, 1, 2, 2, 1, 0, 0)]
    macs = sum(27 * ci * co * v for ci, co, v in zip(_CIN, _COUT, vox))
    acts = sum((ci + co) * v * 4 for ci, co, v in zip(_CIN, _COUT, vox))
    par = sum(27 * ci * co + co for ci, co in zip(_CIN, _COUT)) * 4
    f = 3 if c["kind"] == "train" else 1
    return {"bytes": f * acts + f * par, "flops": f * 2 * macs}


# ---- the results in 64 bits --------------------------------------------------------------------


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _pcg(apply, diag, b, steps, budget):
    """Jacobi-preconditioned CG in FP64 to the rounding limit; None if it is not reached"""
    x, r = torch.zeros_like(b), b.clone()
    z = r / diag
    p, rz = z.clone(), torch.dot(r, z)
    b2 = float(torch.dot(b, b))
    clock_start = torch.cuda.Event(enable_timing=True) if b.is_cuda else None
    if clock_start is not None:
        clock_start.record()
    for k in range(steps):
        a = apply(p)
        al = rz / torch.dot(p, a)
        x += al * p
        r -= al * a
        if k % 25 == 24:
            if float(torch.dot(r, r)) < 1e-26 * b2:
                # once more from the true residual, which the recurrence drifts from
                r = b - apply(x)
                if float(torch.dot(r, r)) < 1e-24 * b2:
                    return x
                z = r / diag
                p, rz = z.clone(), torch.dot(r, z)
                continue
            if clock_start is not None:
                now = torch.cuda.Event(enable_timing=True)
                now.record()
                now.synchronize()
                if clock_start.elapsed_time(now) > 1e3 * budget:
                    return None
        z = r / diag
        rn = torch.dot(r, z)
        p = z + (rn / rz) * p
        rz = rn
    return None


def _exact_solve(c, seed):
    dim, order, n, dev = c["dim"], c["order"], _cells(c), _device()
    h = 1.0 / n
    if order == 1:
        K1, M1 = [[1, -1], [-1, 1]], [[2, 1], [1, 2]]
        K1, M1 = torch.tensor(K1, dtype=torch.float64) / h, torch.tensor(M1).double() * h / 6
    else:
        K1 = torch.tensor([[7, -8, 1], [-8, 16, -8], [1, -8, 7]]).double() / (3 * h)
        M1 = torch.tensor([[4, 2, -1], [2, 16, 2], [-1, 2, 4]]).double() * h / 30
    E = 0
    for k in range(dim):
        m = torch.ones(1, 1, dtype=torch.float64)
        for l in range(dim):
            m = torch.kron(m, K1 if l == k else M1)
        E = E + m
    E = E.to(dev)
    M, w = order * n + 1, order + 1
    kap = _field(c, seed)
    kap = torch.ones(n ** dim, dtype=torch.float64, device=dev) if kap is None else \
        torch.from_numpy(kap.reshape(-1)).to(dev)
    offs = np.indices((w,) * dim).reshape(dim, -1).T
    slices = [tuple(slice(int(o), int(o) + order * (n - 1) + 1, order) for o in d) for d in offs]
    mask = torch.zeros((M,) * dim, dtype=torch.float64, device=dev)
    mask[(slice(1, M - 1),) * dim] = 1

    def apply(v):
        u = v.view((M,) * dim) * mask
        loc = torch.stack([u[s].reshape(-1) for s in slices])
        loc = torch.matmul(E, loc) * kap
        out = torch.zeros_like(u)
        for k, s in enumerate(slices):
            out[s] += loc[k].view((n,) * dim)
        out = out * mask + v.view((M,) * dim) * (1 - mask)
        return out.reshape(-1)

    diag = torch.zeros((M,) * dim, dtype=torch.float64, device=dev)
    for k, s in enumerate(slices):
        diag[s] += (E[k, k] * kap).view((n,) * dim)
    diag = (diag * mask + (1 - mask)).reshape(-1)
    x = _pcg(apply, diag, torch.from_numpy(_rhs(c, seed)).to(dev), 20000, 15.0)
    return None if x is None else {"solution": x.cpu().numpy()}


def _exact_csr(c, seed):
    dev = _device()
    rp, ci, v, rng = _graph(c, seed)
    n = c["rows"]
    b = rng.uniform(-1, 1, n)
    if c["prec"] == "f32":  # the values as they are handed over
        b, v = b.astype(np.float32).astype(np.float64), v.astype(np.float32).astype(np.float64)
    rows = torch.from_numpy(np.repeat(np.arange(n), np.diff(rp))).to(dev)
    cols, vals = torch.from_numpy(ci.astype(np.int64)).to(dev), torch.from_numpy(v).to(dev)

    def apply(x):
        return torch.zeros(n, dtype=torch.float64, device=dev).index_add_(0, rows, vals * x[cols])

    bt = torch.from_numpy(b).to(dev)
    diag = torch.zeros(n, dtype=torch.float64, device=dev)
    on = rows == cols
    diag[rows[on]] = vals[on]
    if c["kind"] == "csr":
        x = _pcg(apply, diag, bt, 5000, 15.0)
        return None if x is None else {"solution": x.cpu().numpy()}
    # the greedy colouring in index order, then the sweeps colour by colour
    colour = np.full(n, -1, np.int64)
    rl, cl = rp.tolist(), ci.tolist()
    col = colour.tolist()
    for i in range(n):
        used = {col[j] for j in cl[rl[i]:rl[i + 1]] if j != i}
        k = 0
        while k in used:
            k += 1
        col[i] = k
    ct = torch.tensor(col, device=dev)
    x = torch.zeros(n, dtype=torch.float64, device=dev)
    for _ in range(c["steps"]):
        for k in range(max(col) + 1):
            m = ct == k
            x = torch.where(m, x + (bt - apply(x)) / diag, x)
    r = bt - apply(x)
    return {"x": x.cpu().numpy(), "residual": r.cpu().numpy(),
            "gradient": apply(r).cpu().numpy()}  # the matrix is symmetric


def _exact_net(c, seed):
    dev = _device()
    theta, x, t = _net_values(c, seed)
    th = torch.from_numpy(theta).double().to(dev).requires_grad_(c["kind"] == "train")
    par, off = [], 0
    for ci, co in zip(_CIN, _COUT):
        W = th[off:off + 27 * ci * co].view(27, ci, co)
        off += 27 * ci * co
        par.append((W, th[off:off + co]))
        off += co

    def conv(v, l, relu=True):
        W, bias = par[l]
        n = v.shape[1]
        p = torch.nn.functional.pad(v, (0, 0, 1, 1, 1, 1, 1, 1))
        out = bias
        for k in range(27):
            z, y, xx = k // 9, k // 3 % 3, k % 3
            s = p[:, z:z + n, y:y + n, xx:xx + n, :].reshape(-1, v.shape[-1])
            out = out + torch.matmul(s, W[k])
        out = out.view(*v.shape[:4], -1)
        return torch.relu(out) if relu else out

    def pool(v):
        B, n, ch = v.shape[0], v.shape[1] // 2, v.shape[-1]
        return v.view(B, n, 2, n, 2, n, 2, ch).mean(dim=(2, 4, 6))

    def up(v):
        for ax in (1, 2, 3):
            v = torch.repeat_interleave(v, 2, dim=ax)
        return v

    with torch.set_grad_enabled(c["kind"] == "train"):
        a1 = conv(conv(torch.from_numpy(x).double().to(dev), 0), 1)
        a3 = conv(conv(pool(a1), 2), 3)
        a5 = conv(conv(pool(a3), 4), 5)
        a6 = conv(torch.cat([up(a5), a3], -1), 6)
        a7 = conv(torch.cat([up(a6), a1], -1), 7)
        y = conv(a7, 8, relu=False).reshape(-1)
        if c["kind"] == "forward":
            return {"y": y.cpu().numpy()}
        loss = ((y - torch.from_numpy(t).double().to(dev).reshape(-1)) ** 2).mean()
        loss.backward()
    return {"loss": float(loss.detach()), "grad": th.grad.cpu().numpy()}


def exact(case, seed):
    if case["kind"] == "solve":
        return _exact_solve(case, seed)
    if case["kind"] in ("csr", "sweep"):
        return _exact_csr(case, seed)
    return _exact_net(case, seed)
