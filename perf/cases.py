"""Measured cases: the work a user of this library has it do, over its public
entry points (the Python mirror of MTL4's interface).

Every listed case says what it stands for.  draw() gives further cases of the
same ranges (grid sides, row counts, layouts, preconditioners), odd sizes
included.  Inputs are made from the seed alone: coefficients, right-hand sides
and start vectors of another seed are other ones.  Right-hand sides of solves
are b = A * x_true, so exact() is x_true; the right-hand sides of a serving
request come from the request's own seed, so there it solves the systems.

Solves run to a tolerance whose error in x lies below the bounds two
implementations are compared by: 1e-10 for CG (relative residual, as in
bench.py), 1e-12 where the error of a converged x varies with rounding
(BiCGSTAB's residual is not monotone).
"""
import math

import numpy as np
import torch

import mtl4_amd as m
from mtl4_amd import _lib
from mtl4_amd import generators as gen

DEV = "cuda"


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # a small 2-D Poisson solve (4096 rows), a solver handle reused by a program that solves often:
        # launch and reduction latency count, not bandwidth
        {"name": "cg_poisson2d_64", "kind": "cg", "matrix": "poisson2d", "size": 64, "layout": "default",
         "call": "handle"},
        # a mid-sized odd 3-D diffusion problem (226,981 rows), MTL4's one-shot call itl::cg(A, x, b, P, iter)
        {"name": "cg_diffusion3d_61", "kind": "cg", "matrix": "diffusion3d", "size": 61, "layout": "default",
         "call": "once"},
        # the headline solve: 4,096,000 rows, the symmetric diagonal layout the autotuner picks for it
        {"name": "cg_diffusion3d_160", "kind": "cg", "matrix": "diffusion3d", "size": 160, "layout": "sym",
         "call": "handle"},
        # an unstructured symmetric system (graph, network): CSR/sliced products inside CG
        {"name": "cg_graph_70001", "kind": "cg", "matrix": "random_spd", "size": 70001, "layout": "default",
         "call": "once"},
        # mixed precision refined to FP64 accuracy (FP32 values and recurrence)
        {"name": "mixed_cg_diffusion3d_110", "kind": "mixed", "matrix": "diffusion3d", "size": 110,
         "layout": "default", "format": "f32"},
        # incomplete Cholesky: the triangular sweeps of a 3-D grid factor dominate
        {"name": "cg_ic0_diffusion3d_100", "kind": "cg_ic0", "matrix": "diffusion3d", "size": 100,
         "layout": "default"},
        # one implicit step of transient convection-diffusion: BiCGSTAB + ILU(0) on a 2-D grid factor
        {"name": "bicgstab_ilu0_convdiff_700", "kind": "bicgstab_ilu0", "matrix": "convdiff2d", "size": 700,
         "layout": "default"},
        # a nonsymmetric unstructured system: BiCGSTAB with the diagonal preconditioner
        {"name": "bicgstab_random_300007", "kind": "bicgstab", "matrix": "random", "size": 300007,
         "layout": "default"},
        # y = A*x with scattered columns and ragged rows, x larger than one XCD's L2
        {"name": "spmv_random_1000003", "kind": "spmv", "matrix": "random", "size": 1000003, "layout": "default"},
        # ILU(0) of an unstructured matrix: solve(P, x) and adjoint_solve(P, x), level-scheduled sweeps
        {"name": "ilu0_solves_graph_120011", "kind": "pc_solves", "matrix": "random_spd", "size": 120011,
         "layout": "default"},
        # many independent systems of uneven size (256 to 16384 rows, three families) in one call, FP64
        {"name": "batched_cg_160", "kind": "batched", "systems": 160, "rows": 16384, "format": "f64"},
        # a burst of serving requests: cg and bicgstab, diagonal and ilu_0, one or two right-hand sides each
        {"name": "serve_burst_48", "kind": "serve", "systems": 16, "rows": 3000, "requests": 48},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cg", "cg", "cg", "cg", "mixed", "cg_ic0", "bicgstab_ilu0", "bicgstab", "spmv", "spmv",
                       "pc_solves", "batched", "serve"])
    if kind == "cg":
        matrix = rng.choice(["poisson2d", "diffusion3d", "diffusion3d", "random_spd"])
        c = {"kind": kind, "matrix": matrix, "call": rng.choice(["once", "handle"])}
        if matrix == "poisson2d":
            c.update(size=_log_int(rng, 12, 700), layout=rng.choice(["default", "sym"]))
        elif matrix == "diffusion3d":
            c.update(size=_log_int(rng, 9, 158), layout=rng.choice(["default", "sym"]))
        else:
            c.update(size=_log_int(rng, 500, 600000), layout="default")
        return c
    if kind == "mixed":
        return {"kind": kind, "matrix": "diffusion3d", "size": rng.randint(20, 130),
                "layout": rng.choice(["default", "sym"]), "format": "f32"}
    if kind == "cg_ic0":
        return {"kind": kind, "matrix": rng.choice(["diffusion3d", "poisson2d"]), "size": rng.randint(21, 110),
                "layout": "default"}
    if kind == "bicgstab_ilu0":
        return {"kind": kind, "matrix": "convdiff2d", "size": _log_int(rng, 40, 900), "layout": "default"}
    if kind == "bicgstab":
        return {"kind": kind, "matrix": rng.choice(["random", "convdiff2d"]), "size": 0, "layout": "default",
                "rows": _log_int(rng, 2000, 700000)}
    if kind == "spmv":
        matrix = rng.choice(["random", "random_spd", "diffusion3d", "convdiff2d"])
        size = {"random": lambda: _log_int(rng, 3000, 1200000), "random_spd": lambda: _log_int(rng, 3000, 1200000),
                "diffusion3d": lambda: _log_int(rng, 15, 130), "convdiff2d": lambda: _log_int(rng, 60, 1200)}[matrix]()
        return {"kind": kind, "matrix": matrix, "size": size, "layout": "default"}
    if kind == "pc_solves":
        return {"kind": kind, "matrix": rng.choice(["random_spd", "convdiff2d"]), "size": 0, "layout": "default",
                "rows": _log_int(rng, 2000, 150000)}
    if kind == "batched":
        return {"kind": kind, "systems": rng.randint(24, 150), "rows": _log_int(rng, 700, 16384),
                "format": rng.choice(["f64", "f32"])}
    return {"kind": "serve", "systems": rng.randint(6, 16), "rows": rng.randint(600, 3000),
            "requests": rng.randint(12, 48)}


# ------------------------------------------------------------------ matrices
def _rand(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1000003 + salt)
    return g


def _uniform(n, seed, salt):
    return torch.rand(n, generator=_rand(seed, salt), device=DEV, dtype=torch.float64) * 2.0 - 1.0


def _stencil_csr(cols, vals, valid):
    """Row-major CSR of (rows, entries) candidates, on the host."""
    counts = valid.sum(1)
    rowptr = torch.zeros(len(counts) + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(counts, 0, out=rowptr[1:])
    return (rowptr.to(torch.int32).cpu().numpy(), cols[valid].to(torch.int32).cpu().numpy(),
            vals[valid].cpu().numpy())


def _diffusion3d(n, seed):
    """7-point diffusion on n^3 cells, face coefficients log-uniform in [1e-2, 1e2], Dirichlet faces."""
    def faces(shape, salt):
        u = torch.rand(shape, generator=_rand(seed, salt), device=DEV, dtype=torch.float64)
        return torch.pow(10.0, u * 4.0 - 2.0)
    kx, ky, kz = faces((n, n, n + 1), 1), faces((n, n + 1, n), 2), faces((n + 1, n, n), 3)
    w, e, s, t, d, u = (kx[:, :, :-1], kx[:, :, 1:], ky[:, :-1, :], ky[:, 1:, :], kz[:-1], kz[1:])
    N = n ** 3
    r = torch.arange(N, device=DEV)
    i, j, k = r % n, (r // n) % n, r // (n * n)
    offs = [-n * n, -n, -1, 0, 1, n, n * n]
    cols = torch.stack([r + o for o in offs], 1)
    valid = torch.stack([k > 0, j > 0, i > 0, r >= 0, i < n - 1, j < n - 1, k < n - 1], 1)
    vals = torch.stack([a.reshape(N) for a in (-d, -s, -w, w + e + s + t + d + u, -e, -t, -u)], 1)
    return _stencil_csr(cols, vals, valid)


def _convdiff2d(n, seed):
    """Upwind convection-diffusion on n x n points with a mass term (an implicit time step), wind from the seed."""
    theta = float(torch.rand(1, generator=_rand(seed, 4), device=DEV, dtype=torch.float64)) * 2.0 * math.pi
    h = 1.0 / (n + 1)
    wx, wy = 10.0 * math.cos(theta), 10.0 * math.sin(theta)
    N = n * n
    r = torch.arange(N, device=DEV)
    i, j = r // n, r % n
    cols = torch.stack([r + o for o in (-n, -1, 0, 1, n)], 1)
    valid = torch.stack([i > 0, j > 0, r >= 0, j < n - 1, i < n - 1], 1)
    coef = [-1.0 - h * max(wy, 0.0), -1.0 - h * max(wx, 0.0), 4.0 + h * (abs(wx) + abs(wy)) + 0.05,
            -1.0 - h * max(-wx, 0.0), -1.0 - h * max(-wy, 0.0)]
    vals = torch.tensor(coef, device=DEV, dtype=torch.float64).repeat(N, 1)
    vals = vals * (1.0 + 0.02 * torch.rand(N, 1, generator=_rand(seed, 5), device=DEV, dtype=torch.float64))
    return _stencil_csr(cols, vals, valid)


def _coo_csr(n, keys, vals):
    """CSR of sorted row*n+col keys; the diagonal becomes sum|offdiag| + 1 (values are multiples of 1/1024, so
    the sum is exact in any order)."""
    rows, cols = keys // n, keys % n
    on = rows == cols
    vals = torch.where(on, torch.zeros_like(vals), vals)
    absum = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, rows, vals.abs())
    vals = torch.where(on, absum[rows] + 1.0, vals)
    rowptr = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(torch.bincount(rows, minlength=n), 0, out=rowptr[1:])
    return rowptr.to(torch.int32).cpu().numpy(), cols.to(torch.int32).cpu().numpy(), vals.cpu().numpy()


def _random(n, seed):
    """Rows of Poisson(16) entries (1 to 256) at uniform columns, dominant diagonal."""
    lens = torch.poisson(torch.full((n,), 16.0, device=DEV), generator=_rand(seed, 6)).clamp(1, 256).long()
    rows = torch.repeat_interleave(torch.arange(n, device=DEV), lens)
    cols = torch.randint(0, n, (len(rows),), generator=_rand(seed, 7), device=DEV)
    diag = torch.arange(n, device=DEV) * (n + 1)
    keys = torch.unique(torch.cat([rows * n + cols, diag]))
    vals = torch.randint(-1024, 1025, (len(keys),), generator=_rand(seed, 8), device=DEV).double() / 1024.0
    return _coo_csr(n, keys, vals)


def _random_spd(n, seed):
    """Symmetric pattern of about 11 entries per row, off-diagonal values in [-1, 0), dominant diagonal."""
    rows = torch.arange(n, device=DEV).repeat_interleave(5)
    cols = torch.randint(0, n, (len(rows),), generator=_rand(seed, 9), device=DEV)
    keep = rows != cols
    lo, hi = torch.minimum(rows, cols)[keep], torch.maximum(rows, cols)[keep]
    up = torch.unique(lo * n + hi)
    v = -torch.randint(1, 1025, (len(up),), generator=_rand(seed, 10), device=DEV).double() / 1024.0
    diag = torch.arange(n, device=DEV) * (n + 1)
    keys = torch.cat([up, (up % n) * n + up // n, diag])
    vals = torch.cat([v, v, torch.zeros(n, dtype=torch.float64, device=DEV)])
    order = torch.argsort(keys)
    return _coo_csr(n, keys[order], vals[order])


def _size(case):
    """Rows or grid side of the case's matrix (drawn cases may give the row count instead)."""
    if case["size"]:
        return case["size"]
    return max(12, int(round(math.sqrt(case["rows"])))) if case["matrix"] == "convdiff2d" else case["rows"]


def _csr(case, seed):
    size = _size(case)
    if case["matrix"] == "poisson2d":
        return gen.laplacian_setup(size, size)
    return {"diffusion3d": _diffusion3d, "convdiff2d": _convdiff2d, "random": _random,
            "random_spd": _random_spd}[case["matrix"]](size, seed)


def _rows(case):
    size = _size(case)
    return {"poisson2d": size ** 2, "diffusion3d": size ** 3, "convdiff2d": size ** 2}.get(case["matrix"], size)


def _nnz(case):
    size, n = _size(case), _rows(case)
    return {"poisson2d": 5 * n - 4 * size, "convdiff2d": 5 * n - 4 * size, "diffusion3d": 7 * n - 6 * size * size,
            "random": 17 * n, "random_spd": 11 * n}[case["matrix"]]


def _systems(case, seed):
    """Uneven SPD systems: rows log-uniform in [256, case rows] (the case alone sets the sizes), 2-D 5-point,
    3-D 7-point and random ones."""
    rng = np.random.default_rng(case["systems"] * 100003 + case["rows"])
    out = []
    for k in range(case["systems"]):
        n = int(round(math.exp(rng.uniform(math.log(256), math.log(case["rows"])))))
        fam = k % 3
        if fam == 0:
            a = max(2, int(round(math.sqrt(n))))
            out.append(gen.laplacian_setup(a, max(2, n // a)))
        elif fam == 1:
            a = max(2, int(round(n ** (1.0 / 3.0))))
            out.append(gen.laplacian3d(a, a, max(2, n // (a * a))))
        else:
            out.append(gen.random_spd(n, seed=seed * 1000 + k))
    return out


# ------------------------------------------------------------------ a pass
class _Vec:
    """A zeroed start vector per pass."""

    def __init__(self, n):
        self.v = m.dense_vector(n)

    def fresh(self):
        self.v.t.zero_()
        return self.v


def _trace(case, seed):
    rng = np.random.default_rng(case["requests"])   # which matrices and how many right-hand sides: the case alone
    n = case["requests"]
    codes = [m.Server.solver(meth, pc) for meth in (m.CG, m.BICGSTAB) for pc in (_lib.PC_DIAGONAL, _lib.PC_ILU0)]
    return {"mat": rng.integers(0, case["systems"], n).astype(np.int32),
            "nrhs": rng.integers(1, 3, n).astype(np.int32),
            "solver": np.array([codes[k % 4] for k in range(n)], np.int32),
            "seed": np.random.default_rng(seed + 17).integers(1, 2 ** 62, n).astype(np.uint64)}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batched":
        B = m.Batch(_systems(case, seed))
        xt = m.dense_vector(_uniform(B.nrows, seed, 11))
        A = m.compressed2D(B.nrows, B.nrows, B.rowptr, B.col, B.val)
        return {"case": case, "B": B, "b": A * xt, "x": _Vec(B.nrows)}
    if kind == "serve":
        B = m.Batch(_systems(case, seed))
        return {"case": case, "B": B, "S": m.Server(B, rtol=1e-12, cap_bytes=8e9), "trace": _trace(case, seed)}
    rp, ci, va = _csr(case, seed)
    n = len(rp) - 1
    A = m.compressed2D(n, n, rp, ci, va)
    if case["layout"] == "sym":
        A.set_kernel(_lib.SPMV_DIA_SYM, 8, 4)
    xt = m.dense_vector(_uniform(n, seed, 11))
    st = {"case": case, "A": A, "x": _Vec(n)}
    if kind == "spmv":
        st["v"], st["w"] = xt, m.dense_vector(n)
        return st
    st["b"] = A * xt
    if kind == "cg":
        st["P"] = m.pc.diagonal(A)
        if case["call"] == "handle":
            st["S"] = m.Solver(A, st["P"], m.CG)
    elif kind == "mixed":
        st["P"] = m.pc.diagonal(A, m.F32)
        A.prepare(m.F32)
    elif kind == "cg_ic0":
        st["P"] = m.pc.ic_0(A)
    elif kind in ("bicgstab_ilu0", "pc_solves"):
        st["P"] = m.pc.ilu_0(A)
        if kind == "pc_solves":
            st["P"].adjoint_solve(st["b"])   # the adjoint's sweeps are laid out once
            st["y"], st["z"] = m.dense_vector(n), m.dense_vector(n)
    elif kind == "bicgstab":
        st["P"] = m.pc.diagonal(A)
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "batched":
        x = st["x"].fresh()
        st["B"].solve(x, st["b"], precision=m.F64 if case["format"] == "f64" else m.F32, rtol=1e-12)
        return x.t
    if kind == "serve":
        t = st["trace"]
        _, _, xs, _ = st["S"].run(t["mat"], t["nrhs"], np.zeros(len(t["mat"])), t["seed"], want_x=True,
                                  solver=t["solver"])
        return xs
    if kind == "spmv":
        return st["A"].mult(st["v"], st["w"]).t
    if kind == "pc_solves":
        st["P"].solve(st["b"], st["y"])
        st["P"].adjoint_solve(st["b"], st["z"])
        return [st["y"].t, st["z"].t]
    A, b, x = st["A"], st["b"], st["x"].fresh()
    if kind in ("bicgstab", "bicgstab_ilu0"):
        m.bicgstab(A, x, b, st["P"], m.basic_iteration(b, 5000, 1e-12))
    elif kind == "mixed":
        m.ir_solve(A, x, b, m.basic_iteration(b, 20000, 1e-10), st["P"], value_format=m.F32)
    elif "S" in st:
        st["S"].solve(x, b, m.basic_iteration(b, 20000, 1e-10))
    else:
        m.cg(A, x, b, st["P"], m.basic_iteration(b, 20000, 1e-10))
    return x.t


# ------------------------------------------------------------------ what a pass cannot do without
def _iterations(case):
    """Iterations of the solves, fitted to counts of these matrices (CG + diagonal takes 984 at 160^3)."""
    size, kind = case["size"] or 1, case["kind"]
    if kind in ("cg", "mixed"):
        return {"poisson2d": 3.1 * size + 5, "diffusion3d": 6.15 * size, "random_spd": 22}[case["matrix"]]
    if kind == "cg_ic0":
        return 2.15 * size if case["matrix"] == "diffusion3d" else 0.9 * size
    if kind == "bicgstab_ilu0":
        return 30
    return 12 if case["matrix"] == "random" else 95


def work(case):
    """Matrix, right-hand side (and inverse diagonal or factor) read once, x written once; the operations of all
    iterations."""
    kind = case["kind"]
    if kind in ("batched", "serve"):
        # mean rows of a log-uniform size, 9 entries per row, about 90 iterations, FP64 vectors
        rows = (case["rows"] - 256) / math.log(case["rows"] / 256.0)
        solves = case["systems"] if kind == "batched" else 1.5 * case["requests"]
        return {"bytes": case["systems"] * rows * 9 * 12 + solves * rows * 8 * 3,
                "flops": solves * rows * 90 * (2 * 9 + 12)}
    n, nnz = _rows(case), _nnz(case)
    grid = case["matrix"] in ("poisson2d", "diffusion3d", "convdiff2d")
    entries = (nnz + n) // 2 if case["matrix"] in ("poisson2d", "diffusion3d") else nnz   # symmetric: half
    mat = entries * (8 if grid else 12)                    # a grid's columns follow from its shape
    if kind == "spmv":
        return {"bytes": mat + 16 * n, "flops": 2 * nnz}
    if kind == "pc_solves":
        return {"bytes": 2 * (nnz * (8 if grid else 12) + 16 * n), "flops": 4 * nnz}
    it = _iterations(case)
    per = {"cg": 2 * nnz + 12 * n, "mixed": 2 * nnz + 12 * n, "cg_ic0": 4 * nnz + 14 * n,
           "bicgstab": 4 * nnz + 22 * n, "bicgstab_ilu0": 8 * nnz + 24 * n}[kind]
    factor = mat if kind in ("cg_ic0", "bicgstab_ilu0") else 8 * n
    return {"bytes": mat + factor + 16 * n, "flops": it * per}


# ------------------------------------------------------------------ 64-bit values by plain means
def _splitmix(seed, n):
    """The serving loop's right-hand side: splitmix64 of (seed, i) mapped to [-1, 1)."""
    i = np.arange(1, n + 1, dtype=np.uint64)
    with np.errstate(over="ignore"):
        z = np.uint64(seed) + i * np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    return (z >> np.uint64(11)).astype(np.float64) * (2.0 / 9007199254740992.0) - 1.0


def _dense(csr):
    rp, ci, va = csr
    n = len(rp) - 1
    a = torch.zeros((n, n), dtype=torch.float64, device=DEV)
    rows = np.repeat(np.arange(n), np.diff(rp))
    a[torch.as_tensor(rows, device=DEV), torch.as_tensor(ci.astype(np.int64), device=DEV)] = \
        torch.as_tensor(va, device=DEV)
    return a


def _product(rp, ci, va, v):
    """A*v row by row in column order, 64 bits, on the host."""
    prod = va * v[ci]
    out = np.zeros(len(rp) - 1)
    lens = np.diff(rp)
    for k in range(int(lens.max())):
        has = np.nonzero(lens > k)[0]
        out[has] += prod[rp[has].astype(np.int64) + k]
    return out


def _ilu0_solves(rp, ci, va, b):
    """solve and adjoint_solve of ILU(0), row by row on the host."""
    n = len(rp) - 1
    rp, ci, f = rp.tolist(), ci.tolist(), va.tolist()
    dpos = [0] * n
    pos = {}
    for r in range(n):
        for j in range(rp[r], rp[r + 1]):
            pos[(r, ci[j])] = j
            if ci[j] == r:
                dpos[r] = j
    for r in range(1, n):
        for j in range(rp[r], dpos[r]):
            k = ci[j]
            f[j] /= f[dpos[k]]
            w = f[j]
            for q in range(dpos[k] + 1, rp[k + 1]):
                p = pos.get((r, ci[q]))
                if p is not None:
                    f[p] -= w * f[q]
    y = b.tolist()
    for r in range(n):
        for j in range(rp[r], dpos[r]):
            y[r] -= f[j] * y[ci[j]]
    for r in range(n - 1, -1, -1):
        for j in range(dpos[r] + 1, rp[r + 1]):
            y[r] -= f[j] * y[ci[j]]
        y[r] /= f[dpos[r]]
    z = b.tolist()
    for r in range(n):          # U^T z = b, then L^T z = z
        z[r] /= f[dpos[r]]
        for j in range(dpos[r] + 1, rp[r + 1]):
            z[ci[j]] -= f[j] * z[r]
    for r in range(n - 1, -1, -1):
        for j in range(rp[r], dpos[r]):
            z[ci[j]] -= f[j] * z[r]
    return [np.array(y), np.array(z)]


def exact(case, seed):
    kind = case["kind"]
    if kind == "serve":
        t = _trace(case, seed)
        systems = _systems(case, seed)
        out = [None] * len(t["mat"])
        for k in range(len(systems)):
            reqs = np.nonzero(t["mat"] == k)[0]
            if not len(reqs):
                continue
            n = len(systems[k][0]) - 1
            # right-hand side q of a request is the sequence of 131 * seed + q
            rhs = [_splitmix((int(t["seed"][r]) * 131 + q) & (2 ** 64 - 1), n)
                   for r in reqs for q in range(t["nrhs"][r])]
            sol = torch.linalg.solve(_dense(systems[k]), torch.as_tensor(np.array(rhs).T.copy(), device=DEV))
            sol = sol.T.contiguous().cpu().numpy()
            at = 0
            for r in reqs:
                out[r] = sol[at:at + t["nrhs"][r]]
                at += t["nrhs"][r]
        return out
    if kind == "batched":
        rows = sum(len(s[0]) - 1 for s in _systems(case, seed))
        return _uniform(rows, seed, 11)
    xt = _uniform(_rows(case), seed, 11)
    if kind == "spmv":
        return _product(*_csr(case, seed), xt.cpu().numpy())
    if kind == "pc_solves":
        csr = _csr(case, seed)
        return _ilu0_solves(*csr, _product(*csr, xt.cpu().numpy()))
    return xt
