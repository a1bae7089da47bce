"""itl::cg with its state on the chip (resident.hip): one launch for many
iterations on systems whose rows fit the registers of the GPU's compute units.
Compared with the launch-per-kernel loop (which runs MTL4's summation order)
after a few iterations, where only the order of the sums differs, and with the
oracle at convergence."""
import ctypes as C
import io
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def m():
    import mtl4_amd
    return mtl4_amd


def _tridiag(n):
    rp = np.concatenate([[0], np.cumsum([1 if n == 1 else 2 if i in (0, n - 1) else 3 for i in range(n)])])
    ci, va = [], []
    for i in range(n):
        for j in (i - 1, i, i + 1):
            if 0 <= j < n:
                ci.append(j)
                va.append(2.5 + 0.001 * (i % 7) if i == j else -1.0)
    return rp.astype(np.int32), np.array(ci, np.int32), np.array(va)


def _matrix(kind, size):
    from mtl4_amd import generators as gen
    if kind == "tridiag":
        return _tridiag(size)
    if kind == "permuted":      # three entries per row, columns anywhere
        import scipy.sparse as sp
        i = np.arange(size)
        A = sp.diags([np.full(size - 1, -1.0), 2.5 + 0.001 * (i % 7), np.full(size - 1, -1.0)], [-1, 0, 1], format="csr")
        q = np.random.default_rng(2).permutation(size)
        A = A[q][:, q].tocsr()
        A.sort_indices()
        return A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data
    if kind == "grid2d":
        return gen.laplacian_setup(*size)
    if kind == "grid3d":
        return gen.laplacian3d(*size)
    if kind == "diffusion":
        return gen.diffusion3d(size, seed=3)
    return gen.random_spd(size, seed=4, nnz_per_row=size % 13 + 6)


# edges: one workgroup (4096 rows) and the next size, waves and workgroups that
# end inside a row block, neighbours at the LDS halo (1024) and just beyond it
# in one workgroup and in several, 2/4/8 rows per lane, the register limits of
# the unstructured operand (8, 16, 24 entries per lane), the largest grid
# The operand that each must run on: 0 the launch-per-kernel loop, 1 / 2 up to 5 / 7
# diagonals, 3, 4, 5 up to 8, 16, 24 entries per lane of any pattern (1 to 8 rows per lane)
CASES = [("tridiag", 1, 3), ("tridiag", 2, 3), ("tridiag", 65, 1), ("tridiag", 513, 1), ("tridiag", 4096, 1),
         ("tridiag", 4097, 1), ("grid2d", (4, 1024), 1), ("grid2d", (3, 1025), 1), ("grid2d", (4, 1023), 1),
         ("grid2d", (9, 1024), 1), ("grid2d", (9, 1025), 1), ("grid2d", (64, 64), 1), ("grid2d", (517, 523), 1),
         ("grid3d", (7, 5, 3), 2), ("grid3d", (33, 32, 31), 2), ("grid3d", (101, 103, 97), 2), ("diffusion", 17, 2),
         ("diffusion", 65, 2), ("random", 37, 3), ("random", 700, 5), ("random", 70003, 5), ("random", 140010, 4),
         ("random", 262150, 0), ("permuted", 300007, 4), ("permuted", 600011, 5)]


def _operand(m):
    """What this thread's last CG solve ran on; no launch was refused."""
    i = m._lib.CgChipInfo()
    m._lib.check(m._lib.lib().mtl4g_cg_chip(C.byref(i)))
    assert i.refused == 0 and (i.launches > 0) == (i.operand > 0)
    return i.operand


def _few(m, A, P, b, steps, general):
    """x and the iteration state after `steps` iterations."""
    x = m.dense_vector(A.num_rows())
    it = m.basic_iteration(b, steps, 0.0)
    with m.reduction_order(m.ORDER_MTL4 if general else m.ORDER_TREE):
        m.cg(A, x, b, P, it)
    return x.numpy(), it


@pytest.mark.parametrize("pc", ["diagonal", "identity"])
@pytest.mark.parametrize("kind,size,operand", CASES)
def test_resident_cg_matches_launch_per_kernel_loop(m, kind, size, operand, pc):
    rp, ci, va = _matrix(kind, size)
    n = len(rp) - 1
    print("resident cg", kind, size, n, pc, flush=True)
    A = m.compressed2D(n, n, rp, ci, va)
    P = m.pc.diagonal(A) if pc == "diagonal" else None
    b = A * m.dense_vector(np.random.default_rng(5).uniform(-1, 1, n))
    # rounding of the sums only: n terms of either order differ by a few
    # 1e-16 relative, amplified by at most a few per iteration
    steps = min(6, n)
    xa, ia = _few(m, A, P, b, steps, False)
    assert _operand(m) == operand
    xb, ib = _few(m, A, P, b, steps, True)
    assert _operand(m) == 0
    assert ia.iterations() == ib.iterations() and ia.error_code() == ib.error_code()
    assert np.linalg.norm(xa - xb) <= 1e-12 * np.linalg.norm(xb)
    xc, _ = _few(m, A, P, b, steps, False)
    assert np.array_equal(xa, xc)   # deterministic


@pytest.mark.parametrize("offsets", [(-3000, -2000), (2000, 3000), (-3000, -1024), (-1025, 0), (1024, 1025), (0, 2000)])
def test_resident_cg_two_diagonals(m, offsets):
    """Both on one side of the main diagonal, in and beyond the LDS halo (1024)."""
    n = 30011   # both diagonals full enough for the diagonal layout
    rng = np.random.default_rng(9)
    row = np.repeat(np.arange(n), 2)
    col = row + np.tile(offsets, n)
    keep = (col >= 0) & (col < n)
    rp = np.concatenate([[0], np.cumsum(np.bincount(row[keep], minlength=n))]).astype(np.int32)
    A = m.compressed2D(n, n, rp, col[keep].astype(np.int32), rng.uniform(1, 2, int(keep.sum())))
    assert A.get_kernel()[0] == m._lib.SPMV_DIA
    b = m.dense_vector(rng.uniform(1, 2, n))
    # not a system CG solves: two iterations.  All terms of the first p.q are
    # positive; 1e-12 leaves room for a cancellation of 1e-3 in the second
    xa, ia = _few(m, A, None, b, 2, False)
    one_side = offsets in ((-3000, -2000), (2000, 3000))
    assert _operand(m) == (3 if one_side else 1)
    xb, ib = _few(m, A, None, b, 2, True)
    assert ia.iterations() == ib.iterations() == 2
    assert np.linalg.norm(xa - xb) <= 1e-12 * np.linalg.norm(xb)


@pytest.mark.parametrize("layout", ["dia", "sym"])
@pytest.mark.parametrize("kind,size", [("grid2d", (61, 64)), ("grid2d", (7, 1500)), ("diffusion", 33)])
def test_resident_cg_layouts_and_oracle(m, kind, size, layout):
    import orc
    rp, ci, va = _matrix(kind, size)
    n = len(rp) - 1
    A = m.compressed2D(n, n, rp, ci, va)
    if layout == "sym":
        A.set_kernel(m._lib.SPMV_DIA_SYM, 4, 4)
    O = orc.Matrix(rp, ci, va)
    xt = np.random.default_rng(6).uniform(-1, 1, n)
    b = orc.spmv(O, xt)
    xo, st, ito, _ = orc.cg(O, b, orc.Preconditioner("diagonal", O), max_iter=5000, rtol=1e-10)
    x, bd = m.dense_vector(n), m.dense_vector(b)
    it = m.basic_iteration(bd, 5000, 1e-10)
    assert m.cg(A, x, bd, m.pc.diagonal(A), it) == 0 and st == 0
    assert _operand(m) == (2 if kind == "diffusion" else 1)
    assert abs(it.iterations() - ito.i) <= 2
    assert np.linalg.norm(x.numpy() - xo) <= 1e-9 * np.linalg.norm(xo)


def test_resident_cg_history_start_vector_and_limits(m):
    rp, ci, va = _matrix("grid2d", (64, 64))
    n = len(rp) - 1
    A = m.compressed2D(n, n, rp, ci, va)
    P = m.pc.diagonal(A)
    rng = np.random.default_rng(7)
    x0 = rng.uniform(-1, 1, n)
    b = m.dense_vector(rng.uniform(-1, 1, n))
    out = io.StringIO()
    it = m.cyclic_iteration(b, 400, 1e-10, 0.0, 1, out)
    x = m.dense_vector(x0)
    assert m.cg(A, x, b, P, it) == 0
    # one residual per finished() call, the last one reported and converged
    assert len(it.history) == it.iterations() + 1 and it.history[-1] == it.resid()
    assert it.resid() <= 1e-10 * it.norm_r0()
    it2 = m.basic_iteration(b, it.iterations() - 1, 1e-10)
    x2 = m.dense_vector(x0)
    assert m.cg(A, x2, b, P, it2) == 1 and it2.iterations() == it.iterations() - 1
    # more iterations than one launch runs: the state goes on in the next one
    big = m.compressed2D(*([len(_matrix("diffusion", 33)[0]) - 1] * 2), *_matrix("diffusion", 33))
    bb = m.dense_vector(rng.uniform(-1, 1, 33 ** 3))
    itb = m.basic_iteration(bb, 700, 0.0)
    xb = m.dense_vector(33 ** 3)
    m.cg(big, xb, bb, m.pc.diagonal(big), itb)
    assert itb.iterations() == 700 and np.isfinite(xb.numpy()).all()


def test_resident_cg_nonfinite(m):
    rp, ci, va = _matrix("grid2d", (40, 40))
    n = len(rp) - 1
    A = m.compressed2D(n, n, rp, ci, va)
    b = np.ones(n)
    b[17] = np.inf
    bd, x = m.dense_vector(b), m.dense_vector(n)
    with pytest.raises(m.nonfinite_error):
        m.cg(A, x, bd, m.pc.diagonal(A), m.basic_iteration(1.0, 50, 1e-10))


def _indefinite(kind):
    """p.q = 0 for p = (1, 1, ..), q nowhere 0, on a size that leaves places without rows."""
    import scipy.sparse as sp
    if kind == "csr":       # one diagonal: the operand for any pattern
        n = 1002
        A = sp.diags(np.tile([1.0, -1.0], n // 2), format="csr")
    elif kind.startswith("dia"):     # antisymmetric, two diagonals; one: a single workgroup
        n = 902 if kind == "dia_one" else 9002
        up = np.arange(1.0, n)
        A = sp.diags([-up, up], [-1, 1], format="csr")
    else:                   # five diagonals, more rows than the registers hold
        n = 1050002
        A = sp.diags([np.ones(n - abs(o)) for o in (-7, -1, 0, 1, 7)], [-7, -1, 0, 1, 7], format="csr")
        row = np.repeat(np.arange(n), np.diff(A.indptr))
        A.data = np.where(A.indices == row, 1.0 - 2.0 * (row % 2), 0.0)   # stored zeros beside the main diagonal
    A.sort_indices()
    return n, A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data


@pytest.mark.parametrize("kind", ["csr", "dia", "dia_one", "large"])
def test_resident_cg_infinite_step(m, kind):
    """alpha = rho / 0: the residual reported is the infinite one of the rows."""
    n, rp, ci, va = _indefinite(kind)
    A = m.compressed2D(n, n, rp, ci, va)
    b = m.dense_vector(np.ones(n))
    got = []
    for order in (m.ORDER_TREE, m.ORDER_MTL4):
        it = m.cyclic_iteration(b, 50, 1e-10, 0.0, 1, io.StringIO())
        with m.reduction_order(order), pytest.raises(m.nonfinite_error):
            m.cg(A, m.dense_vector(n), b, None, it)
        if order == m.ORDER_TREE:
            assert _operand(m) == {"csr": 3, "dia": 1, "dia_one": 1, "large": 6}[kind]
        got.append((it.iterations(), it.resid(), list(it.history)))
    assert got[0] == got[1] == (1, np.inf, [np.sqrt(n), np.inf])


def test_resident_cg_concurrent_threads(m):
    """Solves of several threads on streams of their own: each gets the bits of
    the same solve alone."""
    import torch
    jobs = []
    for k, size in enumerate([(300, 301), (64, 64), (200, 333), (517, 523)]):
        rp, ci, va = _matrix("grid2d", size)
        n = len(rp) - 1
        A = m.compressed2D(n, n, rp, ci, va)
        b = m.dense_vector(np.random.default_rng(k).uniform(-1, 1, n))
        P = m.pc.diagonal(A)
        x = m.dense_vector(n)
        m.cg(A, x, b, P, m.basic_iteration(b, 300, 1e-12))
        jobs.append((A, b, P, n, x.numpy()))
    torch.cuda.synchronize()
    bad = []

    def work(job):
        A, b, P, n, want = job
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(3):
                x = m.dense_vector(n)
                m.cg(A, x, b, P, m.basic_iteration(b, 300, 1e-12))
                if not np.array_equal(x.numpy(), want):
                    bad.append(n)

    ts = [threading.Thread(target=work, args=(j,)) for j in jobs]
    for t in ts:
        t.start()
    for t in ts:
        t.join(60)
    assert not bad and not any(t.is_alive() for t in ts)


# BF16 matrix values converge on the well-conditioned systems only
@pytest.mark.parametrize("kind,size,fmt,operand", [("random", 2000, "F32", 5), ("random", 2000, "BF16", 5),
                                                   ("grid2d", (40, 41), "F32", 1), ("diffusion", 20, "F32", 2),
                                                   ("random", 90000, "F32", 3), ("random", 90000, "BF16", 3)])
def test_resident_mixed_cg(m, kind, size, fmt, operand):
    rp, ci, va = _matrix(kind, size)
    n = len(rp) - 1
    A = m.compressed2D(n, n, rp, ci, va)
    xt = np.random.default_rng(8).uniform(-1, 1, n)
    b = A * m.dense_vector(xt)
    x = m.dense_vector(n)
    err, st = m.ir_solve(A, x, b, m.basic_iteration(b, 20000, 1e-10), m.pc.diagonal(A, m.F32),
                         value_format=getattr(m, fmt))
    assert err == 0 and st["relres"] <= 1e-10 and _operand(m) == operand
    r = b.numpy() - (A * x).numpy()
    assert np.linalg.norm(r) <= 1.01e-10 * np.linalg.norm(b.numpy())
