"""itl::cg on diagonal layouts too large to be held on the chip
(resident_large.hip): against the launch-per-kernel loop, which MTL4's
summation order selects, after a few iterations."""
import numpy as np
import pytest

from test_gpu_resident import _operand

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def m():
    import mtl4_amd
    return mtl4_amd


def _grid(sizes):
    """Diagonally dominant 5- or 7-point operator with varying symmetric values, columns ascending."""
    import scipy.sparse as sp
    n = int(np.prod(sizes))
    i = np.arange(n)
    D, off, diag = [], [], np.full(n, 0.25)
    step = 1
    for s in sizes:
        inside = (i // step) % s + 1 < s                # couples i and i + step
        w = np.where(inside, -1.0 - 0.125 * (i % 5), 0.0)
        diag -= w
        diag[step:] -= w[:-step]
        up = w[:-step]
        D += [up, up]
        off += [step, -step]
        step *= s
    A = sp.diags(D + [diag], off + [0], format="csr")
    A.eliminate_zeros()
    A.sort_indices()
    return A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data


# just above the size held on the chip; outer diagonals inside and beyond the LDS
# halo (1024); odd inner diagonals (rows of a pair in two slices); each count of
# groups per lane up to the largest, grids that end inside a workgroup; an outer
# diagonal of odd offset and an odd row count, which the launch-per-kernel loop takes
SHAPES = [(1024, 1026), (1020, 1040), (1500, 1000), (1001, 1600), (102, 103, 102), (31, 30, 1600), (33, 34, 1200),
          (126, 127, 126), (140, 140, 140), (150, 150, 150), (160, 160, 160), (1025, 1030), (101, 103, 105)]


def _few(m, A, P, b, steps, general):
    x = m.dense_vector(A.num_rows())
    it = m.basic_iteration(b, steps, 0.0)
    with m.reduction_order(m.ORDER_MTL4 if general else m.ORDER_TREE):
        m.cg(A, x, b, P, it)
    return x.numpy(), it


@pytest.mark.parametrize("layout", ["dia", "sym"])
@pytest.mark.parametrize("sizes", SHAPES)
def test_large_cg_matches_launch_per_kernel_loop(m, sizes, layout):
    rp, ci, va = _grid(sizes)
    n = len(rp) - 1
    A = m.compressed2D(n, n, rp, ci, va)
    if layout == "sym":
        A.set_kernel(m._lib.SPMV_DIA_SYM, 4, 4)
    else:
        A.set_kernel(m._lib.SPMV_DIA, 4, 4)
    b = A * m.dense_vector(np.random.default_rng(5).uniform(-1, 1, n))
    for pc in ("diagonal", "identity"):
        print("large cg", sizes, n, layout, pc, flush=True)
        P = m.pc.diagonal(A) if pc == "diagonal" else None
        # the order of the sums differs: a few 1e-16 relative per sum of n terms,
        # amplified by at most a few per iteration
        xa, ia = _few(m, A, P, b, 5, False)
        assert _operand(m) == (0 if sizes in ((1025, 1030), (101, 103, 105)) else 6)
        xb, ib = _few(m, A, P, b, 5, True)
        assert ia.iterations() == ib.iterations() and ia.error_code() == ib.error_code()
        assert np.linalg.norm(xa - xb) <= 1e-12 * np.linalg.norm(xb)
        xc, _ = _few(m, A, P, b, 5, False)
        assert np.array_equal(xa, xc)   # deterministic


@pytest.mark.parametrize("fmt", ["F32", "BF16"])
@pytest.mark.parametrize("layout", ["dia", "sym"])
@pytest.mark.parametrize("sizes", [(1480, 1424), (130, 130, 130), (164, 160, 160)])
def test_large_mixed_cg(m, sizes, layout, fmt):
    """FP32 recurrence on FP32 or BF16 values to the FP64 tolerance; the values
    of _grid are exact in both."""
    rp, ci, va = _grid(sizes)
    n = len(rp) - 1
    A = m.compressed2D(n, n, rp, ci, va)
    A.set_kernel(m._lib.SPMV_DIA_SYM if layout == "sym" else m._lib.SPMV_DIA, 4, 4)
    b = A * m.dense_vector(np.random.default_rng(8).uniform(-1, 1, n))
    for pc in (None, m.pc.diagonal(A, m.F32)):
        print("large mixed cg", sizes, n, layout, fmt, pc is not None, flush=True)
        x = m.dense_vector(n)
        err, st = m.ir_solve(A, x, b, m.basic_iteration(b, 20000, 1e-10), pc, value_format=getattr(m, fmt))
        assert err == 0 and st["relres"] <= 1e-10 and _operand(m) == 6
        r = b.numpy() - (A * x).numpy()
        assert np.linalg.norm(r) <= 1.01e-10 * np.linalg.norm(b.numpy())


@pytest.mark.parametrize("sizes", [(102, 104, 102), (160, 160, 160)])
def test_large_cg_vectors_off_a_16_byte_boundary(m, sizes):
    """x and b that start 8 bytes past one: the same bits."""
    import torch
    rp, ci, va = _grid(sizes)
    n = len(rp) - 1
    A = m.compressed2D(n, n, rp, ci, va)
    A.set_kernel(m._lib.SPMV_DIA_SYM, 4, 4)
    P = m.pc.diagonal(A)
    b = A * m.dense_vector(np.random.default_rng(5).uniform(-1, 1, n))
    xs = []
    for shift in (0, 1):
        print("large cg shifted", sizes, shift, flush=True)
        buf = torch.zeros(n + 2, dtype=torch.float64, device="cuda")
        bb = torch.zeros(n + 2, dtype=torch.float64, device="cuda")
        bb[shift:shift + n] = b.t
        x, bd = m.dense_vector(buf[shift:shift + n]), m.dense_vector(bb[shift:shift + n])
        assert x.t.data_ptr() % 16 == 8 * shift
        m.cg(A, x, bd, P, m.basic_iteration(bd, 6, 0.0))
        assert _operand(m) == 6
        xs.append(x.numpy().copy())
        assert float(buf[:shift].abs().sum() + buf[shift + n:].abs().sum()) == 0.0
    assert np.array_equal(xs[0], xs[1])


@pytest.mark.parametrize("sizes,mixed", [((1500, 1000), False), ((1001, 1600), False), ((102, 103, 102), False),
                                         ((1480, 1424), True), ((130, 130, 130), True)])
def test_large_cg_halo_is_whole_groups(m, sizes, mixed):
    """The workgroup's rows lie behind the halo in LDS and are read 16 bytes at a
    time: 2 FP64 or 4 FP32 values."""
    import ctypes as C
    rp, ci, va = _grid(sizes)
    n = len(rp) - 1
    A = m.compressed2D(n, n, rp, ci, va)
    A.set_kernel(m._lib.SPMV_DIA, 4, 4)
    b = A * m.dense_vector(np.random.default_rng(5).uniform(-1, 1, n))
    x = m.dense_vector(n)
    if mixed:
        m.ir_solve(A, x, b, m.basic_iteration(b, 20000, 1e-10), m.pc.diagonal(A, m.F32))
    else:
        m.cg(A, x, b, None, m.basic_iteration(b, 3, 0.0))
    info = m._lib.CgChipInfo()
    m._lib.check(m._lib.lib().mtl4g_cg_chip(C.byref(info)))
    near = max(o for o in (1, sizes[0], n // sizes[-1]) if o <= 1024)
    assert info.operand == 6 and near <= info.halo < near + 4 and info.halo % (4 if mixed else 2) == 0
