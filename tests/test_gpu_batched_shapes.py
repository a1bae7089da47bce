"""Batched CG at the edges of its row loops and triangular sweeps: row counts
around the rows a thread works on at once, rows longer than one pass of eight
entries, factor rows longer than the entries requested ahead, levels wider
than the workgroup, and systems on both sides of the sweep kept in LDS."""
import numpy as np
import pytest
import scipy.sparse as sp

import orc
from test_gpu_serving import splitmix_uniform

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def m():
    import mtl4_amd
    return mtl4_amd


def _csr(M):
    M = sp.csr_matrix(M)
    M.sort_indices()
    return M.indptr, M.indices, M.data


def _systems(threads):
    """Diagonally dominant (condition number below 10)."""
    def tri(n):
        return sp.diags([np.full(n - 1, -1.0), np.full(n, 3.0), np.full(n - 1, -1.0)], [-1, 0, 1])

    def banded(n, w):   # 2w + 1 entries per row
        D = [np.full(n - k, -1.0 / w) for k in range(1, w + 1)]
        return sp.diags(D[::-1] + [np.full(n, 3.0)] + D, list(range(-w, 0)) + list(range(0, w + 1)))

    def arrow(n):       # one row and column full: a row of n entries beside rows of two
        A = sp.diags([np.full(n, 3.0)], [0]).tolil()
        A[0, 1:] = -1.0 / n
        A[1:, 0] = -1.0 / n
        return A

    M = [tri(n) for n in (2, threads - 1, threads + 1, 4 * threads - 1, 4 * threads, 4 * threads + 1)]
    M += [sp.diags([np.arange(1.0, 2.0, 1.0 / 1500)], [0]), arrow(1300), banded(700, 4), banded(333, 9),
          tri(4095), tri(4096), tri(4097), sp.identity(1)]
    return [_csr(A) for A in M]


# eight iterations on condition numbers below 10: the solutions of two summation
# orders differ by less than 8 * 10 * sqrt(n) * eps * 10 = 1.2e-11
TOL = 2e-11


@pytest.mark.parametrize("pc", ["identity", "diagonal"])
@pytest.mark.parametrize("threads", [256, 512, 1024])
def test_batch_shapes_match_oracle(m, threads, pc):
    S = _systems(threads)
    rng = np.random.default_rng(threads)
    bs = [rng.uniform(-1, 1, len(s[0]) - 1) for s in S]
    B = m.Batch(S)
    B.set_shape(m.F64, threads, 1)
    x = m.dense_vector(B.nrows)
    kind = m._lib.PC_IDENTITY if pc == "identity" else m._lib.PC_DIAGONAL
    res = B.solve(x, m.dense_vector(np.concatenate(bs)), pc_kind=kind, precision=m.F64, rtol=1e-13, max_iter=8)
    xs = x.numpy()
    for k, (s, b) in enumerate(zip(S, bs)):
        O = orc.Matrix(*s)
        P = orc.Preconditioner(pc, O) if pc != "identity" else None
        xo = orc.cg(O, b, P, max_iter=8, rtol=1e-13)[0]
        got = xs[B.sys_row[k]:B.sys_row[k + 1]]
        assert res[k]["status"] == 0, (k, res[k])
        assert np.linalg.norm(got - xo) <= TOL * np.linalg.norm(xo), (k, res[k], np.linalg.norm(got - xo))


@pytest.mark.parametrize("method", ["cg", "bicgstab"])
@pytest.mark.parametrize("threads", [256, 512, 1024])
def test_batch_ilu0_shapes_match_oracle(m, threads, method):
    """Factors are built by the server.  Both solutions have a relative residual
    of 1e-12 at most: they differ by less than 2 * 10 * 1e-12 = TOL."""
    S = _systems(threads)
    B = m.Batch(S)
    B.set_shape(m.F64, threads, 1)
    srv = m.Server(B, precision=m.F64, rtol=1e-12, big_rows=10 ** 9, streams=2, max_items=64, cap_bytes=1e9)
    code = m.Server.solver(m.CG if method == "cg" else m.BICGSTAB, m._lib.PC_ILU0)
    n = len(S)
    seeds = np.arange(1, n + 1, dtype=np.uint64)
    _, _, xs, st = srv.run(np.arange(n), np.ones(n, np.int32), np.zeros(n), seeds, want_x=True,
                           solver=np.full(n, code, np.int32))
    assert st["errors"] == 0
    for k, s in enumerate(S):
        O = orc.Matrix(*s)
        b = splitmix_uniform(int(seeds[k]) * 131, len(s[0]) - 1)
        fn = orc.cg if method == "cg" else orc.bicgstab
        xo = fn(O, b, orc.Preconditioner("ilu_0", O), max_iter=1000, rtol=1e-12)[0]
        assert np.linalg.norm(xs[k][0] - xo) <= TOL * np.linalg.norm(xo), (k, np.linalg.norm(xs[k][0] - xo))
