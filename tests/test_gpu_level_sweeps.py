"""Level-scheduled triangular sweeps: factors of each mean row length that
selects how many entries of a row are requested ahead (4, 8 or 16), with rows
just below, at and above those counts and levels around a workgroup's 128
rows; solve and adjoint_solve are the oracle's bit for bit."""
import numpy as np
import pytest
import scipy.sparse as sp

import orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def m():
    import mtl4_amd
    return mtl4_amd


def _matrix(n, mean, seed):
    """n rows, about `mean` entries on each side of the diagonal; a few long rows."""
    rng = np.random.default_rng(seed)
    r = rng.integers(0, n, int(n * mean))
    c = rng.integers(0, n, int(n * mean))
    A = sp.coo_matrix((rng.uniform(-1, -0.1, len(r)), (r, c)), shape=(n, n)).tocsr()
    A = sp.tril(A, -1)
    long = [sp.coo_matrix((rng.uniform(-1, -0.1, k), (np.full(k, n - 1 - i), rng.choice(n - 10, k, replace=False))),
                          shape=(n, n)) for i, k in enumerate((3, 4, 5, 8, 9, 16, 17, 33))] if n > 60 else []
    A = sp.tril(sum(long, A), -1)
    A = (A + A.T).tocsr()
    A = (A + sp.diags(2.0 - np.asarray(A.sum(axis=1)).ravel())).tocsr()
    A.sort_indices()
    return A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data


@pytest.mark.parametrize("vb", [8, 4])
@pytest.mark.parametrize("n,mean", [(1, 0), (128, 1), (129, 4), (700, 2), (700, 7), (3000, 2), (3000, 7), (3000, 14)])
def test_level_sweeps_bitwise(m, n, mean, vb):
    csr = _matrix(n, mean, n + mean)
    nl = (len(csr[1]) - n) // 2
    print("level sweeps", n, mean, "entries per factor row %.2f" % (nl / n), flush=True)
    A = m.compressed2D(n, n, *csr)
    O = orc.Matrix(*csr)
    x = np.random.default_rng(1).uniform(-1, 1, n)
    for kind in ("ilu_0", "ic_0"):
        P = getattr(m.pc, kind)(A, m.F64 if vb == 8 else m.F32)
        OP = orc.Preconditioner(kind, O, vb)
        assert np.array_equal(P.solve(m.dense_vector(x)).numpy(), OP.solve(x))
        assert np.array_equal(P.adjoint_solve(m.dense_vector(x)).numpy(), OP.adjoint_solve(x))
