"""Level-scheduled triangular sweeps: factors that select 4, 8 or 16 entries of a
row requested ahead (by how many levels have a longer row), with rows just below,
at and above those counts and levels around a workgroup's 128 rows; solve and
adjoint_solve are the oracle's bit for bit."""
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
    """n rows, about mean / 2 entries on each side of the diagonal (mean 0: each row
    coupled to the next, one row per level); a few long rows."""
    rng = np.random.default_rng(seed)
    r = rng.integers(0, n, int(n * mean))
    c = rng.integers(0, n, int(n * mean))
    A = sp.coo_matrix((rng.uniform(-1, -0.1, len(r)), (r, c)), shape=(n, n)).tocsr()
    A = sp.tril(A, -1)
    if mean == 0 and n > 1:
        A = sp.diags(rng.uniform(-1, -0.1, n - 1), -1, shape=(n, n), format="csr")
    long = [sp.coo_matrix((rng.uniform(-1, -0.1, k), (np.full(k, n - 1 - i), rng.choice(n - 10, k, replace=False))),
                          shape=(n, n)) for i, k in enumerate((3, 4, 5, 8, 9, 16, 17, 33))] if n > 60 else []
    A = sp.tril(sum(long, A), -1)
    A = (A + A.T).tocsr()
    A = (A + sp.diags(2.0 - np.asarray(A.sum(axis=1)).ravel())).tocsr()
    A.sort_indices()
    return A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data


def _ahead(csr, lower):
    """Entries the sweep of this pattern's factor requests ahead."""
    rp, ci = csr[0], csr[1]
    n = len(rp) - 1
    lev, length = np.zeros(n, int), np.zeros(n, int)
    for r in range(n) if lower else range(n - 1, -1, -1):
        c = ci[rp[r]:rp[r + 1]]
        c = c[c < r] if lower else c[c > r]
        length[r] = len(c)
        lev[r] = lev[c].max() + 1 if len(c) else 0
    longest = np.zeros(lev.max() + 1, int)
    np.maximum.at(longest, lev, length)
    return 16 if 2 * (longest > 8).sum() > len(longest) else 8 if 4 * (longest > 4).sum() > len(longest) else 4


@pytest.mark.parametrize("vb", [8, 4])
@pytest.mark.parametrize("n,mean,ahead", [(1, 0, (4, 4)), (128, 1, (16, 8)), (129, 4, (8, 8)), (700, 2, (8, 8)),
                                          (700, 7, (16, 16)), (1500, 0, (4, 4)), (3000, 2, (8, 8)),
                                          (3000, 7, (16, 16)), (3000, 14, (16, 16))])
def test_level_sweeps_bitwise(m, n, mean, ahead, vb):
    csr = _matrix(n, mean, n + mean)
    assert (_ahead(csr, True), _ahead(csr, False)) == ahead
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
