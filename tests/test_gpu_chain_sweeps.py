"""Triangular sweeps of grid factors (chain.hpp) at the sizes where the
pipeline's blocks, tiles and exchange slots end, against the level schedule:
the same bits for every row, also with holes in the pattern, signed zeros,
infinities and NaN in the input."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def m():
    import mtl4_amd
    return mtl4_amd


def _grid(shape, holes, seed):
    """A diagonally dominant nonsymmetric-valued 5- or 7-point matrix; with
    holes a few off-diagonal pairs are missing."""
    from mtl4_amd import generators as gen
    rp, ci, va = gen.laplacian_setup(*shape) if len(shape) == 2 else gen.laplacian3d(*shape)
    n = len(rp) - 1
    rng = np.random.default_rng(seed)
    rows = np.repeat(np.arange(n), np.diff(rp))
    va = np.where(rows == ci, 8.0 + rng.uniform(0, 1, len(va)), -rng.uniform(0.5, 1.5, len(va)))
    if holes:
        lo, hi = np.minimum(rows, ci), np.maximum(rows, ci)
        keep = (lo == hi) | ((lo * 7919 + hi * 104729) % 29 != 0)
        rows, ci, va = rows[keep], ci[keep], va[keep]
        rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))])
    return rp.astype(np.int32), ci.astype(np.int32), va


# laplacian_setup(m, n): chains of n rows, m of them; laplacian3d(nx, ny, nz):
# chains of nx rows, planes of ny chains.  Chains shorter than a block of 8
# steps, one block, one more; one tile (64 x 1, 8 x 8), one chain more, cut
# tiles in both directions; four blocks (the movers' turn) and five.
SHAPES = [(2, 3), (64, 8), (65, 9), (70, 5), (63, 33), (130, 40), (200, 7), (3, 300),
          (5, 4, 3), (8, 8, 8), (9, 9, 9), (7, 17, 8), (16, 8, 16), (33, 20, 25), (100, 3, 9)]


@pytest.mark.parametrize("holes", [False, True])
@pytest.mark.parametrize("kind,fmt", [("ilu_0", "F64"), ("ic_0", "F64"), ("ilu_0", "F32"), ("ilu_0", "BF16")])
@pytest.mark.parametrize("shape", SHAPES)
def test_chain_sweeps_same_bits_as_levels(m, shape, kind, fmt, holes):
    rp, ci, va = _grid(shape, holes, 11)
    n = len(rp) - 1
    A = m.compressed2D(n, n, rp, ci, va)
    L = m._lib.lib()
    rng = np.random.default_rng(12)
    plain = rng.uniform(-1, 1, n)
    odd = plain.copy()
    odd[:: max(1, n // 5)] = [-0.0, np.inf, 0.0, -np.inf, np.nan, -0.0][: len(odd[:: max(1, n // 5)])]
    out = {}
    for sched in (m._lib.SWEEP_AUTO, m._lib.SWEEP_LEVELS):
        m._lib.check(L.mtl4g_set_sweep_schedule(sched))
        try:
            P = getattr(m.pc, kind)(A, getattr(m, fmt))
        finally:
            m._lib.check(L.mtl4g_set_sweep_schedule(m._lib.SWEEP_AUTO))
        got = []
        for b in (plain, odd, plain):   # the last: nothing of the odd input is left behind
            bd = m.dense_vector(b)
            got += [P.solve(bd).numpy(), P.adjoint_solve(bd).numpy()]
        out[sched] = got
    for a, b in zip(out[m._lib.SWEEP_AUTO], out[m._lib.SWEEP_LEVELS]):
        same = (a.view(np.uint64) == b.view(np.uint64)) | (np.isnan(a) & np.isnan(b))
        assert same.all(), int((~same).sum())
