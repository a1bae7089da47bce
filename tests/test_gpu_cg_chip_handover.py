"""itl::cg on the chip when launches are refused (another kernel holds the
compute units): the iterations launched one by one go on from the same state
and give the same bits; and when a wait between workgroups gives up.  Refusals
and short waits are set from the host, every kernel ends normally."""
import contextlib
import ctypes as C
import threading
import time

import numpy as np
import pytest

from test_gpu_resident import _matrix
from test_gpu_resident_large import _grid

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def m():
    import mtl4_amd
    return mtl4_amd


@contextlib.contextmanager
def _limits(m, first=0, count=0, polls=0):
    L = m._lib.lib()
    m._lib.check(L.mtl4g_set_cg_chip_limits(first, count, polls))
    try:
        yield
    finally:
        m._lib.check(L.mtl4g_set_cg_chip_limits(0, 0, 0))


def _info(m):
    i = m._lib.CgChipInfo()
    m._lib.check(m._lib.lib().mtl4g_cg_chip(C.byref(i)))
    return i


def _cg(m, A, P, b, steps):
    import io
    x = m.dense_vector(A.num_rows())
    it = m.cyclic_iteration(b, steps, 0.0, 0.0, 1, io.StringIO())
    m.cg(A, x, b, P, it)
    return x.numpy(), it.history, _info(m)


# each operand; one workgroup that reads p from memory, up to 128 workgroups
# (sums of all) and more (sums of groups, a number that 8 does not divide),
# workgroups that end inside their rows; x and the inverse diagonal kept and streamed
CASES = [("grid2d", (3, 1025), 1), ("grid2d", (300, 301), 1), ("grid3d", (61, 61, 61), 2), ("grid3d", (101, 103, 97), 2),
         ("random", 700, None), ("random", 70003, None), ("large", (1500, 1000), 6), ("large", (102, 103, 102), 6),
         ("large", (160, 160, 160), 6)]


@pytest.mark.parametrize("pc", ["diagonal", "identity"])
@pytest.mark.parametrize("kind,size,operand", CASES)
def test_refused_launches_give_the_same_bits(m, kind, size, operand, pc):
    rp, ci, va = _grid(size) if kind == "large" else _matrix(kind, size)
    n = len(rp) - 1
    print("handover", kind, size, n, pc, flush=True)
    A = m.compressed2D(n, n, rp, ci, va)
    P = m.pc.diagonal(A) if pc == "diagonal" else None
    b = A * m.dense_vector(np.random.default_rng(5).uniform(-1, 1, n))
    steps = 70
    want, hist, info = _cg(m, A, P, b, steps)
    assert info.operand == operand if operand else 3 <= info.operand <= 5
    assert info.refused == info.single_steps == 0 and info.launches >= 1
    # every launch refused; the first one only: the chip takes over from the single steps
    for first, count in ((0, 10 ** 6), (0, 1)):
        with _limits(m, first, count):
            x, h, info = _cg(m, A, P, b, steps)
        assert np.array_equal(x, want) and np.array_equal(h, hist)
        assert info.refused >= 1 and info.single_steps >= 32
        assert (info.refused == info.launches) == (count > 1)


def test_solve_resumed_after_launches_on_the_chip(m):
    rp, ci, va = _matrix("diffusion", 33)
    n = len(rp) - 1
    A = m.compressed2D(n, n, rp, ci, va)
    P = m.pc.diagonal(A)
    b = m.dense_vector(np.random.default_rng(7).uniform(-1, 1, n))
    want, hist, _ = _cg(m, A, P, b, 700)
    with _limits(m, 1, 6):
        x, h, info = _cg(m, A, P, b, 700)
    assert info.refused >= 4 and info.launches > info.refused and info.single_steps >= 32
    assert np.array_equal(x, want) and np.array_equal(h, hist)


@pytest.mark.parametrize("kind,size,fmt", [("random", 90000, "F32"), ("random", 90000, "BF16"),
                                           ("grid3d", (61, 61, 61), "F32"), ("large", (130, 130, 130), "F32"),
                                           ("large", (164, 160, 160), "BF16")])
def test_refused_launches_of_a_mixed_solve(m, kind, size, fmt):
    rp, ci, va = _grid(size) if kind == "large" else _matrix(kind, size)
    n = len(rp) - 1
    print("handover, mixed", kind, size, n, fmt, flush=True)
    A = m.compressed2D(n, n, rp, ci, va)
    P = m.pc.diagonal(A, m.F32)
    b = A * m.dense_vector(np.random.default_rng(8).uniform(-1, 1, n))

    def solve():
        x = m.dense_vector(n)
        err, st = m.ir_solve(A, x, b, m.basic_iteration(b, 20000, 1e-10), P, value_format=getattr(m, fmt))
        assert err == 0 and st["relres"] <= 1e-10
        return x.numpy(), st, _info(m)

    want, st, info = solve()
    assert info.operand != 0 and info.refused == 0
    for first, count in ((0, 10 ** 6), (1, 2)):
        with _limits(m, first, count):
            x, st2, info = solve()
        assert info.refused >= 1 and st2 == st
        assert np.array_equal(x, want)


@pytest.mark.parametrize("kind,size", [("grid3d", (61, 61, 61)), ("random", 70003), ("large", (140, 140, 140))])
def test_a_wait_that_gives_up_ends_the_solve(m, kind, size):
    rp, ci, va = _grid(size) if kind == "large" else _matrix(kind, size)
    n = len(rp) - 1
    print("wait gives up", kind, size, n, flush=True)
    A = m.compressed2D(n, n, rp, ci, va)
    P = m.pc.diagonal(A)
    b = m.dense_vector(np.random.default_rng(5).uniform(-1, 1, n))
    want, hist, _ = _cg(m, A, P, b, 20)
    S = m.Solver(A, P)
    with _limits(m, polls=1), pytest.raises(m._lib.MtlError, match="bounded wait"):
        S.solve(m.dense_vector(n), b, m.basic_iteration(b, 20, 0.0))
    # the handle solves again
    x = m.dense_vector(n)
    S.solve(x, b, m.basic_iteration(b, 20, 0.0))
    assert np.array_equal(x.numpy(), want)


def test_solve_beside_a_batch_that_holds_compute_units(m):
    """A batched solve keeps a workgroup on every compute unit for milliseconds;
    the CG solves beside it give their bits and do not stand still."""
    import torch
    from mtl4_amd import generators as gen
    rp, ci, va = _matrix("grid3d", (61, 61, 61))
    n = len(rp) - 1
    A = m.compressed2D(n, n, rp, ci, va)
    P = m.pc.diagonal(A)
    b = m.dense_vector(np.random.default_rng(5).uniform(-1, 1, n))
    want, hist, _ = _cg(m, A, P, b, 400)
    systems = [gen.laplacian_setup(96, 96)] * 300
    B = m.Batch(systems)
    nb = sum(len(s[0]) - 1 for s in systems)
    bb = m.dense_vector(np.random.default_rng(6).uniform(-1, 1, nb))
    xb = m.dense_vector(nb)
    B.solve(xb, bb, rtol=1e-8)   # its graph is recorded here
    stop, failed = threading.Event(), []

    def batches():
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                while not stop.is_set():
                    xb.t.zero_()
                    B.solve(xb, bb, rtol=1e-8)
        except Exception as e:   # noqa: BLE001
            failed.append(e)

    t = threading.Thread(target=batches)
    t.start()
    try:
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(5):
                t0 = time.time()
                x, h, info = _cg(m, A, P, b, 400)
                print("beside a batch: %.1f ms, %d launches, %d refused, %d single steps"
                      % (1e3 * (time.time() - t0), info.launches, info.refused, info.single_steps), flush=True)
                assert np.array_equal(x, want) and np.array_equal(h, hist)
    finally:
        stop.set()
        t.join(60)
    assert not failed and not t.is_alive()


@pytest.mark.parametrize("sizes", [(102, 103, 102), (160, 160, 160)])
def test_a_launch_of_a_large_system_stays_short(m, sizes):
    """All compute units are held for about 5 ms at most: iterations per launch
    fall with the rows where these set an iteration's time."""
    rp, ci, va = _grid(sizes)
    n = len(rp) - 1
    A = m.compressed2D(n, n, rp, ci, va)
    b = A * m.dense_vector(np.random.default_rng(5).uniform(-1, 1, n))
    x, h, info = _cg(m, A, m.pc.diagonal(A), b, 300)
    assert info.operand == 6 and info.steps * n * 8 <= 256 * (8 << 20) < (info.steps + 1) * n * 8
    assert info.launches >= -(-300 // info.steps) and len(h) == 301 and np.isfinite(h).all()


def test_a_waiting_solve_is_served_in_turn(m):
    """Two solves that each need the whole GPU: the one that came later does not
    wait until the other has finished all its iterations."""
    import torch
    rp, ci, va = _matrix("grid3d", (99, 99, 99))
    n = len(rp) - 1
    A = m.compressed2D(n, n, rp, ci, va)
    b = m.dense_vector(np.random.default_rng(5).uniform(-1, 1, n))
    done = {}

    def work(name, steps, delay):
        with torch.cuda.stream(torch.cuda.Stream()):
            time.sleep(delay)
            x = m.dense_vector(n)
            m.cg(A, x, b, None, m.basic_iteration(b, steps, 0.0))
            done[name] = time.time()

    work("first", 8, 0)
    # 30,000 iterations of about 18 us: more than half a second
    ts = [threading.Thread(target=work, args=a) for a in (("long", 30000, 0), ("short", 600, 0.1))]
    for t in ts:
        t.start()
    for t in ts:
        t.join(60)
    assert not any(t.is_alive() for t in ts)
    print("short ended %.0f ms before long" % (1e3 * (done["long"] - done["short"])), flush=True)
    assert done["short"] < done["long"]


def test_a_solve_behind_queued_work_keeps_nobody_waiting(m):
    """A solve on a stream with other work under way has claimed compute units that it
    does not use yet: a solve on an idle stream waits for them for a while at most, and
    ends first."""
    import torch
    rp, ci, va = _matrix("grid3d", (61, 61, 61))
    n = len(rp) - 1
    A = m.compressed2D(n, n, rp, ci, va)
    b = m.dense_vector(np.random.default_rng(5).uniform(-1, 1, n))
    want, hist, _ = _cg(m, A, None, b, 50)
    y = torch.zeros(64, device="cuda")
    solvers = {k: m.Solver(A) for k in ("queued", "idle")}   # no allocation, which waits for the device, in the solves
    for S in solvers.values():
        S.solve(m.dense_vector(n), b, m.basic_iteration(1.0, 2, 0.0))

    def timed(f):
        torch.cuda.synchronize()
        t0 = time.time()
        f()
        return time.time() - t0

    def nap(count, s):   # kernels of one workgroup that end by the clock
        with torch.cuda.stream(s):
            for _ in range(count):
                torch.cuda._sleep(10 ** 6)

    def add(s):
        with torch.cuda.stream(s):
            y.add_(1)
        s.synchronize()

    queued = torch.cuda.Stream()
    nap(1, queued)
    each = timed(lambda: (nap(10, queued), queued.synchronize())) / 10
    naps = max(1, min(2000, int(0.4 / each)))
    # a stream that does not share the other's hardware queue
    idle = None
    for s in [torch.cuda.Stream() for _ in range(8)]:
        add(s)
        if timed(lambda: (nap(naps, queued), add(s))) < 0.2:
            idle = s
            break
    torch.cuda.synchronize()
    assert idle is not None
    ended, xs = {}, {}

    def work(name, s, delay, count):
        with torch.cuda.stream(s):
            time.sleep(delay)
            x = m.dense_vector(n)
            s.synchronize()
            nap(count, s)
            solvers[name].solve(x, b, m.basic_iteration(1.0, 50, 0.0))
            ended[name], xs[name] = time.time(), x.numpy()

    ts = [threading.Thread(target=work, args=a)
          for a in (("queued", queued, 0, naps), ("idle", idle, 0.1, 0))]
    for t in ts:
        t.start()
    for t in ts:
        t.join(60)
    assert not any(t.is_alive() for t in ts)
    print("%d naps of %.2f ms; idle ended %.0f ms before queued"
          % (naps, 1e3 * each, 1e3 * (ended["queued"] - ended["idle"])), flush=True)
    assert ended["idle"] < ended["queued"]
    assert np.array_equal(xs["idle"], want) and np.array_equal(xs["queued"], want)
