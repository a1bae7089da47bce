#!/usr/bin/env python3
"""Benchmark of the MTL4 sparse Krylov path on one MI355X.

Workload (one step = one complete solve, inputs resident in HBM):
  itl::cg + itl::pc::diagonal, FP64, relative tolerance 1e-10, on the 160^3
  7-point variable-coefficient diffusion matrix (N = 4,096,000,
  nnz = 28,518,400, face coefficients log-uniform in [1e-2, 1e2], seed 0),
  b = A*x_true with x_true ~ U[-1, 1] (seed 1), x0 = 0.
Reported beside it (same matrix, same b):
  * mixed-precision refinement (FP64 residual/correction/norm on the GPU,
    inner CG in FP32 on FP32 values) to the same 1e-10, and its speedup;
  * p50/p99 latency per solve for both;
  * SpMV GB/s (y = A*x, FP64 values, int32 indices) on this matrix and on the
    random N = 2M Poisson(16) matrix, with the roofline of the SpMV kernel;
  * the CPU oracle timed on a bounded sample on this host's cores.

    python bench.py [--steps K] [--warmup W] [--gpus 1]
"""
import argparse
import ctypes as C
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "CG solves/s + p99 latency, mixed-prec vs FP64 at rel resid 1e-10; SpMV GB/s"
HBM_PEAK_GBS = 8000.0


def spmv_bytes(n, nnz, vb=8, ib=4):
    """Algorithmic bytes of y = A*x: values+indices, row pointers, x once, y once."""
    return nnz * (vb + ib) + (n + 1) * ib + n * vb + n * vb


def sliced_bytes(rowptr, vb=8, ib=4):
    """Algorithmic bytes of y = A*x on the sliced ELL layout: the padded
    values+indices of slices of 64 rows, one 8-byte offset per slice, x
    once, y once (no row pointers)."""
    lens = np.diff(np.asarray(rowptr, dtype=np.int64))
    n = len(lens)
    nsl = (n + 63) // 64
    padded = np.zeros(nsl * 64, dtype=np.int64)
    padded[:n] = lens
    entries = int(padded.reshape(nsl, 64).max(axis=1).sum()) * 64
    return entries * (vb + ib) + (nsl + 1) * 8 + n * vb + n * vb


def dia_bytes(rowptr, col, vb=8):
    """Algorithmic bytes of y = A*x on the diagonal layout: one value per row
    and diagonal (absent entries included), the diagonal offsets, x once, y
    once (no column indices, no row pointers)."""
    lens = np.diff(np.asarray(rowptr, dtype=np.int64))
    rows = np.repeat(np.arange(len(lens), dtype=np.int64), lens)
    ndiag = len(np.unique(np.asarray(col, dtype=np.int64) - rows))
    n = len(lens)
    padded_rows = (n + 63) // 64 * 64   # slice-major: the last slice of 64 rows is whole
    return ndiag * padded_rows * vb + ndiag * 4 + n * vb + n * vb


def dia_sym_bytes(rowptr, col, vb=8):
    """Algorithmic bytes of y = A*x on the symmetric diagonal layout: one
    value per row and stored diagonal (offsets >= 0, absent entries
    included), the offsets and their map, x once, y once; the entries below
    the diagonal are the stored ones of other rows, read again."""
    lens = np.diff(np.asarray(rowptr, dtype=np.int64))
    rows = np.repeat(np.arange(len(lens), dtype=np.int64), lens)
    offs = np.unique(np.asarray(col, dtype=np.int64) - rows)
    nst = int((offs >= 0).sum())
    n = len(lens)
    padded_rows = (n + 63) // 64 * 64
    return nst * padded_rows * vb + 2 * len(offs) * 4 + n * vb + n * vb


def timed_spmv(m, torch, A, x, y, reps):
    """Average duration of the SpMV kernel, HIP events on the launch stream."""
    for _ in range(3):
        A.mult(x, y)
    s = torch.cuda.current_stream()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record(s)
    for _ in range(reps):
        A.mult(x, y)
    e1.record(s)
    e1.synchronize()
    return e0.elapsed_time(e1) / 1000.0 / reps


def timed_spmv_in_cg(m, torch, A, p, q, reps):
    """Average duration of the SpMV q = A*p where each launch follows the
    vector passes of one CG iteration (x += a*p; r -= a*q; z = d.*r;
    p = 0.5*p + z: 14 passes of n doubles, 459 MB at 160^3), as inside the
    solve: the matrix is then read from HBM, not left in the 256 MB MALL by
    the previous product.  HIP events bracket each SpMV on its launch
    stream; the first 3 are warm-up."""
    n = len(p.t)
    gen = torch.Generator(device="cuda").manual_seed(3)
    xv, rv, zv, dv = (torch.rand(n, dtype=torch.float64, device="cuda", generator=gen) for _ in range(4))
    s = torch.cuda.current_stream()
    ev = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
          for _ in range(reps + 3)]
    for e0, e1 in ev:
        xv.add_(p.t, alpha=1e-6)
        rv.sub_(q.t, alpha=1e-6)
        torch.mul(dv, rv, out=zv)
        p.t.mul_(0.5).add_(zv)
        e0.record(s)
        A.mult(p, q)
        e1.record(s)
    s.synchronize()
    return sum(e0.elapsed_time(e1) for e0, e1 in ev[3:]) / 1000.0 / reps


def hbm_context(torch):
    """What plain library kernels reach on this GPU (context for the
    roofline, not a ceiling of the SpMV): a 2 GiB device copy (torch copy_)
    and a 2 GiB read (torch.sum), 5 repetitions each after a warm-up."""
    src = torch.ones(256 << 20, dtype=torch.float64, device="cuda")
    dst = torch.empty_like(src)
    nbytes = src.numel() * 8
    out = {}
    for name, fn, moved in (("copy_GBs", lambda: dst.copy_(src), 2 * nbytes),
                            ("sum_read_GBs", lambda: torch.sum(src), nbytes)):
        fn()
        s = torch.cuda.current_stream()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(s)
        for _ in range(5):
            fn()
        e1.record(s)
        e1.synchronize()
        out[name] = round(moved / (e0.elapsed_time(e1) / 5 / 1000.0) / 1e9, 1)
    del src, dst
    return out


def traffic_key(m, kern, grid=0):
    """Name of a CSR kernel configuration as in the PMC traffic table (the
    persistent kernels by the workgroups per CU they actually launch)."""
    kind, group, rows = kern
    if grid:
        group = grid // 256
    if kind == m._lib.SPMV_STREAM:
        return "stream/%d/%d" % (rows, group)
    if kind == m._lib.SPMV_STREAM2:
        return "stream2/%d/%d" % (rows, group)
    if kind == m._lib.SPMV_TILE:
        return "tile/%d" % rows
    if kind == m._lib.SPMV_SCALAR:
        return "scalar/%d" % group
    if kind == m._lib.SPMV_SLICED:
        return "sliced/%d/%d" % (rows, group)
    if kind == m._lib.SPMV_DIA:
        return "dia/%d/%d" % (rows, group)
    if kind == m._lib.SPMV_DIA_SYM:
        return "dia_sym/%d/%d" % (rows, group)
    return None


def load_traffic(key):
    """HBM bytes per launch of this SpMV configuration, from the two
    rocprofv3 PMC passes (FETCH_SIZE, WRITE_SIZE) recorded under profiles/,
    scaled by the counters' readings on a 512 MiB device copy."""
    p = os.path.join(ROOT, "profiles", "spmv_diffusion3d_160_traffic.json")
    if key is None or not os.path.exists(p):
        return None
    try:
        cfg = json.load(open(p))["configs"].get(key)
        return cfg["traffic_bytes"] if cfg else None
    except (OSError, ValueError, KeyError):
        return None


def cpu_model():
    """The host CPU's model name and the cores this process may use."""
    model = "unknown"
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    try:
        avail = len(os.sched_getaffinity(0))
    except AttributeError:
        avail = os.cpu_count()
    return model, avail


def cpu_baseline(rp, ci, va, b, iters_gpu, cpu_iters, max_solve_s=25.0):
    """The CPU oracle's cg + diagonal on the same system: MTL4's OpenMP build
    restated (mat_vec_mult.hpp:648-674, dot.hpp:112-134, reduction.hpp,
    vec_vec_aop_expr.hpp) on the host cores OpenMP is given (OMP_NUM_THREADS),
    full solves after a 20-iteration warm-up (the median of up to 5 while
    they fit max_solve_s in total); and MTL4's default single-thread build,
    timed on cpu_iters iterations and scaled to the GPU's iteration count."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import orc
    O = orc.Matrix(rp, ci, va)
    model, avail = cpu_model()
    threads = orc.omp_threads()
    orc.cg_diag_omp(O, b, threads=threads, max_iter=20, rtol=1e-10)   # warm-up (page-in, thread team)
    times, its = [], []
    t_all = time.perf_counter()
    while len(times) < 5:
        t0 = time.perf_counter()
        _, st, it = orc.cg_diag_omp(O, b, threads=threads, max_iter=4 * iters_gpu, rtol=1e-10)
        times.append(time.perf_counter() - t0)
        its.append(it.i)
        if time.perf_counter() - t_all + times[-1] > max_solve_s:
            break
    t_omp = float(np.median(times))
    # single thread, MTL4's default build
    P = orc.Preconditioner("diagonal", O)
    t0 = time.perf_counter()
    orc.cg(O, b, P, max_iter=cpu_iters, rtol=1e-10)
    dt = time.perf_counter() - t0
    per_iter = dt / cpu_iters
    return {"value": round(1.0 / t_omp, 5), "unit": "solves/s", "cores": threads, "kind": "port",
            "sample": "%d full CG+diagonal solves of the 160^3 system (%d iterations, median %.2f s) with MTL4's "
                      "OpenMP passes on %d threads" % (len(times), its[-1], t_omp, threads),
            "cpu_model": model, "cores_available": avail,
            "single_thread": {"value": round(1.0 / (per_iter * iters_gpu), 5), "unit": "solves/s", "cores": 1,
                              "sample": "%d CG+diagonal iterations (%.1f s, %.1f ms/iteration), scaled to the "
                                        "GPU's %d iterations" % (cpu_iters, dt, per_iter * 1e3, iters_gpu)}}


T_START = time.perf_counter()


def log(msg):
    """Progress on stderr (the JSON result is the only line on stdout)."""
    print("[bench %7.1fs] %s" % (time.perf_counter() - T_START, msg), file=sys.stderr, flush=True)


def guarded(fn):
    """Run one extra measurement; a failure is recorded, not fatal."""
    try:
        return fn()
    except Exception as e:   # the headline line must still be printed
        return {"error": "%s: %s" % (type(e).__name__, e)}


def relres_of(m, A, x, b, bnorm):
    r = m.dense_vector(A.num_rows())
    r.assign(b)
    A.mult(x, r, m.MINUS)
    return m.two_norm(r) / bnorm


def pair_section(m, torch, A, b, bnorm, pc, method, x_ref=None):
    """One FP64 solve and one mixed-precision (FP32 values, reliable
    updates) solve of A x = b with the given preconditioner; relative
    residuals in FP64 and the mixed solution's error against the FP64 one."""
    n = A.num_rows()
    log("%s: preconditioners (%s, n=%d)" % ("cg" if method == m.CG else "bicgstab", pc, n))
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    P64 = getattr(m.pc, pc)(A)
    t_setup = time.perf_counter() - t0
    P64.refactor()   # warm: the factorization kernels' first launch
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    P64.refactor()   # the device factorization alone, with the plan made at construction
    torch.cuda.synchronize()
    t_refactor = time.perf_counter() - t0
    log("  setup %.3f s (pattern plan, device factorization, sweeps), refactor %.4f s" % (t_setup, t_refactor))
    P32 = getattr(m.pc, pc)(A, m.F32)
    # the FP32 and BF16 value copies and their product's tuning are set-up,
    # like the preconditioners: built before the timed solves
    A.prepare(m.F32)
    A.prepare(m.BF16)
    torch.cuda.synchronize()
    S = m.Solver(A, P64, method=method)
    x = m.dense_vector(n)
    it = m.basic_iteration(bnorm, 100000, 1e-10)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    err = S.solve(x, b, it)
    torch.cuda.synchronize()
    t64 = time.perf_counter() - t0
    log("  FP64 solve: %d iterations, %.3f s" % (it.iterations(), t64))
    xm = m.dense_vector(n)
    # a recurrence that stagnates stops at 2x the FP64 iteration count
    itm = m.basic_iteration(bnorm, 2 * max(it.iterations(), 10), 1e-10)
    t0 = time.perf_counter()
    failure = None
    try:
        errm, st = m.ir_solve(A, xm, b, itm, P32, method=method, value_format=m.F32, mode="reliable")
    except m.MtlError as e:   # the FP32 recurrence broke down or overflowed
        errm, st, failure = -1, {"inner_total": itm.iterations(), "outer": -1}, "%s: %s" % (type(e).__name__, e)
    torch.cuda.synchronize()
    tm = time.perf_counter() - t0
    log("  mixed solve: %d iterations, error %d, %.3f s" % (st["inner_total"], errm, tm))
    ref = x.t if x_ref is None else x_ref
    rel_err = float(torch.linalg.vector_norm(xm.t - ref) / torch.linalg.vector_norm(ref))
    # BF16-stored preconditioner values (FP32 matrix values), same refinement
    P16 = getattr(m.pc, pc)(A, m.BF16)
    xb = m.dense_vector(n)
    itb = m.basic_iteration(bnorm, 2 * max(it.iterations(), 10), 1e-10)
    t0 = time.perf_counter()
    fail16 = None
    try:
        errb, stb = m.ir_solve(A, xb, b, itb, P16, method=method, value_format=m.F32, mode="reliable")
    except m.MtlError as e:
        errb, stb, fail16 = -1, {"inner_total": itb.iterations(), "outer": -1}, "%s: %s" % (type(e).__name__, e)
    torch.cuda.synchronize()
    tb = time.perf_counter() - t0
    log("  mixed solve, BF16 preconditioner: %d iterations, error %d, %.3f s" % (stb["inner_total"], errb, tb))
    rel_err_b = float(torch.linalg.vector_norm(xb.t - ref) / torch.linalg.vector_norm(ref))
    rec = ("FP32 recurrence on FP32 values" if method == m.CG else
           "FP64 vectors on FP32 values") + ", FP32 preconditioner values, FP64 refresh at 0.1x"
    return {"fp64": {"solves_per_s": round(1 / t64, 4), "iterations": it.iterations(), "error_code": err,
                     "relres": relres_of(m, A, x, b, bnorm)},
            "mixed_f32": {"solves_per_s": round(1 / tm, 4), "iterations": st["inner_total"],
                          "fp64_refreshes": st["outer"], "error_code": errm, "failure": failure,
                          "relres": relres_of(m, A, xm, b, bnorm), "rel_err_vs_fp64": rel_err,
                          "recurrence": rec},
            "mixed_bf16_pc": {"solves_per_s": round(1 / tb, 4), "iterations": stb["inner_total"],
                              "fp64_refreshes": stb["outer"], "error_code": errb, "failure": fail16,
                              "relres": relres_of(m, A, xb, b, bnorm), "rel_err_vs_fp64": rel_err_b,
                              "speedup": round(t64 / tb, 3),
                              "recurrence": rec.replace("FP32 preconditioner", "BF16 preconditioner")},
            "speedup": round(t64 / tm, 3), "steps": 1,
            "pc_setup_s": round(t_setup, 4), "pc_refactor_s": round(t_refactor, 5)}


def c3_section(m, torch, gen):
    """Mixed-precision cases: cg + ic_0 on 128^3 diffusion; bicgstab + ilu_0
    on the 1024^2 upwind convection-diffusion problem (Peclet 10)."""
    def case(make, pc, method):
        rp, ci, va = make()
        n = len(rp) - 1
        A = m.compressed2D(n, n, rp, ci, va)
        A.autotune()
        b = A * m.dense_vector(np.random.default_rng(1).uniform(-1.0, 1.0, n))
        return pair_section(m, torch, A, b, m.two_norm(b), pc, method)

    log("c3: diffusion3d 128^3")
    out = {"cg_ic0_diffusion3d_128": guarded(lambda: case(lambda: gen.diffusion3d(128, seed=0), "ic_0", m.CG))}
    log("c3: convection-diffusion 1024^2")
    out["bicgstab_ilu0_convdiff_1024"] = guarded(lambda: case(
        lambda: gen.convection_diffusion2d(1024, peclet=10.0, seed=0), "ilu_0", m.BICGSTAB))
    return out


def solvers_section(m, torch, gen):
    """Every Krylov method of the library on one workload: diffusion3d 128^3
    (2,097,152 rows), b = A*x_true, diagonal preconditioner (left for the
    methods that take two), FP64, rtol 1e-10, default reduction order.
    Per method: iterations, best of two solves, time per iteration and per
    product A*v.  GMRES runs MTL4's algorithm, whose cycles of more than one
    Krylov vector follow no textbook identity: it gets a fixed budget of 300
    iterations and reports its residual instead of a convergence time."""
    rp, ci, va = gen.diffusion3d(128, seed=0)
    n = len(rp) - 1
    A = m.compressed2D(n, n, rp, ci, va)
    A.autotune()
    b = A * m.dense_vector(np.random.default_rng(1).uniform(-1.0, 1.0, n))
    bnorm = m.two_norm(b)
    P = m.pc.diagonal(A)
    runs = [("cg", 1, lambda x, it: m.cg(A, x, b, P, it)),
            ("bicgstab", 2, lambda x, it: m.bicgstab(A, x, b, P, it)),
            ("cgs", 2, lambda x, it: m.cgs(A, x, b, P, it)),
            ("tfqmr", 2, lambda x, it: m.tfqmr(A, x, b, P, None, it)),
            ("bicgstab_2", 4, lambda x, it: m.bicgstab_2(A, x, b, P, it)),
            ("bicgstab_ell_4", 8, lambda x, it: m.bicgstab_ell(A, x, b, P, None, it, 4)),
            ("gmres_30", 1, lambda x, it: m.gmres(A, x, b, P, None, it, 30))]
    out = {"workload": "diffusion3d 128^3, pc::diagonal, FP64, rtol 1e-10", "products_per_iteration": {}}
    for name, prods, fn in runs:
        def one():
            best, it_n, err, rel = 1e30, 0, 0, 0.0
            for _ in range(2):
                x = m.dense_vector(n)
                it = m.basic_iteration(bnorm, 300 if name.startswith("gmres") else 5000, 1e-10)
                torch.cuda.synchronize()
                t0 = time.perf_counter()
                err = fn(x, it)
                torch.cuda.synchronize()
                best = min(best, time.perf_counter() - t0)
                it_n = it.iterations()
                rel = relres_of(m, A, x, b, bnorm)
            return {"iterations": it_n, "error_code": err, "relres": rel, "solve_s": round(best, 4),
                    "ms_per_iteration": round(1000 * best / max(it_n, 1), 4),
                    "ms_per_product": round(1000 * best / max(it_n * prods, 1), 4)}
        log("solvers: %s" % name)
        out[name] = guarded(one)
        out["products_per_iteration"][name] = prods
    return out


def batch_systems(gen, count, seed=0):
    """Uneven SPD systems: N log-uniform in [256, 65536], families 2D 5-point,
    3D 7-point and random diagonally dominant (about 12 non-zeros per row)."""
    rng = np.random.default_rng(seed)
    out = []
    for k in range(count):
        n = int(round(np.exp(rng.uniform(np.log(256), np.log(65536)))))
        fam = int(rng.integers(0, 3))
        if fam == 0:
            a = max(2, int(round(np.sqrt(n))))
            out.append(gen.laplacian_setup(a, max(2, int(round(n / a)))))
        elif fam == 1:
            a = max(2, int(round(n ** (1.0 / 3.0))))
            out.append(gen.laplacian3d(a, a, max(2, int(round(n / (a * a))))))
        else:
            out.append(gen.random_spd(n, seed=seed * 100000 + k))
    return out


def batched_section(m, torch, gen, count):
    """All systems in one persistent graph-replayed launch, cg + diagonal to
    relative residual 1e-10: FP64 against mixed precision (FP32 values,
    FP64 reliable updates)."""
    t0 = time.perf_counter()
    log("batched: generating %d systems" % count)
    systems = batch_systems(gen, count)
    log("batched: uploading")
    B = m.Batch(systems)
    rows = int(B.nrows)
    b = m.dense_vector(np.random.default_rng(7).uniform(-1.0, 1.0, rows))
    x = m.dense_vector(rows)
    x0 = m.dense_vector(rows)
    setup_s = time.perf_counter() - t0
    out = {"systems": count, "rows": rows, "nnz": int(len(B.col)), "setup_s": round(setup_s, 2)}
    for name, prec in (("fp64", m.F64), ("mixed_f32", m.F32)):
        log("batched: %s tune" % name)
        tune_ms, shape = B.tune(x, x0, b, precision=prec, rtol=1e-10)
        log("batched: %s solves (tuned %.1f ms)" % (name, tune_ms))
        times = []
        for rep in range(3):
            x.t.zero_()
            torch.cuda.synchronize()
            t1 = time.perf_counter()
            res = B.solve(x, b, precision=prec, rtol=1e-10)
            times.append(time.perf_counter() - t1)
        its = np.array([r["iterations"] for r in res])
        errs = sum(1 for r in res if r["error"] or r["status"])
        rel = np.array([r["resid"] / r["norm_r0"] for r in res if r["norm_r0"] > 0])
        tbest = min(times)
        out[name] = {"systems_per_s": round(count / tbest, 2), "batch_ms": round(1000 * tbest, 3),
                     "shape": list(shape), "tune_best_ms": round(tune_ms, 3), "errors": errs,
                     "iterations_mean": round(float(its.mean()), 1), "iterations_max": int(its.max()),
                     "max_relres_reported": float(rel.max()) if rel.size else None}
    out["mixed_speedup"] = round(out["mixed_f32"]["systems_per_s"] / out["fp64"]["systems_per_s"], 3)
    out["graph"] = dict(zip(("captures", "replays"), B.graph_info()))
    return out


def serving_section(m, torch, gen, nreq, sweep_requests=400, big_rows=65536):
    """Continuous batching over 512 resident matrices (the batched families
    plus 3D stencils up to 96^3), Poisson arrivals, 1-8 right-hand sides per
    request, each request itl::cg or itl::bicgstab with pc::diagonal or
    pc::ilu_0 (uniformly), mixed precision refined to 1e-10: systems above
    65536 rows (the larger 3D stencils) on 8 whole-GPU workers, the rest
    continuously batched on 8 streams.  Against plain FP64 per-request
    launches on one stream (on the first quarter of each trace).  The fixed
    rates 2k, 8k and 20k req/s are above this capacity (their latencies are
    queueing time); a sweep of lower rates finds the highest one the server
    keeps up with (sustained: no backlog builds up over the trace -- the
    median latency of the last quarter of the requests is at most 1.5 x
    that of the first quarter + 50 ms; the p99 then is the service time of
    the largest requests, not queueing)."""
    log("serving: generating 512 matrices")
    systems = batch_systems(gen, 480, seed=1)
    rng = np.random.default_rng(3)
    for k in range(32):
        a = int(round(np.exp(rng.uniform(np.log(32), np.log(96)))))
        systems.append(gen.laplacian3d(a, a, a))
    B = m.Batch(systems)
    sizes = np.diff(B.sys_row)
    out = {"matrices": len(systems), "requests_per_rate": nreq, "cap_bytes": 200e9,
           "solvers": "cg | bicgstab  x  diagonal | ilu_0, uniform per request",
           "big_rows": big_rows, "whole_gpu_matrices": int((sizes > big_rows).sum())}
    codes = [m.Server.solver(meth, pc) for meth in (m.CG, m.BICGSTAB)
             for pc in (m._lib.PC_DIAGONAL, m._lib.PC_ILU0)]

    def make_trace(rate, count):
        rg = np.random.default_rng(int(rate))
        return (rg.integers(0, len(systems), count), rg.integers(1, 9, count),
                np.cumsum(rg.exponential(1.0 / rate, count)),
                rg.integers(1, 2 ** 62, count, dtype=np.uint64),
                np.array(codes, np.int32)[rg.integers(0, len(codes), count)])

    def record(lat, arr, st):
        drain = st["wall_s"] - float(arr[-1])
        q = max(1, len(lat) // 4)
        first, last = float(np.median(lat[:q])), float(np.median(lat[-q:]))
        return {"p50_ms": round(1000 * float(np.percentile(lat, 50)), 3),
                "p99_ms": round(1000 * float(np.percentile(lat, 99)), 3),
                "solves_per_s": round(st["solves"] / st["wall_s"], 1),
                "wall_s": round(st["wall_s"], 3), "last_arrival_s": round(float(arr[-1]), 3),
                "drain_s": round(drain, 3),
                "p50_first_quarter_ms": round(1000 * first, 3), "p50_last_quarter_ms": round(1000 * last, 3),
                "sustained": bool(last <= 1.5 * first + 0.05),
                "launches": st["launches"], "max_inflight": st["max_inflight"], "errors": st["errors"],
                "big_solves": st["big_solves"], "peak_bytes": st["peak_bytes"]}

    rates = (2000.0, 8000.0, 20000.0)
    traces = {rate: make_trace(rate, nreq) for rate in rates}
    for rate in rates:
        out["%dk_req_s" % int(rate / 1000)] = {}
    nbase = max(1, nreq // 4)
    out["baseline_requests_per_rate"] = nbase
    for name, kw in (("mixed", dict(precision=m.F32, streams=8, max_items=1024)),
                     ("fp64_per_request", dict(precision=m.F64, streams=1, max_items=8,
                                                per_request=True))):
        log("serving: %s server" % name)
        Sv = m.Server(B, rtol=1e-10, big_rows=big_rows, cap_bytes=200e9, **kw)
        for rate in rates:
            log("serving: %s at %d req/s" % (name, rate))
            mat, nrhs, arr, seeds, sv = traces[rate]
            if name == "fp64_per_request":
                mat, nrhs, arr, seeds, sv = mat[:nbase], nrhs[:nbase], arr[:nbase], seeds[:nbase], sv[:nbase]
            lat, its, _, st = Sv.run(mat, nrhs, arr, seeds, solver=sv)
            out["%dk_req_s" % int(rate / 1000)][name] = record(lat, arr, st)
        if name == "mixed":
            sweep = {}
            best = None
            for rate in (62.5, 125.0, 250.0, 500.0, 1000.0):
                log("serving: mixed sweep at %d req/s" % rate)
                mat, nrhs, arr, seeds, sv = make_trace(rate, sweep_requests)
                lat, its, _, st = Sv.run(mat, nrhs, arr, seeds, solver=sv)
                sweep["%d_req_s" % int(rate)] = rec = record(lat, arr, st)
                if rec["sustained"] and rec["errors"] == 0:
                    best = rate
            out["mixed_rate_sweep"] = sweep
            out["mixed_sustained_req_s"] = best
        del Sv
    for rate in rates:
        row = out["%dk_req_s" % int(rate / 1000)]
        row["speedup_solves_per_s"] = round(row["mixed"]["solves_per_s"] /
                                            row["fp64_per_request"]["solves_per_s"], 3)
    return out


def random_spmv(m, torch, gen, reps, copy_calibration=False):
    """y = A*x on the random N = 2M matrix (Poisson(16) row lengths, uniform
    columns), the autotuner's kernel: time per launch and GB/s of the CSR
    bytes."""
    log("random SpMV: generating")
    rr = gen.random_sparse(2_000_000, seed=0)
    R = m.compressed2D(2_000_000, 2_000_000, *rr)
    R.autotune()
    xr = m.dense_vector(np.random.default_rng(2).uniform(-1.0, 1.0, 2_000_000))
    yr = m.dense_vector(2_000_000)
    t = timed_spmv(m, torch, R, xr, yr, reps)
    by = spmv_bytes(2_000_000, len(rr[1]))
    kern = R.get_kernel()
    if copy_calibration:   # a copy of known size for the PMC byte counters
        src = torch.rand(64 << 20, dtype=torch.float64, device="cuda")
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        del src, dst
    torch.cuda.synchronize()
    return {"nnz": int(len(rr[1])), "us": round(t * 1e6, 2), "bytes": by, "GBs": round(by / t / 1e9, 1),
            "kernel": list(kern)}


def sweeps_only(m, torch, gen, steps):
    """solve(P, x) of IC(0) on diffusion3d 160^3 and of ILU(0) on the 1024^2
    convection-diffusion matrix, `steps` times each after one warm-up, with
    the chain pipeline (the default for these grid factors) and with the
    level schedule: time per solve (two sweeps) and the sweeps' algorithmic
    bytes (per sweep nnz_tri*(8+4) + (n+1)*4 + 3*n*8)."""
    import ctypes as C
    L = m._lib.lib()
    out = {}
    for name, mk, kind in (("ic0_diffusion3d_160", lambda: gen.diffusion3d(160, seed=0), "ic_0"),
                           ("ilu0_convdiff_1024", lambda: gen.convection_diffusion2d(1024, peclet=10.0, seed=0),
                            "ilu_0")):
        log("sweeps: %s" % name)
        rp, ci, va = mk()
        n = len(rp) - 1
        A = m.compressed2D(n, n, rp, ci, va)
        x = m.dense_vector(np.random.default_rng(0).uniform(-1.0, 1.0, n))
        row = {"n": n}
        ys = {}
        for sched_name, sched in (("chain", m._lib.SWEEP_AUTO), ("levels", m._lib.SWEEP_LEVELS)):
            m._lib.check(L.mtl4g_set_sweep_schedule(sched))
            try:
                P = getattr(m.pc, kind)(A)
            finally:
                m._lib.check(L.mtl4g_set_sweep_schedule(m._lib.SWEEP_AUTO))
            lo, up = C.c_int(), C.c_int()
            m._lib.check(L.mtl4g_pc_sweeps(P.h, C.byref(lo), C.byref(up)))
            nlo, nup = P.levels()
            nnz_l = len(P.get_L()[1])
            nnz_u = len(P.get_U()[1])
            y = m.dense_vector(n)
            P.solve(x, y)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(steps):
                P.solve(x, y)
            torch.cuda.synchronize()
            dt = (time.perf_counter() - t0) / steps
            by = (nnz_l + nnz_u) * 12 + 2 * ((n + 1) * 4 + 3 * n * 8)
            ys[sched_name] = y.numpy().copy()
            row[sched_name] = {"schedules": [lo.value, up.value], "levels": [nlo, nup],
                               "ms_per_solve": round(1e3 * dt, 4), "bytes_per_solve": by,
                               "GBs": round(by / dt / 1e9, 1)}
            del P
        row["same_bits"] = bool(np.array_equal(ys["chain"].view(np.uint64), ys["levels"].view(np.uint64)))
        row["speedup"] = round(row["levels"]["ms_per_solve"] / row["chain"]["ms_per_solve"], 3)
        out[name] = row
        log("sweeps: %s %s" % (name, json.dumps(row)))
        del A
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--grid", type=int, default=160)
    ap.add_argument("--cpu-iters", type=int, default=150)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--cpu-seconds", type=float, default=25.0,
                    help="time budget of the all-core CPU baseline's full solves")
    ap.add_argument("--spmv-reps", type=int, default=50)
    ap.add_argument("--only-spmv", action="store_true", help="SpMV timing only (profiling runs)")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="with --only-spmv: also copy 512 MiB on the device (PMC calibration)")
    ap.add_argument("--only-sweeps", action="store_true",
                    help="triangular sweep timing only (profiling runs): IC(0) of diffusion3d 160^3 and "
                         "ILU(0) of convection-diffusion 1024^2, --steps solves each")
    ap.add_argument("--sections", default="all",
                    help="extra measurements: all, none, or a list of ic0,c3,solvers,batched,serving")
    ap.add_argument("--kernel", default="",
                    help="SpMV configuration instead of the autotuner's choice, as "
                         "dia_sym|dia|sliced/<entries per chunk 4|8>/<workgroups per CU> "
                         "(profiling runs, where the profiler distorts the autotuner's timings)")
    ap.add_argument("--only", default="", choices=["", "batched", "random-spmv", "serving"],
                    help="one measurement alone (profiling runs): the batched or the serving section, "
                         "or the random N = 2M SpMV (with --copy-calibration: plus a 512 MiB device copy)")
    ap.add_argument("--batch-systems", type=int, default=4096)
    ap.add_argument("--serve-requests", type=int, default=1000)
    ap.add_argument("--serve-big-rows", type=int, default=65536,
                    help="serving: systems above this many rows go to the whole-GPU workers")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py measures one GPU: this build has no multi-GPU path "
              "(--gpus %d requested)" % args.gpus, file=sys.stderr)
        sys.exit(2)

    import torch
    import mtl4_amd as m
    from mtl4_amd import generators as gen
    torch.cuda.set_device(0)
    if args.only_sweeps:
        print(json.dumps(sweeps_only(m, torch, gen, args.steps)))
        return
    if args.only == "batched":
        print(json.dumps(batched_section(m, torch, gen, args.batch_systems)))
        return
    if args.only == "serving":
        print(json.dumps(serving_section(m, torch, gen, args.serve_requests, big_rows=args.serve_big_rows)))
        return
    if args.only == "random-spmv":
        print(json.dumps(random_spmv(m, torch, gen, args.spmv_reps, args.copy_calibration)))
        return

    g = args.grid
    log("diffusion3d %d^3: generating" % g)
    rp, ci, va = gen.diffusion3d(g, seed=0)
    n, nnz = len(rp) - 1, len(ci)
    A = m.compressed2D(n, n, rp, ci, va)
    if args.kernel:
        kinds = {"dia_sym": m._lib.SPMV_DIA_SYM, "dia": m._lib.SPMV_DIA, "sliced": m._lib.SPMV_SLICED}
        kind, unr, pcu = args.kernel.split("/")
        A.set_kernel(kinds[kind], int(pcu), int(unr))
    else:
        A.autotune()                      # CSR kernel and shape for this matrix
    xt = m.dense_vector(np.random.default_rng(1).uniform(-1.0, 1.0, n))
    b = A * xt
    bnorm = m.two_norm(b)

    # ---- SpMV (the dominant kernel of the CG iteration)
    y = m.dense_vector(n)
    t_spmv = timed_spmv(m, torch, A, xt, y, args.spmv_reps)
    pv = m.dense_vector(np.random.default_rng(4).uniform(-1.0, 1.0, n))
    t_ctx = timed_spmv_in_cg(m, torch, A, pv, y, args.spmv_reps)
    del pv
    kern = A.get_kernel()
    # algorithmic bytes of the CSR SpMV (the roofline figure), and the bytes
    # the device layout the autotuner chose moves once: the sliced copy has no
    # row pointers but pads slices of 64 rows, the diagonal copy has no
    # column indices
    by = spmv_bytes(n, nnz)
    layout, by_layout = "csr", by
    if kern[0] == m._lib.SPMV_SLICED:
        layout, by_layout = "sliced_ell", sliced_bytes(rp)
    elif kern[0] == m._lib.SPMV_DIA:
        layout, by_layout = "diagonal", dia_bytes(rp, ci)
    elif kern[0] == m._lib.SPMV_DIA_SYM:
        layout, by_layout = "symmetric_diagonal", dia_sym_bytes(rp, ci)
    spmv_gbs = by / t_spmv / 1e9
    ctx_gbs = by / t_ctx / 1e9
    grid = A.grid()
    traffic = load_traffic(traffic_key(m, kern, grid))
    if kern[0] == m._lib.SPMV_DIA:
        kname = "k_dia (diagonal layout, one lane per row, %d diagonals per chunk, %d workgroups/CU)" % (kern[2], kern[1])
    elif kern[0] == m._lib.SPMV_DIA_SYM:
        kname = ("k_dia_sym (symmetric diagonal layout: offsets >= 0 stored, entries below the diagonal read "
                 "from their mirror images; one lane per row, %d diagonals per chunk, %d workgroups/CU)"
                 % (kern[2], kern[1]))
    elif kern[0] == m._lib.SPMV_SLICED:
        kname = "k_sell (sliced ELL, one lane per row, %d entries per chunk, %d workgroups/CU)" % (kern[2], kern[1])
    elif kern[0] == m._lib.SPMV_VECTOR:
        kname = "k_csrv<%d lanes/row>" % kern[1]
    elif kern[0] == m._lib.SPMV_STREAM:
        kname = "k_csrp (persistent LDS tiles, %d workgroups/CU, %d rows/block)" % (kern[1], kern[2])
    elif kern[0] == m._lib.SPMV_STREAM2:
        kname = "k_csrp (persistent LDS tiles, two blocks ahead, %d workgroups/CU, %d rows/block)" % (kern[1], kern[2])
    elif kern[0] == m._lib.SPMV_SCALAR:
        kname = "k_csrs (one lane per row, %d values per step)" % kern[1]
    else:
        kname = "k_csr (LDS tiles, %d rows/block)" % kern[2]
    roofline = {"bound": "hbm", "kernel": "%s<EpiAssign> (y = A*x, FP64, diffusion3d %d^3)" % (kname, g),
                "config": traffic_key(m, kern, grid), "workgroups": grid,
                "timing": ("in CG context: each timed launch follows one CG iteration's vector "
                           "passes (459 MB), so the matrix comes from HBM as inside the solve"),
                # the kernel's own algorithmic bytes: the layout it reads
                "achieved": round(by_layout / t_ctx / 1e9, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": round(by_layout / t_ctx / 1e9 / HBM_PEAK_GBS, 4), "traffic": traffic,
                "layout": layout, "bytes_per_launch": by_layout,
                "csr_equivalent": {"bytes_per_launch": by, "achieved": round(ctx_gbs, 1),
                                   "frac": round(ctx_gbs / HBM_PEAK_GBS, 4),
                                   "note": "the CSR bytes of y = A*x over the same time"},
                "avg_launch_us": round(t_ctx * 1e6, 2),
                "back_to_back": {"avg_launch_us": round(t_spmv * 1e6, 2),
                                 "achieved": round(by_layout / t_spmv / 1e9, 1),
                                 "csr_equivalent_GBs": round(spmv_gbs, 1),
                                 "note": ("launches in a row: a layout smaller than the 256 MB MALL "
                                          "is then partly read from that cache, not from HBM")}}
    if by_layout < by:
        roofline["note"] = ("achieved counts the bytes the %s layout moves; csr_equivalent counts "
                            "the CSR product's bytes over the same time (more than the layout "
                            "moves, so its frac can exceed 1)" % layout)
    if args.only_spmv:   # the roofline kernel alone (profiling runs)
        if args.copy_calibration:   # a copy of known size for the PMC byte counters
            src = torch.rand(64 << 20, dtype=torch.float64, device="cuda")
            dst = torch.empty_like(src)
            for _ in range(3):
                dst.copy_(src)
            del src, dst
        torch.cuda.synchronize()
        print(json.dumps({"spmv_gbs": spmv_gbs, "roofline": roofline}))
        return
    roofline["hbm_context"] = hbm_context(torch)
    rnd = random_spmv(m, torch, gen, args.spmv_reps)
    rnd_gbs = rnd["GBs"]

    log("SpMV %.1f GB/s; FP64 cg + diagonal" % spmv_gbs)
    # ---- FP64 CG + diagonal: the drop-in path
    P = m.pc.diagonal(A)
    S = m.Solver(A, P)
    x = m.dense_vector(n)

    def fp64_solve():
        x.t.zero_()
        it = m.basic_iteration(bnorm, 100000, 1e-10)
        err = S.solve(x, b, it)
        return err, it

    for _ in range(args.warmup):
        fp64_solve()
    torch.cuda.synchronize()
    lat = []
    t0 = time.perf_counter()
    for _ in range(args.steps):
        t1 = time.perf_counter()
        err, it = fp64_solve()
        lat.append(time.perf_counter() - t1)
    torch.cuda.synchronize()
    t_fp64 = time.perf_counter() - t0
    iters = it.iterations()
    Lb = m._lib.lib()
    chip = m._lib.CgChipInfo()   # how the timed solves ran (operand 0: launch per kernel)
    m._lib.check(Lb.mtl4g_cg_chip(C.byref(chip)))
    # the product q = A*p of that solve: one more solve with HIP events around
    # each of its products (on the solve's stream).  An on-chip solve forms it
    # inside its kernel; the product's own kernel then runs beside each iteration
    tot_us, cnt = C.c_double(), C.c_int64()
    m._lib.check(Lb.mtl4g_set_product_timing(1))
    m._lib.check(Lb.mtl4g_product_timing(C.byref(tot_us), C.byref(cnt)))
    fp64_solve()
    torch.cuda.synchronize()
    m._lib.check(Lb.mtl4g_product_timing(C.byref(tot_us), C.byref(cnt)))
    m._lib.check(Lb.mtl4g_set_product_timing(0))
    q_us = tot_us.value / max(cnt.value, 1)
    if cnt.value > 0 and kern[0] == m._lib.SPMV_DIA_SYM:
        cold = {k: roofline.pop(k) for k in ("kernel", "timing", "achieved", "frac", "traffic", "csr_equivalent",
                                             "avg_launch_us")}
        cold["note"] = ("the same product with y = A*x alone, each launch after 14 vector passes of torch "
                        "kernels (459 MB) that leave little of the matrix in the MALL")
        # the PMC record of the in-solve product holds for the configuration it was
        # taken on, and for the product fused with p.q of a launch-per-kernel solve
        try:
            rec = json.load(open(os.path.join(ROOT, "profiles", "spmv_diffusion3d_160_traffic.json")))
            rec = rec["configs"]["cg_product_in_solve"]
            q_traffic = rec["traffic_bytes"] if not chip.operand and rec.get("config") == traffic_key(m, kern, grid) else None
        except (OSError, ValueError, KeyError):
            q_traffic = None
        roofline.update({
            "kernel": ("%s<EpiCgProduct> (q = A*p launched beside each iteration of an on-chip FP64 CG solve, "
                       "which forms it inside its own kernel; diffusion3d %d^3)" if chip.operand else
                       "%s<EpiCgQ> (q = A*p fused with p.q inside the timed FP64 CG solve, diffusion3d %d^3)")
                      % (kname, g),
            "timing": ("HIP events around each of the %d products of one FP64 CG solve, on the solve's "
                       "stream (mtl4g_set_product_timing)" % cnt.value),
            "achieved": round(by_layout / (q_us * 1e-6) / 1e9, 1),
            "frac": round(by_layout / (q_us * 1e-6) / 1e9 / HBM_PEAK_GBS, 4),
            "traffic": q_traffic,
            "csr_equivalent": {"bytes_per_launch": by, "achieved": round(by / (q_us * 1e-6) / 1e9, 1),
                               "frac": round(by / (q_us * 1e-6) / 1e9 / HBM_PEAK_GBS, 4),
                               "note": "the CSR bytes of y = A*x over the same time"},
            "avg_launch_us": round(q_us, 2),
            "cold_mall_context": cold})
    chip_bytes = None
    if chip.operand == 6:
        # the kernel of the timed solves: per iteration its stored matrix values,
        # p at the diagonals beyond the LDS halo, p written once and, where a lane
        # has more than 16 rows, the inverse diagonal and x twice
        far = 2 if g * g > 1024 else 0
        chip_bytes = by_layout - 16 * n + 8 * n * (far + 1 + (3 if chip.rows_per_lane > 16 else 0))
        it_us = 1e6 * t_fp64 / args.steps / max(iters, 1)
        key = "%s/%d" % (layout, chip.rows_per_lane)
        try:
            rec = json.load(open(os.path.join(ROOT, "profiles", "cg_on_chip_traffic.json")))["configs"].get(key)
            chip_traffic = rec["traffic_bytes_per_iteration"] if rec and rec["N"] == n else None
        except (OSError, ValueError, KeyError):
            chip_traffic = None
        roofline = {"bound": "hbm",
                    "kernel": "k_cg_large (itl::cg + pc::diagonal, FP64, whole iterations on the chip, %d per launch, "
                              "%s layout streamed, %d rows per lane; diffusion3d %d^3)"
                              % (chip.steps, layout, chip.rows_per_lane, g),
                    "config": key, "workgroups": chip.workgroups,
                    "timing": "wall time of the timed solves by their iterations",
                    "achieved": round(chip_bytes / it_us / 1e3, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                    "frac": round(chip_bytes / it_us / 1e3 / HBM_PEAK_GBS, 4), "traffic": chip_traffic,
                    "layout": layout, "bytes_per_iteration": chip_bytes, "us_per_iteration": round(it_us, 2),
                    "note": "bytes the iteration cannot do without; traffic: bytes past the L2 per iteration "
                            "(rocprofv3), with the registers that are kept in scratch",
                    "hbm_context": roofline.pop("hbm_context"), "product": roofline}
    r = m.dense_vector(n)
    r.assign(b)
    A.mult(x, r, m.MINUS)
    relres = m.two_norm(r) / bnorm
    x64 = x.t.clone()

    # ---- mixed precision (reliable updates) to the same FP64 tolerance
    P32 = m.pc.diagonal(A, m.F32)
    xm = m.dense_vector(n)

    def mixed_solve(fmt, max_iter):
        xm.t.zero_()
        itm = m.basic_iteration(bnorm, max_iter, 1e-10)
        try:
            errm, st = m.ir_solve(A, xm, b, itm, P32, value_format=fmt, mode="reliable",
                                  inner_rtol=0.1)
        except m.nonfinite_error:
            errm, st = -6, {"inner_total": itm.iterations(), "outer": -1}
        return errm, itm, st

    def run_mixed(fmt, steps, warmup, max_iter):
        for _ in range(warmup):
            mixed_solve(fmt, max_iter)
        torch.cuda.synchronize()
        latm = []
        t0 = time.perf_counter()
        for _ in range(steps):
            t1 = time.perf_counter()
            errm, itm, st = mixed_solve(fmt, max_iter)
            latm.append(time.perf_counter() - t1)
        torch.cuda.synchronize()
        t_mixed = time.perf_counter() - t0
        r.assign(b)
        A.mult(xm, r, m.MINUS)
        relres_m = m.two_norm(r) / bnorm
        rel_err = float(torch.linalg.vector_norm(xm.t - x64) / torch.linalg.vector_norm(x64))
        vm = steps / t_mixed
        return {"solves_per_s": round(vm, 4), "speedup_vs_fp64": None,
                "relres": relres_m, "rel_err_vs_fp64_solution": rel_err, "error_code": errm,
                "fp32_iterations": st["inner_total"], "fp64_refreshes": st["outer"],
                "p50_ms": round(1000 * float(np.percentile(latm, 50)), 3),
                "p99_ms": round(1000 * float(np.percentile(latm, 99)), 3)}

    log("mixed precision")
    mixed = run_mixed(m.F32, args.steps, args.warmup, 100000)
    # BF16-stored values: one solve, capped at 3x the FP64 iteration count
    # (on this conditioning it stagnates; the record says so)
    mixed_bf16 = run_mixed(m.BF16, 1, 0, 3 * iters)

    cpu = None
    log("CPU baseline")
    if not args.no_cpu:
        cpu = cpu_baseline(rp, ci, va, b.numpy(), iters, args.cpu_iters, args.cpu_seconds)

    sections = (set(args.sections.split(",")) if args.sections != "all"
                else {"ic0", "c3", "solvers", "batched", "serving"})
    extra = {}
    if "ic0" in sections:
        extra["cg_ic0_160"] = guarded(lambda: pair_section(m, torch, A, b, bnorm, "ic_0", m.CG, x64))
    del S, P, P32
    if "c3" in sections:
        extra["c3"] = guarded(lambda: c3_section(m, torch, gen))
    if "solvers" in sections:
        extra["solvers"] = guarded(lambda: solvers_section(m, torch, gen))
    if "batched" in sections:
        extra["batched"] = guarded(lambda: batched_section(m, torch, gen, args.batch_systems))
    if "serving" in sections:
        extra["serving"] = guarded(lambda: serving_section(m, torch, gen, args.serve_requests,
                                                           big_rows=args.serve_big_rows))

    v = args.steps / t_fp64
    it_bytes = chip_bytes or by_layout + 11 * 8 * n
    mixed["speedup_vs_fp64"] = round(mixed["solves_per_s"] / v, 3)
    mixed_bf16["speedup_vs_fp64"] = round(mixed_bf16["solves_per_s"] / v, 3)
    mixed["recurrence"] = "cg + diagonal in FP32 on FP32 values, FP64 residual refresh at 0.1x"
    mixed_bf16["recurrence"] = "cg + diagonal in FP32 on BF16-stored values, FP64 refresh at 0.1x"
    out = {
        "metric": METRIC,
        "value": round(v, 4),
        "unit": "solves/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(1000.0 * t_fp64 / args.steps, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": {"workload": "itl::cg + pc::diagonal, FP64, rtol 1e-10, diffusion3d %d^3" % g,
                   "N": n, "nnz": nnz, "matrix": "7-point variable-coefficient diffusion, "
                   "kappa log-uniform [1e-2,1e2], seed 0", "rhs": "b = A*x_true, x_true~U[-1,1] seed 1"},
        "iterations": iters,
        "error_code": err,
        "relres": relres,
        "p50_ms": round(1000 * float(np.percentile(lat, 50)), 3),
        "p99_ms": round(1000 * float(np.percentile(lat, 99)), 3),
        "mixed": mixed,
        "mixed_bf16": mixed_bf16,
        "cg_iteration": {"operand": chip.operand, "us": round(1e6 * t_fp64 / args.steps / max(iters, 1), 2),
                         "bytes": it_bytes, "GBs": round(it_bytes * iters * args.steps / t_fp64 / 1e9, 1),
                         "frac": round(it_bytes * iters * args.steps / t_fp64 / 1e9 / HBM_PEAK_GBS, 4),
                         "note": "the bytes of roofline.bytes_per_iteration" if chip_bytes else
                                 "the layout's SpMV bytes + 11 vector passes (P: 4, XR: 7): the bytes of the "
                                 "launch-per-kernel loop; a solve kept on the chip moves fewer"},
        "spmv": {"diffusion3d_f64_GBs": round(ctx_gbs, 1), "diffusion3d_f64_back_to_back_GBs": round(spmv_gbs, 1),
                 "random_2M_poisson16_f64_GBs": round(rnd_gbs, 1),
                 "random_frac_of_peak": round(rnd_gbs / HBM_PEAK_GBS, 4)},
        "roofline": roofline,
        "cpu_baseline": cpu,
    }
    out.update(extra)
    print(json.dumps(out))


if __name__ == "__main__":
    main()
