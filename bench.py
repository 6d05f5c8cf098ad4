#!/usr/bin/env python
"""Benchmark of the BTA solver path on one MI355X.

Workload (default): the Gaussian spatio-temporal model with nt = 200 time
steps, ns = 2000 mesh nodes (50 x 40 grid, hx = 1/49, hy = 1/39), nb = 6 fixed
effects, dim(theta) = 4, m = 4 ns nt observations.  One step = one f(theta) +
grad f evaluation.  ``value`` is adjoint evaluations per second (forward:
assemble Q_c and Q_p, two FP64 BTA Cholesky factorizations, log-determinants,
one solve; backward: two selected inversions in place plus trace
contractions).  The finite-difference path (2 dim(theta) + 1 = 9 f
evaluations, 18 factorizations, as the reference's _objective_function) is
timed beside it.  All inputs are resident on the GPU before the timed region.

Prints one JSON line (rank 0, N = 1 only).
"""
from __future__ import annotations

import argparse
import json
from pathlib import Path
import os
import sys
import time

import numpy as np

ROOT = Path(__file__).resolve().parent
METRIC = "f(θ)+∇f evals/s, adjoint vs FD; pobtaf/pobtasi FP64 TFLOP/s vs peak"
PEAK_FP64_TFLOPS = 78.6
PEAK_HBM_GBS = 8000.0


def flops_potrf(n, b, a):
    """Algorithmic FLOPs of the BTA Cholesky (a = 0: BT variant)."""
    return (n * b**3 / 3 + (n - 1) * 2 * b**3 + n * (a * b**2 + a**2 * b)
            + (n - 1) * 2 * a * b**2 + a**3 / 3)


def flops_potrf_split(n, b, a):
    """(panel, update) parts of flops_potrf: the per-column panel kernel does
    the diagonal-block Cholesky and both TRSMs, the update kernel the SYRK /
    GEMM updates of the next block, arrow and tip."""
    panel = n * b**3 / 3 + (n - 1) * b**3 + n * a * b**2
    update = (n - 1) * b**3 + n * a**2 * b + (n - 1) * 2 * a * b**2
    return panel, update


def flops_potri(n, b, a):
    """Algorithmic FLOPs of the BTA selected inversion (lower-only Sigma_ii update)."""
    return n * (2 / 3) * b**3 + (n - 1) * 4 * b**3 + n * (7 * a * b**2 + 2 * a**2 * b) + a**3


def bytes_potrs(n, b, a):
    return 16 * (n * b**2 + (n - 1) * b**2 + n * a * b + a**2)


def class_kernel(cls, b, panel_launches, blocks):
    """Kernels whose launches a timing class holds; the panel variants are told
    apart by their launches for ``blocks`` blocks of edge ``b``."""
    if cls == 0:
        if panel_launches < blocks:
            return "k_chain64"
        return "k_panel_flow" if b > 64 and panel_launches == blocks else "k_panel_step"
    return {1: "k_gemm_nt_sub / k_gemm_grouped", 2: "k_gemm_direct / k_gemm_grouped",
            3: "k_sweep_solo" if b <= 64 else "k_sweep", 4: "rocblas_dgemm"}[cls]


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--nt", type=int, default=200)
    ap.add_argument("--nx", type=int, default=50)
    ap.add_argument("--ny", type=int, default=40)
    ap.add_argument("--nb", type=int, default=6)
    ap.add_argument("--fd-steps", type=int, default=1)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--cpu-nt", type=int, default=4, help="time steps of the bounded CPU sample")
    ap.add_argument("--graph", action="store_true", help="replay solver operations from hipGraphs")
    ap.add_argument("--selinv-blas", type=int, default=None, choices=[0, 1],
                    help="selected inversion: 1 = Sigma_{i+1,i} products through rocBLAS dgemm, 0 = every product "
                         "in the library's grouped kernel (default: the library's default)")
    ap.add_argument("--copy-calibration", type=int, default=0, metavar="MIB",
                    help="first run a plain device-to-device copy of MIB MiB (a known-size kernel to scale "
                         "rocprofv3 FETCH_SIZE / WRITE_SIZE counters against)")
    ap.add_argument("--skip-fd", action="store_true", help="skip the FD comparison (profiling runs)")
    ap.add_argument("--autotune", action="store_true",
                    help="tune the solvers' launch options on Q_prior / Q_cond first (pyinla_amd.autotune)")
    ap.add_argument("--workload", default="adjoint",
                    choices=["adjoint", "fd-batch", "mixed-batch", "coregional-lbfgs"],
                    help="adjoint: the headline line; the others measure the batched FD stencil, the "
                         "mixed-size batch and coregional L-BFGS (their own JSON lines)")
    ap.add_argument("--fd-wave", type=int, default=0, help="stencil points per batched FD wave (0 = all)")
    ap.add_argument("--batch-lanes", type=int, nargs="*", default=[],
                    help="mixed batch: also time these lane counts (problems run side by side)")
    ap.add_argument("--lbfgs-iters", type=int, default=20)
    ap.add_argument("--lbfgs-fd-iters", type=int, default=1)
    return ap.parse_args()


def _num(x):
    """JSON-safe number (None for NaN / inf)."""
    return None if x is None or not np.isfinite(x) else float(x)


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def cpu_baseline(args, prob_full):
    """Oracle (numpy/scipy BTA restatement + the reference's f and FD loop) on
    a bounded sample: the same mesh with cpu_nt time steps; the FD gradient
    cost is extrapolated linearly in nt to the full workload."""
    from oracle import model as om
    from pyinla_amd.coefficients import CoefficientModel
    from pyinla_amd.workloads import st_problem
    try:
        from threadpoolctl import threadpool_info
        threads = max([d.get("num_threads", 1) for d in threadpool_info()] or [1])
    except Exception:
        threads = os.cpu_count() or 1
    nts = args.cpu_nt
    prob = st_problem(nt=nts, nx=args.nx, ny=args.ny, nb=args.nb, seed=3,
                      hx=1.0 / (args.nx - 1), hy=1.0 / (args.ny - 1))
    cm = CoefficientModel("baseline")
    om.evaluate_f(prob, cm.table, prob.theta)  # warm-up
    times = []
    for _ in range(3):
        t0 = time.perf_counter()
        om.evaluate_f(prob, cm.table, prob.theta)
        times.append(time.perf_counter() - t0)
    t_f = float(np.median(times))
    d = 4
    t_grad_full = (2 * d + 1) * t_f * (args.nt / nts)
    try:
        nproc = len(os.sched_getaffinity(0))
    except Exception:
        nproc = os.cpu_count() or 1
    cpu_model = ""
    try:
        for line in Path("/proc/cpuinfo").read_text().splitlines():
            if line.startswith("model name"):
                cpu_model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    return {"value": 1.0 / t_grad_full, "unit": "evals/s", "cores": int(threads), "kind": "port",
            "host_cpus_nproc": int(nproc), "host_cpu_model": cpu_model,
            "sample": (f"oracle f(theta) (numpy/scipy BTA restatement, LAPACK/BLAS with {threads} threads) "
                       f"at nt={nts} on the same {args.nx}x{args.ny} mesh, median of 3 = {t_f:.3f} s; "
                       f"FD gradient = {2 * d + 1} f evaluations (reference order), extrapolated linearly "
                       f"in nt to nt={args.nt}"),
            "sample_f_seconds": t_f, "extrapolated_fd_grad_seconds": t_grad_full}


def bench_fd_batch(args, dev):
    """2 dim(theta) + 1 = 9 FD evaluations of the nt x ns model: sequential
    (the reference's loop) against all 18 factorizations in one batched graph."""
    import torch
    from pyinla_amd.st_model import STGaussianModel
    from pyinla_amd.workloads import st_problem
    prob = st_problem(nt=args.nt, nx=args.nx, ny=args.ny, nb=args.nb, seed=2)
    n, b, a = prob.nt, prob.ns, prob.nb
    model = STGaussianModel(prob, device=dev)
    th = prob.theta.copy()
    wave = args.fd_wave or None
    model.fd_gradient(th)
    model.fd_gradient_batched(th, wave=wave)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    f1, g1 = model.fd_gradient(th)
    torch.cuda.synchronize()
    t_seq = time.perf_counter() - t0
    t0 = time.perf_counter()
    f2, g2 = model.fd_gradient_batched(th, wave=wave)
    torch.cuda.synchronize()
    t_bat = time.perf_counter() - t0
    fl = 9 * (flops_potrf(n, b, a) + flops_potrf(n, b, 0))
    return {"metric": "FD f+grad (9 evaluations, 18 factorizations) wall time", "unit": "s",
            "config": {"workload": f"gaussian spatio-temporal FD stencil nt={n} ns={b} nb={a}", "wave": wave or 9},
            "sequential_s": t_seq, "batched_s": t_bat, "speedup": t_seq / t_bat,
            "batched_factorization_tflops_incl_solves": fl / t_bat / 1e12,
            "grad_max_rel_diff": float(np.abs(g1 - g2).max() / np.abs(g1).max()),
            "f_rel_diff": abs(f1 - f2) / abs(f1)}


def bench_mixed_batch(args, dev):
    """24 known-factor BTA matrices, nt in {50,100,200}, b in {256,...,2048}
    (seeded draw), a = 6: one batched graph against sequential factorizations."""
    import torch
    from pyinla_amd.batch import BatchedFactorization
    from pyinla_amd.solver import SerinvSolver
    from pyinla_amd.workloads import known_factor_bta_torch
    rng = np.random.default_rng(2)
    shapes = [(int(rng.choice([50, 100, 200])), int(rng.choice([256, 512, 1024, 2048]))) for _ in range(24)]
    a = 6
    solvers, Qs, total, ld_exact = [], [], 0.0, []
    for q, (n, b) in enumerate(shapes):
        # off-diagonal draws scaled to the block norms of the b = 92 construction
        # (unscaled, Q is numerically singular at these sizes)
        Lf, Q = known_factor_bta_torch(n, b, a, seed=100 + q, device=dev, norm_b=92)
        ld_exact.append(2.0 * (torch.log(torch.diagonal(Lf[0], dim1=1, dim2=2)).sum()
                               + torch.log(torch.diag(Lf[3])).sum()).item())
        del Lf
        s = SerinvSolver(None, b, n, a, device=dev, reserve="factor")
        Qs.append(Q)
        solvers.append(s)
        total += flops_potrf(n, b, a)

    def load_all():
        for s, Q in zip(solvers, Qs):
            s.load_blocks(*Q)
    batch = BatchedFactorization(solvers, ["bta"] * len(solvers))
    load_all()
    batch.factorize()
    for s in solvers:
        s.factorize("bta")
    torch.cuda.synchronize()
    load_all()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    batch.factorize()
    torch.cuda.synchronize()
    t_bat = time.perf_counter() - t0
    ld_b = [s.status()[1] for s in solvers]
    load_all()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for s in solvers:
        s.factorize("bta")
    torch.cuda.synchronize()
    t_seq = time.perf_counter() - t0
    ld_s = [s.status()[1] for s in solvers]
    lanes_s = {}
    for lanes in args.batch_lanes:
        solvers[0].set_batch_lanes(lanes)
        bl = BatchedFactorization(solvers, ["bta"] * len(solvers))
        load_all()
        bl.factorize()
        load_all()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        bl.factorize()
        torch.cuda.synchronize()
        lanes_s[str(lanes)] = time.perf_counter() - t0
        del bl
    solvers[0].set_batch_lanes(0)
    return {"metric": "mixed batch of 24 BTA factorizations", "unit": "TFLOP/s",
            "config": {"workload": "24 known-factor BTA matrices, nt in {50,100,200}, b in {256,512,1024,2048}, a=6",
                       "shapes": shapes},
            "batched_s": t_bat, "sequential_s": t_seq, "batched_tflops": total / t_bat / 1e12,
            "sequential_tflops": total / t_seq / 1e12, "batched_s_by_lanes": lanes_s,
            "max_logdet_rel_diff": max(abs(x - y) / abs(y) for x, y in zip(ld_b, ld_s)),
            "max_logdet_rel_err_vs_known_factor": max(abs(x - y) / abs(y) for x, y in zip(ld_b, ld_exact)),
            "construction": "config-0 known factor, off-diagonal draws scaled by sqrt(92/b)"}


def bench_coregional(args, dev):
    """Trivariate coregional model (3 x 1500 nodes interleaved, b = 4500,
    nt = 100, 9 fixed effects, dim theta = 15): L-BFGS-B with the adjoint
    gradient; the FD (31 evaluations) run is timed for a few iterations."""
    import torch
    from pyinla_amd.optimize import minimize
    from pyinla_amd.st_model import STGaussianModel
    from pyinla_amd.workloads import coregional_problem
    prob = coregional_problem(nv=3, nt=args.nt, nx=50, ny=30, nb_per=3, obs_per_node=2, seed=4)
    model = STGaussianModel(prob, device=dev)
    th0 = prob.theta.copy()
    model.value_and_grad(th0)
    torch.cuda.synchronize()
    log(f"coregional model resident: n={prob.nt} b={model.b} a={model.a}")
    r_adj = minimize(model, th0, gradient="adjoint", max_iter=args.lbfgs_iters, verbose=True)
    torch.cuda.synchronize()
    r_fd = minimize(model, th0, gradient="fd", max_iter=args.lbfgs_fd_iters, verbose=True)
    torch.cuda.synchronize()
    r_fdb = minimize(model, th0, gradient="fd_batched", max_iter=args.lbfgs_fd_iters, verbose=True,
                     fd_wave=args.fd_wave if args.fd_wave > 0 else None)
    torch.cuda.synchronize()
    fd_wave = len(model._fd_pool[0]) if getattr(model, "_fd_pool", None) else 0

    def summary(r):
        it = max(r["iterations"], 1)
        return {"iterations": r["iterations"], "objective_calls": r["objective_calls"], "wall_s": r["wall_time"],
                "s_per_iter": r["wall_time"] / it, "s_per_objective_call": float(np.mean(r["objective_time"])),
                "f": r["f"], "message": r["message"]}

    adj, fd, fdb = summary(r_adj), summary(r_fd), summary(r_fdb)
    fdb["wave"] = fd_wave
    return {"metric": "coregional L-BFGS wall time per iteration", "unit": "s",
            "config": {"workload": f"coregional nv=3 ns=1500 nt={args.nt} b=4500 nb=9 dim_theta=15"},
            "adjoint": adj, "fd": fd, "fd_batched": fdb,
            "fd_over_adjoint_per_objective_call": fd["s_per_objective_call"] / adj["s_per_objective_call"],
            "fd_batched_over_adjoint_per_objective_call":
                fdb["s_per_objective_call"] / adj["s_per_objective_call"]}


def main():
    args = parse()
    if args.gpus != 1:
        print(f"bench.py measures one GPU only (asked for --gpus {args.gpus}); this build has no "
              "multi-GPU path. Run with --gpus 1.", file=sys.stderr)
        sys.exit(2)
    import torch
    from pyinla_amd import _lib
    from pyinla_amd.st_model import STGaussianModel
    from pyinla_amd.workloads import st_problem

    assert torch.cuda.is_available(), "bench.py needs a GPU"
    dev = torch.device("cuda", 0)
    lib = _lib.load()
    if args.workload != "adjoint":
        fn = {"fd-batch": bench_fd_batch, "mixed-batch": bench_mixed_batch,
              "coregional-lbfgs": bench_coregional}[args.workload]
        print(json.dumps(fn(args, dev)), flush=True)
        return
    if args.copy_calibration:
        nel = args.copy_calibration * (1 << 20) // 8
        src = torch.ones(nel, dtype=torch.float64, device=dev)
        dst = torch.empty_like(src)
        dst.copy_(src)
        torch.cuda.synchronize()
        log(f"copy calibration: {args.copy_calibration} MiB read + written")
        del src, dst
    t0 = time.perf_counter()
    prob = st_problem(nt=args.nt, nx=args.nx, ny=args.ny, nb=args.nb, seed=3,
                      hx=1.0 / (args.nx - 1), hy=1.0 / (args.ny - 1))
    n, b, a = prob.nt, prob.ns, prob.nb
    log(f"problem nt={n} ns={b} nb={a} m={prob.A.shape[0]} built in {time.perf_counter() - t0:.1f}s")
    model = STGaussianModel(prob, device=dev, use_graph=args.graph)
    if args.selinv_blas is not None:
        for s_ in (model.cond, model.prior):
            s_.set_selinv_blas(bool(args.selinv_blas))
    theta = prob.theta.copy()
    log("model resident on GPU")
    tuned = None
    if args.autotune:
        t0 = time.perf_counter()
        tuned = model.autotune(theta)
        tuned = {k: {n: v for n, v in c.items() if n != "times_ms"} for k, c in tuned.items()}
        log(f"autotuned in {time.perf_counter() - t0:.1f}s: {tuned}")

    for w in range(args.warmup):
        f0, g_adj = model.value_and_grad(theta)
        torch.cuda.synchronize()
        log(f"warmup {w}: f={f0:.10e}")

    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        f_adj, g_adj = model.value_and_grad(theta)
    torch.cuda.synchronize()
    t_adj = (time.perf_counter() - t0) / args.steps
    log(f"adjoint f+grad: {t_adj * 1e3:.1f} ms/step")

    # plain GPU FD path (9 f evaluations, reference order), step 1e-3
    t_fd, grad_rel = float("nan"), float("nan")
    grad_rel4, t_fdb, fd_wave = float("nan"), float("nan"), 0
    if not args.skip_fd:
        f_fd, g_fd = model.fd_gradient(theta, eps=1e-3)  # warm
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(args.fd_steps):
            f_fd, g_fd = model.fd_gradient(theta, eps=1e-3)
        torch.cuda.synchronize()
        t_fd = (time.perf_counter() - t0) / args.fd_steps
        log(f"FD f+grad: {t_fd * 1e3:.1f} ms/step")
        grad_rel = float(np.abs(g_adj - g_fd).max() / max(np.abs(g_fd).max(), 1e-300))
        # the same 2 d + 1 = 9-point central FD with step 1e-4 (the gradient check)
        f_fd4, g_fd4 = model.fd_gradient(theta, eps=1e-4)
        grad_rel4 = float(np.abs(g_adj - g_fd4).max() / max(np.abs(g_fd4).max(), 1e-300))
        log(f"adjoint vs 9-point FD (step 1e-4): rel {grad_rel4:.2e}")
        # batched FD: the 18 factorizations in batched, graph-replayed waves
        wave = args.fd_wave if args.fd_wave > 0 else None
        model.fd_gradient_batched(theta, eps=1e-3, wave=wave)  # pool + graph set-up
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        f_fdb, g_fdb = model.fd_gradient_batched(theta, eps=1e-3, wave=wave)
        torch.cuda.synchronize()
        t_fdb = time.perf_counter() - t0
        fd_wave = len(model._fd_pool[0])
        model._fd_pool = None  # release the pool before the remaining measurements
        torch.cuda.empty_cache()
        log(f"batched FD f+grad: {t_fdb * 1e3:.1f} ms/step (waves of {fd_wave} stencil points)")

    # live per-kernel-class timing (HIP events on the launch stream) of one
    # adjoint evaluation
    classes = {0: "panel", 1: "update", 2: "grouped", 3: "gemv", 4: "blas"}
    tot = {c: 0.0 for c in classes}
    cnt = {c: 0 for c in classes}
    import ctypes as C
    for s in (model.cond, model.prior):
        _lib.check(lib.bta_ws_set_timing(s._ws, 1), "set_timing")
    model.value_and_grad(theta)
    torch.cuda.synchronize()
    for s in (model.cond, model.prior):
        for c in classes:
            ms = C.c_double()
            k = C.c_int64()
            _lib.check(lib.bta_ws_get_timing(s._ws, c, C.byref(ms), C.byref(k)), "get_timing")
            tot[c] += ms.value
            cnt[c] += k.value
        _lib.check(lib.bta_ws_set_timing(s._ws, 0), "set_timing")
    fp_c, fu_c = flops_potrf_split(n, b, a)
    fp_p, fu_p = flops_potrf_split(n, b, 0)
    flow = cnt[1] == 0  # persistent panel launches carry the block updates too
    if flow:
        flops_cls = {0: flops_potrf(n, b, a) + flops_potrf(n, b, 0), 1: 0.0}
    else:
        flops_cls = {0: fp_c + fp_p, 1: fu_c + fu_p}
    # the rocBLAS dgemm calls (class 4) are the Sigma_{i+1,i} products, 2 b^3 each
    flops_cls[4] = cnt[4] * 2.0 * b**3
    flops_cls[2] = flops_potri(n, b, a) + flops_potri(n, b, 0) - flops_cls[4]
    potrf_ms = tot[0] + tot[1]
    potrf_tflops = (flops_potrf(n, b, a) + flops_potrf(n, b, 0)) / (potrf_ms * 1e-3) / 1e12 if potrf_ms else None
    potri_ms = tot[2] + tot[4]
    potri_tflops = (flops_cls[2] + flops_cls[4]) / (potri_ms * 1e-3) / 1e12 if potri_ms else None
    dom = max(classes, key=lambda c: tot[c])
    if dom == 3:
        ach = bytes_potrs(n, b, a) / (tot[3] * 1e-3 / max(cnt[3], 1) * cnt[3]) / 1e9
        roof = {"bound": "hbm", "achieved": ach, "peak": PEAK_HBM_GBS, "unit": "GB/s", "frac": ach / PEAK_HBM_GBS,
                "traffic": None}
    else:
        per_launch_flops = flops_cls[dom] / max(cnt[dom], 1)
        avg_ms = tot[dom] / max(cnt[dom], 1)
        ach = per_launch_flops / (avg_ms * 1e-3) / 1e12
        roof = {"bound": "mfma", "achieved": ach, "peak": PEAK_FP64_TFLOPS, "unit": "TFLOP/s",
                "frac": ach / PEAK_FP64_TFLOPS, "traffic": None}
    roof["kernel"] = class_kernel(dom, b, cnt[0], 2 * n)
    # HBM bytes per launch from the committed rocprofv3 PMC summary (FETCH_SIZE /
    # WRITE_SIZE, scaled by a 1 GiB copy), where the class is one kernel in it
    tr_path = ROOT / "profiles" / "pmc_traffic.json"
    if tr_path.exists():
        try:
            tr = json.loads(tr_path.read_text())
            k = tr.get("kernels", {}).get("bta::" + roof["kernel"])
            if k:
                roof["traffic"] = k["traffic_bytes"]
                roof["traffic_source"] = f"profiles/pmc_traffic.json ({tr.get('workload', '')})"
        except (ValueError, KeyError):
            pass
    roof["launches"] = cnt[dom]
    roof["avg_launch_ms"] = tot[dom] / max(cnt[dom], 1)
    if roof["kernel"] == "k_panel_flow":
        # the two matrices' panel launches run side by side on two streams, so
        # the per-launch rate above is half the device's: also time the pair
        # of factorizations by wall clock
        pair = []
        for _ in range(2):
            model.assemble_prior(theta)
            model.assemble_cond(theta)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            cur = model._fork()
            with torch.cuda.stream(model.s_prior):
                model.prior.factorize("bt")
            with torch.cuda.stream(model.s_cond):
                model.cond.factorize("bta")
            model._join(cur)
            torch.cuda.synchronize()
            pair.append(time.perf_counter() - t0)
        t_pair = min(pair)
        dev = (flops_potrf(n, b, a) + flops_potrf(n, b, 0)) / t_pair / 1e12
        roof["concurrent_launches"] = 2
        roof["pair_wall_ms"] = t_pair * 1e3
        roof["device_achieved"] = dev
        roof["device_frac"] = dev / PEAK_FP64_TFLOPS
    breakdown = {classes[c]: {"ms": tot[c], "launches": cnt[c]} for c in classes}

    cpu = None
    if not args.no_cpu:
        log("CPU baseline (bounded sample)")
        cpu = cpu_baseline(args, prob)

    out = {
        "metric": METRIC,
        "value": 1.0 / t_adj,
        "unit": "evals/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": t_adj * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": {"workload": f"gaussian spatio-temporal f+grad (adjoint), nt={n}, ns={b} "
                               f"({args.nx}x{args.ny} grid), nb={a}, dim_theta=4",
                   "nt": n, "ns": b, "nb": a, "dim_theta": 4, "observations": int(prob.A.shape[0])},
        "fd": {"value": _num(1.0 / t_fd), "unit": "evals/s", "ms_per_step": _num(t_fd * 1e3),
               "adjoint_speedup": _num(t_fd / t_adj), "grad_rel_diff_adjoint_vs_fd1e-3": _num(grad_rel),
               "grad_rel_diff_adjoint_vs_fd9pt_step1e-4": _num(grad_rel4),
               "batched_ms_per_step": _num(t_fdb * 1e3), "batched_wave": fd_wave,
               "adjoint_speedup_vs_batched": _num(t_fdb / t_adj)},
        "pobtaf_tflops": potrf_tflops,
        "pobtaf_frac_peak": potrf_tflops / PEAK_FP64_TFLOPS if potrf_tflops else None,
        "pobtasi_tflops": potri_tflops,
        "pobtasi_frac_peak": potri_tflops / PEAK_FP64_TFLOPS if potri_tflops else None,
        "kernel_ms": breakdown,
        "roofline": roof,
        "cpu_baseline": cpu,
        "autotuned": tuned,
        "f": f_adj,
    }
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
