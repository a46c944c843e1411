"""Benchmark: batched mixed-precision Beyn CFIE-Kress windows on one MI355X.

Workload (default): star billiard r = 1 + 0.2 cos(5 t), CFIE-Kress, N = 8192,
one Beyn window k0 = 800, R = 0.5, 48 contour nodes, seeded complex Gaussian
probes starting at 64 and doubled until the rank of A0 no longer saturates
(the disk holds ~400 levels, more than 64 probes can resolve; the grown r is
fixed in warmup and reported).  Two full-accuracy paths run the same
windows: the complex128 path, and complex64 LU on MFMA + FP64 iterative
refinement to refine_tol; `value` is the faster one's (config.path), the
other's figures sit beside it (paths, mixed_vs_fp64).  --inflight n keeps n
windows in flight on separate device contexts.

A step is one full window: contour nodes -> tables -> assembly of all 48
T(z_j) -> LU of all nodes -> moment solves -> thin SVD, rank, B, eig(B).
Eigenvalues counted: the real roots inside the disk (|lambda - k0| <= R,
|Im lambda| <= 1e-8 |lambda|) that match a real root of the complex128 path
within 1e-10 relative.  On the warmup window the reference's residual filter
(imag_k_check_EXPERIMENTAL with every candidate examined) is run once and
its kept set is reported beside the real-root set; the two are the same at
this workload (tests/test_gpu_configs.py).
"""
import argparse
import json
import math
import os
import sys
import threading
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path[:0] = [ROOT, os.path.join(ROOT, "quantumbilliards.jl_amd")]

import numpy as np  # noqa: E402

PEAK = {"c64": 157.3, "c128": 78.6, "i8": 5000.0}  # dense MFMA TFLOP/s (fp32, fp64), int8 TOPS
# HBM bytes per GEMM launch over the windows of the default workload, from
# FETCH_SIZE / WRITE_SIZE counter runs scaled by a copy kernel of known size
# (profiles/beyn_window_star_N8192_pmc_traffic.txt)
TRAFFIC_PER_LAUNCH = {"c128": 560.6e6, "c64": 515.8e6}


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--N", type=int, default=8192)
    ap.add_argument("--nq", type=int, default=48)
    ap.add_argument("--k0", type=float, default=800.0)
    ap.add_argument("--R", type=float, default=0.5)
    ap.add_argument("--r0", type=int, default=64)
    ap.add_argument("--r", type=int, default=0, help="fix the probe count (skip growth)")
    ap.add_argument("--svd-tol", type=float, default=1e-10)
    ap.add_argument("--cheb-tol", type=float, default=1e-12)
    ap.add_argument("--refine-tol", type=float, default=1e-12)
    ap.add_argument("--no-fp64", action="store_true", help="time the mixed path only")
    ap.add_argument("--no-mixed", action="store_true", help="time the complex128 path only")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-filter-check", action="store_true",
                    help="skip the residual filter run on the warmup window")
    ap.add_argument("--inflight", type=int, default=1,
                    help="mixed windows in flight at once, each on its own device context")
    ap.add_argument("--cpu-cols", type=int, default=512)
    ap.add_argument("--serve", action="store_true",
                    help="serving stream (Poisson arrivals of mixed windows) instead")
    ap.add_argument("--serve-requests", type=int, default=24)
    ap.add_argument("--serve-rate", type=float, default=1.0, help="arrivals per second")
    ap.add_argument("--serve-kmax", type=float, default=1000.0)
    ap.add_argument("--serve-slots", type=int, default=2)
    ap.add_argument("--serve-precision", default="fp64", choices=["fp64", "mixed"])
    ap.add_argument("--serve-irreps-separate", dest="serve_irreps_batched",
                    action="store_false",
                    help="with --serve-symmetry: one job per irrep instead of one window")
    ap.add_argument("--serve-symmetry", action="store_true",
                    help="serve each request as the symmetry-reduced windows of its shape")
    ap.add_argument("--symmetry", action="store_true",
                    help="the same disk on the C_5-reduced star: one window per irrep "
                         "(Rotation(5, m), m = 0..4), eigenvalues checked against the "
                         "unreduced FP64 window")
    ap.add_argument("--sym-precision", default="fp64")
    ap.add_argument("--sym-slots", type=int, default=2,
                    help="contexts that take irrep windows concurrently (--no-sym-batched)")
    ap.add_argument("--no-sym-batched", dest="sym_batched", action="store_false",
                    help="one window per irrep instead of one window over all irreps")
    ap.add_argument("--assembly", action="store_true",
                    help="assembly throughput: DLP-Kress on the ellipse (1, 0.6), N = 4096, "
                         "64 nodes at k0 = 400, and CFIE-Kress on the star, N = 8192, 48 nodes")
    ap.add_argument("--uneven", action="store_true",
                    help="uneven batched windows: the disk with a hole, k0 uniform in "
                         "[100, 800], N from 10 points per wavelength rounded up to 256")
    ap.add_argument("--uneven-windows", type=int, default=128)
    ap.add_argument("--uneven-kmax", type=float, default=800.0)
    ap.add_argument("--uneven-precision", default="fp64",
                    help="fp64 (default: faster on this workload) or mixed")
    ap.add_argument("--tune-n", type=int, default=0, metavar="N",
                    help="serving and uneven runs: time the GEMM tiles of each slot for the shape "
                         "classes of an N-point window at warm-up (0: untuned defaults)")
    ap.add_argument("--uneven-slots", type=int, default=2)
    ap.add_argument("--uneven-max-group", type=int, default=16)
    ap.add_argument("--group", action="store_true",
                    help="batch windows that share N into one window (qb_window_create_multi)")
    ap.add_argument("--graphs", action="store_true",
                    help="replay each window's LU from a captured hipGraph (qb_ctx_set_graphs; "
                         "only without the per-launch events, so with --no-kernel-stats)")
    ap.add_argument("--no-kernel-stats", action="store_true",
                    help="time without the library's per-launch HIP events (no roofline fields)")
    ap.add_argument("--copy-ref", type=int, default=0, metavar="MIB",
                    help="first run a plain device copy of MIB MiB (read once, written once): "
                         "the calibration of HBM byte counters in rocprofv3 --pmc runs")
    return ap.parse_args()


def copy_ref(mib: int):
    """A plain device copy of a known size (an elementwise kernel that reads
    `mib` MiB and writes `mib` MiB, launched twice), run before the workload
    so a FETCH_SIZE / WRITE_SIZE counter run holds its own calibration."""
    import torch
    n = (mib << 20) // 4
    src = torch.ones(n, dtype=torch.float32, device="cuda:0")
    dst = torch.empty_like(src)
    for _ in range(2):
        torch.neg(src, out=dst)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    torch.neg(src, out=dst)
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    print(f"# copy reference: {mib} MiB read + {mib} MiB written, {2 * n * 4 / dt / 1e9:.0f} GB/s",
          file=sys.stderr, flush=True)
    del src, dst
    torch.cuda.empty_cache()


def run_serve(a):
    """Serving workload: a seeded Poisson stream of window requests mixing the
    ellipse (1, 0.6), the stadium (radius 1, half-length 1) and the star,
    k0 log-uniform in [50, kmax], R in [0.25, 0.5], tol 1e-8 or 1e-12, N from
    10 points per wavelength, 32 contour nodes, mixed precision; admission by
    HBM footprint into `slots` device contexts.  Untimed warmup windows first
    (one per slot, then one of the stream's kind).  Prints one JSON line with eigenvalues/s and p50/p99 latency."""
    from qbhip import serve as S
    reqs = S.poisson_stream(a.serve_requests, rate=a.serve_rate, seed=5, kmax=a.serve_kmax,
                            symmetry=a.serve_symmetry, precision=a.serve_precision)
    srv = S.Server(slots=a.serve_slots, irreps_batched=a.serve_irreps_batched)
    srv.warm_up(tune_N=a.tune_n, precisions=(a.serve_precision,))
    srv.submit(S.WindowRequest(-1, "ellipse", 60.0, 0.3, tol=1e-8, nq=32,
                               symmetry=a.serve_symmetry)).result()
    t0 = time.perf_counter()
    res = srv.run_stream(reqs)
    span = time.perf_counter() - t0
    srv.close()
    summ = S.summarize(res)
    Ns = [r.N for r in res]
    print(json.dumps({
        "metric": "serving: eigenvalues/sec + p50/p99 window latency (Poisson stream of Beyn windows)",
        "value": summ["eigenvalues_per_s"], "unit": "eigenvalues/s", "n_gpus": 1,
        "p50_window_s": summ["p50_latency_s"], "p99_window_s": summ["p99_latency_s"],
        "windows": summ["windows"], "eigenvalues": summ["eigenvalues"],
        "candidates_in_disks": summ["candidates"],
        "counted": "real roots inside each disk (|Im k| <= 1e-8 |k|)", "span_s": span,
        "higher_is_better": True,
        "dtype": "c64+c128-refine" if a.serve_precision == "mixed" else "c128",
        "data": "synthetic (seeded)",
        "config": {"workload": "serving stream ellipse/stadium/star", "requests": len(reqs),
                   "rate_per_s": a.serve_rate, "k0": [50.0, a.serve_kmax], "nq": 32,
                   "slots": a.serve_slots, "N_min": min(Ns), "N_max": max(Ns),
                   "symmetry_reduced": a.serve_symmetry,
                   "irreps_in_one_window": a.serve_symmetry and a.serve_irreps_batched}}),
          flush=True)


def run_assembly(a):
    """Assembly throughput (K1/K2), the device assembly of T(z_j) at every
    contour node of a window, timed by the library's HIP events on its own
    stream over `--steps` windows (FP64, so only the complex128 matrices are
    written):
      DLP-Kress, full ellipse (1, 0.6), N = 4096, 64 nodes 400 + 0.5 e^{i theta};
      CFIE-Kress, star r = 1 + 0.2 cos 5t, N = 8192, 48 nodes 800 + 0.5 e^{i theta};
    tables tuned to 1e-12 on the device (chebyshev_params; the windows'
    conjugate-pair kernel reads its own envelope tables instead, see
    k_assemble_env).  Algorithmic bytes: 16 per entry written; FP64 flops per
    entry: 3(M_h+M_j)+22 (DLP), 6(M_h+M_j)+50 (CFIE), the reference's count
    for its table route.  Prints one JSON line per operator."""
    import qbhip as q
    cases = [("DLP_kress", q.make_full_ellipse(1.0, 0.6), 4096, 64, 400.0),
             ("CFIE_kress", q.make_star_polar_boundary(1.0, 0.2, 5), 8192, 48, 800.0)]
    for name, b, N, nq, k0 in cases:
        ctx = q.Context(0)
        solver = (q.DLP_kress if name == "DLP_kress" else q.CFIE_kress)(10.0, b)
        pts = q.evaluate_points(solver, b, k0, N=[N])
        geom = q.Geometry(pts, ctx, solver)
        zj = k0 + 0.5 * np.exp(2j * np.pi * np.arange(nq) / nq)
        nh, mh, nj, mj, _ = q.chebyshev_params(solver, pts, zj, tol=1e-12, geom=geom)
        cheb = dict(n_panels_h=nh, M_h=mh, n_panels_j=nj, M_j=mj)
        q.Window(solver, pts, k0, 0.5, nq, precision="fp64", geom=geom, **cheb).close()
        ctx.set_profiling(True)
        for _ in range(a.steps):
            q.Window(solver, pts, k0, 0.5, nq, precision="fp64", geom=geom, **cheb).close()
        ks = ctx.kernel_stats()
        ctx.set_profiling(False)
        asm = ks["assemble"]
        t = asm["ms"] / max(asm["launches"], 1) * 1e-3
        ent = float(N) * N * nq
        flops_per = (3 * (mh + mj) + 22) if name == "DLP_kress" else (6 * (mh + mj) + 50)
        gbs = ent * 16 / t / 1e9
        print(json.dumps({
            "metric": f"{name} assembly throughput (GB/s written, complex128 T(z_j))",
            "value": gbs, "unit": "GB/s", "n_gpus": 1, "steps": a.steps,
            "ms_per_launch": t * 1e3, "entries_per_s": ent / t,
            "fp64_tflops": ent * flops_per / t / 1e12, "higher_is_better": True,
            "dtype": "c128", "data": "synthetic (geometry nodes)",
            "config": {"workload": name, "N": N, "nq": nq, "k0": k0, "R": 0.5, "cheb": cheb,
                       "cheb_tol": 1e-12},
            "roofline": {"kernel": ("k_assemble_conj (uniform tables)"
                                    if os.environ.get("QB_ASM_TABLES") else
                                    "k_assemble_env (envelope tables in LDS)"),
                         "bound": "hbm", "achieved": gbs, "peak": 8000.0,
                         "unit": "GB/s", "frac": gbs / 8000.0,
                         "fp64_frac": ent * flops_per / t / 1e12 / 78.6}}), flush=True)
        geom.close()
        ctx.close()


def run_uneven(a):
    """Uneven batched windows: `--uneven-windows` disks (R = 0.5, 32 contour
    nodes) on the unit disk with a hole of radius 0.3 at (0.35, 0), k0 seeded
    uniform in [100, 800], N = 10 k L / 2 pi rounded up to a multiple of 256
    (1536 ... 10496, outer : hole = 10 : 3), all submitted at once to the
    serving loop: windows run side by side in `--uneven-slots` contexts,
    admitted by HBM footprint; with `--group`, windows that share N are
    batched into one window (one assembly, one batched LU and solve over all
    their contour nodes).  Counted: the real roots inside each disk.  One
    untimed warmup window first.  Prints one JSON line."""
    from qbhip import serve as S
    reqs = S.uneven_windows(a.uneven_windows, seed=4, precision=a.uneven_precision,
                            kmax=a.uneven_kmax)
    srv = S.Server(slots=a.uneven_slots, group=a.group, max_group=a.uneven_max_group)
    srv.warm_up(tune_N=a.tune_n, precisions=(a.uneven_precision,))
    srv.submit(S.WindowRequest(-1, "circle_hole", 100.0, 0.5, nq=32,
                               precision=a.uneven_precision,
                               N=S.hole_node_counts(100.5))).result()
    t0 = time.perf_counter()
    done = [0]
    lock = threading.Lock()

    def progress(f):
        with lock:
            done[0] += 1
            if done[0] % 8 == 0 or done[0] == len(reqs):
                print(f"[uneven] {done[0]}/{len(reqs)} windows done at "
                      f"{time.perf_counter() - t0:.1f} s", file=sys.stderr, flush=True)

    futs = []
    for rq in reqs:  # all arrive at once
        f = srv.submit(rq, t0)
        f.add_done_callback(progress)
        futs.append(f)
    res = []
    for f in futs:
        try:
            res.append(f.result())
        except Exception as e:  # noqa: BLE001 - reported per window
            res.append(e)
    span = time.perf_counter() - t0
    srv.close()
    summ = S.summarize(res, t_span=span)
    ok = [r for r in res if isinstance(r, S.WindowResult)]
    Ns = sorted({r.N for r in ok})
    groups = [r.stats.get("group", 1) for r in ok]
    print(json.dumps({
        "metric": "uneven batched windows: eigenvalues/sec (Beyn CFIE-Kress, N 1536-10496)",
        "value": summ["eigenvalues_per_s"], "unit": "eigenvalues/s", "n_gpus": 1,
        "windows": summ["windows"], "rejected": summ["rejected"],
        "eigenvalues": summ["eigenvalues"], "candidates_in_disks": summ["candidates"],
        "counted": "real roots inside each disk (|Im k| <= 1e-8 |k|)", "span_s": span,
        "p50_window_s": summ["p50_latency_s"], "p99_window_s": summ["p99_latency_s"],
        "N_classes": len(Ns), "mean_group": float(np.mean(groups)) if groups else None,
        "higher_is_better": True,
        "dtype": "c64+c128-refine" if a.uneven_precision == "mixed" else "c128",
        "data": "synthetic (seeded)",
        "config": {"workload": "circle with hole (0.3 at (0.35, 0)), k0 ~ U[100, %g], R=0.5"
                               % a.uneven_kmax,
                   "windows": len(reqs), "nq": 32, "N_min": min(Ns), "N_max": max(Ns),
                   "slots": a.uneven_slots, "grouped": a.group,
                   "max_group": a.uneven_max_group}}), flush=True)


def run_symmetry(a):
    """Symmetry-reduced windows (_all_k_symm_CFIE_chebyshev!, cheb-CFIE:698-824,
    as the reference's examples run the star, example_beyn_kress.jl:51): the
    disk |k - k0| <= R of star(1, 0.2, 5) with N nodes (a multiple of 10) as
    five reduced problems of N/5 unknowns, one per C_5 irrep.  By default a
    pass is one window on a multi-irrep geometry (one assembly pass for all
    irreps, one batched LU of 5 x nq matrices), its moments reduced on the
    device (qb_window_moments_qr), and the host stage (B and eig(B) per irrep)
    of pass s overlaps pass s+1 on the device.  With --no-sym-batched the five
    irrep windows are independent and `--sym-slots` contexts (one HIP stream
    pair and one host thread each) take them from a queue.  Prints one JSON
    line: eigenvalues/s over all irreps, per-window latencies, and the match
    of the union of the irrep spectra against the unreduced FP64 window."""
    import queue
    import threading
    import qbhip as q
    b = q.make_star_polar_boundary(1.0, 0.2, 5)
    N = a.N + (-a.N) % 10
    full = q.CFIE_kress(10.0, b)
    pts = q.evaluate_points(full, b, a.k0, N=[N])
    ctxs = [q.default_context()] + [q.Context(0) for _ in range(max(1, a.sym_slots) - 1)]
    gfull = q.Geometry(pts, ctxs[0])
    zj = a.k0 + a.R * np.exp(2j * np.pi * np.arange(a.nq) / a.nq)
    nh, mh, nj, mj, errs = q.chebyshev_params(full, pts, zj, tol=a.cheb_tol, geom=gfull)
    cheb = dict(n_panels_h=nh, M_h=mh, n_panels_j=nj, M_j=mj)
    solvers = [q.CFIE_kress(10.0, b, symmetry=q.Rotation(5, m)) for m in range(5)]
    geoms = [[q.Geometry(pts, c, s) for s in solvers] for c in ctxs]
    m_dim = geoms[0][0].dim
    bf = q.make_star_polar_boundary(1.0, 0.2, 5)
    bf.area = b.area / 5  # probes from the Weyl count of one sector
    bf.length = b.length / 5
    r_irrep = a.r or q.probe_count(bf, a.k0, a.R, a.nq, a.svd_tol, 32)
    V = q.probe_block(np.random.default_rng(1), m_dim, r_irrep, pinned=True)
    if a.sym_batched:
        # one window over all five irreps: a single assembly evaluates every
        # image term once for all characters, one LU factors 5 x nq matrices
        ctxs = ctxs[:1]
        gmulti = q.Geometry(pts, ctxs[0], irreps=solvers)
        rep = ctxs[0].autotune(m_dim, a.nq * 5, r_irrep, a.sym_precision)
    else:
        for c in ctxs:
            rep = c.autotune(m_dim, a.nq, r_irrep, a.sym_precision)
    print("# gemm autotune:\n" + rep, file=sys.stderr, flush=True)

    def batched_pass():
        t0 = time.perf_counter()
        ts = time.perf_counter()
        win = q.Window(solvers[0], pts, complex(a.k0), a.R, a.nq, precision=a.sym_precision,
                       geom=gmulti, ctx=ctxs[0], **cheb)
        Rm, Cm = win.moments_qr(V, a.refine_tol)
        win.close()
        t_dev = time.perf_counter() - ts
        res = []
        for m in range(5):
            B, Ur, S, rk = q.B_from_qr(Rm[m], Cm[m], a.svd_tol)
            lam = np.linalg.eigvals(B) if B.size else np.zeros(0, complex)
            res.append((lam, rk, t_dev))
        return res, time.perf_counter() - t0

    def one_pass():
        if a.sym_batched:
            return batched_pass()
        """All five irrep windows; returns per-irrep (lam, rk, latency) and the
        span from the first window's start to the last result."""
        work = queue.Queue()
        for m in range(5):
            work.put(m)
        res = [None] * 5
        t0 = time.perf_counter()

        def worker(ci):
            c = ctxs[ci]
            while True:
                try:
                    m = work.get_nowait()
                except queue.Empty:
                    return
                ts = time.perf_counter()
                win = q.Window(solvers[m], pts, complex(a.k0), a.R, a.nq,
                               precision=a.sym_precision, geom=geoms[ci][m], ctx=c, **cheb)
                Rm, Cm = win.moments_qr(V, a.refine_tol)
                win.close()
                B, Ur, S, rk = q.B_from_qr(Rm, Cm, a.svd_tol)
                lam = np.linalg.eigvals(B) if B.size else np.zeros(0, complex)
                res[m] = (lam, rk, time.perf_counter() - ts)

        th = [threading.Thread(target=worker, args=(i,)) for i in range(len(ctxs))]
        for t in th:
            t.start()
        for t in th:
            t.join()
        return res, time.perf_counter() - t0

    # a pass is ~0.2 s: at least 4 untimed passes (in a process started after
    # another one on the same device, the first passes run slower)
    for w in range(max(4, a.warmup)):
        res, sp = one_pass()
        print(f"# warmup {w}: {sp:.3f}s rk={[x[1] for x in res]}", file=sys.stderr, flush=True)
    for c in ctxs:
        c.set_profiling(True)
    spans, last = [], None
    host_s, dev_s = [], []
    if a.sym_batched:
        # pipelined like the main bench: the host stage (SVD of R, B, eig per
        # irrep) of pass s runs on a host thread while pass s+1 is on the device
        qu = queue.Queue()
        done = [None] * a.steps
        host_s, dev_s = [], []

        def host_stage():
            ncpu = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else 4
            try:  # small problems (r x r, r = 192): a few LAPACK threads
                from threadpoolctl import threadpool_limits
                lim = threadpool_limits(limits=max(1, min(4, ncpu - 2)), user_api="blas")
            except Exception:
                lim = None
            while True:
                item = qu.get()
                if item is None:
                    if lim is not None:
                        lim.restore_original_limits()
                    return
                s_, Rm, Cm, t_dev = item
                th = time.perf_counter()
                res = []
                for m in range(5):
                    B, Ur, S, rk = q.B_from_qr(Rm[m], Cm[m], a.svd_tol)
                    lam = np.linalg.eigvals(B) if B.size else np.zeros(0, complex)
                    res.append((lam, rk, t_dev))
                done[s_] = (res, time.perf_counter())
                host_s.append(done[s_][1] - th)
                dev_s.append(t_dev)

        hth = threading.Thread(target=host_stage)
        hth.start()
        t_begin = time.perf_counter()
        for s in range(a.steps):
            ts = time.perf_counter()
            win = q.Window(solvers[0], pts, complex(a.k0), a.R, a.nq,
                           precision=a.sym_precision, geom=gmulti, ctx=ctxs[0], **cheb)
            Rm, Cm = win.moments_qr(V, a.refine_tol)
            win.close()
            qu.put((s, Rm, Cm, time.perf_counter() - ts))
        qu.put(None)
        hth.join()
        spans = [done[-1][1] - t_begin]
        last = done[-1][0]
    else:
        for s in range(a.steps):
            last, sp = one_pass()
            spans.append(sp)
    ks = ctxs[0].kernel_stats()
    for c in ctxs:
        c.set_profiling(False)
    # the unreduced FP64 window of the same disk as the reference spectrum
    lam_ref, t_full, _ = window(q, full, pts, gfull, a, cheb, "fp64",
                                a.r or q.probe_count(b, a.k0, a.R, a.nq, a.svd_tol, a.r0), 1,
                                a.r == 0)
    lams = np.concatenate([x[0] for x in last])
    n, worst, nin = match_count(lams, lam_ref, a.k0, a.R)
    nref = int(np.count_nonzero(np.abs(lam_ref - a.k0) <= a.R))
    per_pass = float(np.sum(spans)) / a.steps  # batched: the pipelined span over the passes
    out = {
        "metric": "eigenvalues/sec, C5-reduced Beyn CFIE star N=%d (5 irrep windows of %d)"
                  % (N, m_dim),
        "value": n / per_pass, "unit": "eigenvalues/s", "n_gpus": 1, "steps": a.steps,
        "warmup": max(4, a.warmup), "ms_per_step": per_pass * 1e3, "higher_is_better": True,
        "dtype": "c64+c128-refine" if a.sym_precision == "mixed" else "c128",
        "config": {"workload": "beyn-cfie-kress star(1,0.2,5) Rotation(5,m) m=0..4 k0=%g R=%g"
                               % (a.k0, a.R), "N": N, "m": m_dim, "nq": a.nq, "r": r_irrep,
                   "cheb": cheb, "precision": a.sym_precision, "slots": len(ctxs),
                   "irreps_batched": bool(a.sym_batched)},
        "irrep_window_latency_s": [round(x[2], 4) for x in last],
        "eigenvalues_matched": n, "eigenvalues_in_disk_reduced": nin,
        "eigenvalues_in_disk_full_fp64": nref, "max_rel_eig_err_vs_full_fp64": worst,
        "full_fp64_window_s": t_full,
        "pass_device_s": [round(x, 4) for x in dev_s] if a.sym_batched else None,
        "pass_host_stage_s": [round(x, 4) for x in host_s] if a.sym_batched else None,
        "kernels_first_context": {k: {"ms": round(v["ms"], 3), "launches": v["launches"]}
                                  for k, v in ks.items()},
    }
    for gl in geoms:
        for g in gl:
            g.close()
    if a.sym_batched:
        gmulti.close()
    gfull.close()
    for c in ctxs[1:]:
        c.close()
    print(json.dumps(out), flush=True)


REAL_TOL = 1e-8  # |Im lambda| <= REAL_TOL |lambda|: a real root (qbhip.serve.REAL_TOL)


def match_count(lam, ref, k0, R, tol=1e-10, real_only=False):
    """Eigenvalues inside the disk that match a reference eigenvalue (with
    real_only: real roots of both sets only).  Returns (matched, worst
    relative difference, candidates inside the disk)."""
    lam = lam[np.abs(lam - k0) <= R]
    ref = ref[np.abs(ref - k0) <= R + 1e-6]
    if real_only:
        lam = lam[np.abs(lam.imag) <= REAL_TOL * np.abs(lam)]
        ref = ref[np.abs(ref.imag) <= REAL_TOL * np.abs(ref)]
    used = np.zeros(len(ref), bool)
    n, worst = 0, 0.0
    for x in lam:
        if len(ref) == 0:
            break
        d = np.abs(ref - x) / np.abs(x)
        d[used] = np.inf
        i = int(np.argmin(d))
        if d[i] <= tol:
            used[i] = True
            n += 1
            worst = max(worst, d[i])
    return n, worst, len(lam)


def window(q, solver, pts, geom, a, cheb, precision, r, rng_seed, grow, filter_check=False):
    t0 = time.perf_counter()
    win = q.Window(solver, pts, complex(a.k0), a.R, a.nq, precision=precision, geom=geom, **cheb)
    B, Uk, info = q.construct_B_matrix(solver, pts, geom.dim, complex(a.k0), a.R, nq=a.nq, r=r,
                                       svd_tol=a.svd_tol, rng=np.random.default_rng(rng_seed),
                                       precision=precision, refine_tol=a.refine_tol,
                                       grow_r=grow, window=win, return_info=True)
    te = time.perf_counter()
    if filter_check and B.size:
        lam, Y = np.linalg.eig(B)
    else:
        lam = np.linalg.eigvals(B) if B.size else np.zeros(0, complex)
    info["t_host_eig_s"] = time.perf_counter() - te
    dt = time.perf_counter() - t0
    st = dict(win.stats)
    win.close()
    info["window_stats"] = st
    if filter_check and B.size:
        # the reference's spurious-root filter over every candidate in the
        # disk (beyn.jl:623-721), against the real-root count of the bench
        tf = time.perf_counter()
        idx, resid = q.imag_k_check_EXPERIMENTAL(solver, [lam], [Uk], [Y], [complex(a.k0)],
                                                 [a.R], [pts], res_tol=1e-6, pad=10 ** 6,
                                                 group_size=64, geoms=[geom], **cheb)
        ins = np.flatnonzero(np.abs(lam - a.k0) <= a.R)
        real = ins[np.abs(lam[ins].imag) <= REAL_TOL * np.abs(lam[ins])]
        info["residual_filter"] = {
            "candidates_in_disk": int(len(ins)), "kept_by_residual_filter": int(len(idx[0])),
            "real_roots": int(len(real)),
            "same_set": bool(set(idx[0].tolist()) == set(real.tolist())),
            "max_kept_residual": float(np.max(resid[0])) if len(resid[0]) else None,
            "seconds": round(time.perf_counter() - tf, 2)}
    return lam, dt, info


def cpu_baseline(a, cheb, r_used, count, nodes: int = 4):
    """The oracle on a bounded sample of the same window, on this host's cores:
    `nodes` contour nodes end to end -- AMOS tables (SciPy), the full N x N
    CFIE assembly (C/OpenMP restatement, oracle/qb_oracle.c), LU
    (SciPy/OpenBLAS zgetrf) and the solve with r_used probes (zgetrs) --
    extrapolated to the window's nq nodes (the nodes are independent and of
    the same cost)."""
    import scipy.linalg as sla
    from oracle import oracle as O
    try:
        from threadpoolctl import threadpool_info
        pools = threadpool_info()
        blas = max([d.get("num_threads", 1) for d in pools] or [1])
        blas_lib = ",".join(sorted({f"{d.get('internal_api')} {d.get('version')}"
                                    for d in pools if d.get("user_api") == "blas"}))
    except Exception:
        blas, blas_lib = 1, None
    omp = int(os.environ.get("OMP_NUM_THREADS", "0") or 0) or (os.cpu_count() or 1)
    cpu_model = None
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    cpu_model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    affinity = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else None
    comp = O.make_geometry("star", [a.N])[0]
    cp = O.ChebParams(cheb["n_panels_h"], cheb["M_h"], cheb["n_panels_j"], cheb["M_j"])
    rmin, rmax = O._rrange_single_fast(comp)
    V = q_probe(a.N, r_used)
    nodes = max(1, min(nodes, a.nq))
    t_asm = t_lu = t_sv = 0.0
    for j in range(nodes):
        z = complex(a.k0 + a.R * np.exp(2j * np.pi * j / a.nq))
        t0 = time.perf_counter()
        T = O.cfie_cols_c(comp, z, cp, 0, a.N, rmin, rmax)
        t_asm += time.perf_counter() - t0
        T = np.asfortranarray(T)
        t0 = time.perf_counter()
        lu = sla.lu_factor(T, overwrite_a=True, check_finite=False)
        t_lu += time.perf_counter() - t0
        t0 = time.perf_counter()
        sla.lu_solve(lu, V, check_finite=False)
        t_sv += time.perf_counter() - t0
        del T, lu
    t_win = a.nq / nodes * (t_asm + t_lu + t_sv)
    return {"value": count / t_win if t_win > 0 else None, "unit": "eigenvalues/s",
            "cores": int(max(blas, omp)), "kind": "port",
            "cpu_model": cpu_model, "nproc": os.cpu_count(), "affinity_cpus": affinity,
            "OMP_NUM_THREADS": os.environ.get("OMP_NUM_THREADS"),
            "OPENBLAS_NUM_THREADS": os.environ.get("OPENBLAS_NUM_THREADS"),
            "blas_threads": int(blas), "blas": blas_lib,
            "sampled_fraction": f"{nodes}/{a.nq} contour nodes, extrapolated",
            "sample": (f"{nodes} contour nodes of the same window: AMOS tables + C/OpenMP "
                       f"assembly ({t_asm:.1f}s) + zgetrf ({t_lu:.1f}s) + zgetrs with {r_used} "
                       f"probes ({t_sv:.1f}s); x{a.nq}/{nodes} -> {t_win:.0f} s per window, "
                       f"same eigenvalue count"),
            "window_s": t_win}


def q_probe(N, r):
    rng = np.random.default_rng(0)
    return np.asfortranarray((rng.standard_normal((N, r)) + 1j * rng.standard_normal((N, r)))
                             * np.sqrt(0.5))


def pipelined(q, ctx, solver, pts, geom, a, cheb, precision, V, steps, lanes=None):
    """Device windows back to back on this thread (moments reduced on the
    device to R and C = Q^H A1, qb_window_moments_qr); the host SVD of R, B
    and eig(B) of window s run on a second thread while the device works on
    window s+1 (NumPy's LAPACK and the ctypes calls release the GIL).  Returns
    per-window results and the span from the first window's start to the last
    result."""
    import queue
    import threading
    qu = queue.Queue()
    res = [None] * steps

    def host_stage():
        # LAPACK on all but two of this process's cores: one core keeps
        # driving the device (launches, stream waits) for the next window
        ncpu = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else 4
        try:
            from threadpoolctl import threadpool_limits
            lim = threadpool_limits(limits=max(1, ncpu - 2), user_api="blas")
        except Exception:
            lim = None
        while True:
            item = qu.get()
            if item is None:
                if lim is not None:
                    lim.restore_original_limits()
                return
            s, Rm, Cm, t_start, t_dev, st = item
            th = time.perf_counter()
            B, Ur, S, rk = q.B_from_qr(Rm, Cm, a.svd_tol)
            lam = np.linalg.eigvals(B) if B.size else np.zeros(0, complex)
            t_end = time.perf_counter()
            res[s] = (lam, rk, t_start, t_end, t_dev, t_end - th, st)

    hth = threading.Thread(target=host_stage)
    hth.start()
    t_begin = time.perf_counter()
    lanes = lanes or [(ctx, geom)]
    nxt = [0]
    lock = threading.Lock()

    def device(c, g):
        # windows taken in order from a shared counter; with several lanes
        # (device contexts) that many windows are in flight at once
        t_prev = t_begin
        while True:
            with lock:
                s = nxt[0]
                nxt[0] += 1
            if s >= steps:
                return
            t_start = time.perf_counter()
            win = q.Window(solver, pts, complex(a.k0), a.R, a.nq, precision=precision, geom=g,
                           ctx=c, **cheb)
            t_c = time.perf_counter()
            Rm, Cm = win.moments_qr(V, a.refine_tol)
            t_m = time.perf_counter()
            st = dict(win.stats)
            win.close()
            t_e = time.perf_counter()
            st["host_phases_s"] = {"create": round(t_c - t_start, 4),
                                   "moments": round(t_m - t_c, 4), "close": round(t_e - t_m, 4),
                                   "since_prev": round(t_start - t_prev, 4)}
            t_prev = t_e
            qu.put((s, Rm, Cm, t_start, time.perf_counter() - t_start, st))

    if len(lanes) == 1:
        device(*lanes[0])
    else:
        dth = [threading.Thread(target=device, args=lane) for lane in lanes]
        for t in dth:
            t.start()
        for t in dth:
            t.join()
    qu.put(None)
    hth.join()
    return res, max(x[3] for x in res) - t_begin


def main():
    a = parse()
    if a.gpus != 1:
        print(json.dumps({"error": "this build runs on one GPU; --gpus must be 1 "
                          "(multi-GPU sharding of contour nodes is a design note only)"}))
        sys.exit(2)
    if a.copy_ref:
        copy_ref(a.copy_ref)
    if a.serve:
        run_serve(a)
        return
    if a.symmetry:
        run_symmetry(a)
        return
    if a.uneven:
        run_uneven(a)
        return
    if a.assembly:
        run_assembly(a)
        return
    import qbhip as q
    ctx = q.default_context()
    # one context runs every window of this process: let its buffer cache
    # keep a whole mixed window (matrices, int8 residues, solve buffers), so
    # windows of one size allocate nothing after the first
    ctx.set_cache_limit(224 << 30)
    b = q.make_star_polar_boundary(1.0, 0.2, 5)
    solver = q.CFIE_kress(10.0, b)
    pts = q.evaluate_points(solver, b, a.k0, N=[a.N])
    geom = q.Geometry(pts, ctx)
    zj = a.k0 + a.R * np.exp(2j * np.pi * np.arange(a.nq) / a.nq)
    nh, mh, nj, mj, errs = q.chebyshev_params(solver, pts, zj, tol=a.cheb_tol, geom=geom)
    cheb = dict(n_panels_h=nh, M_h=mh, n_panels_j=nj, M_j=mj)
    print(f"# cheb tables {cheb} errs {errs}", file=sys.stderr, flush=True)

    # probes from Weyl's law for the captured interval; warmup doubles r if
    # the rank still saturates and keeps the r that does not
    r_used = a.r or q.probe_count(b, a.k0, a.R, a.nq, a.svd_tol, a.r0)
    filt = None
    for w in range(max(1, a.warmup)):
        last = w == max(1, a.warmup) - 1
        lam_m, dt, info = window(q, solver, pts, geom, a, cheb, "mixed", r_used, 1, a.r == 0,
                                 filter_check=last and not a.no_filter_check)
        r_used = info["r"]
        filt = info.get("residual_filter", filt)
        print(f"# warmup {w}: {dt:.2f}s rk={info['rk']} r={r_used} svd={info['t_host_svd_s']:.2f}s "
              f"eig={info['t_host_eig_s']:.2f}s stats={info['window_stats']} filter={filt}",
              file=sys.stderr, flush=True)
    rep = ctx.autotune(a.N, a.nq, r_used, "fp64") + ctx.autotune(a.N, a.nq, r_used, "mixed")
    print("# gemm autotune:\n" + rep, file=sys.stderr, flush=True)
    lanes = [(ctx, geom)]
    for _ in range(max(1, a.inflight) - 1):
        c2 = q.Context(0)
        c2.set_cache_limit(224 << 30)
        c2.autotune(a.N, a.nq, r_used, "fp64")
        c2.autotune(a.N, a.nq, r_used, "mixed")
        lanes.append((c2, q.Geometry(pts, c2)))
    if a.graphs:
        for c, _ in lanes:
            c.set_graphs(True)
    V = q.probe_block(np.random.default_rng(1), a.N, r_used, pinned=True)
    # both full-accuracy paths over the same windows: the complex128 path and
    # the complex64 LU refined to refine_tol; the faster one is the headline
    paths = ["fp64"] if a.no_mixed else (["mixed"] if a.no_fp64 else ["fp64", "mixed"])
    runs = {}
    for prec in paths:
        for c, _ in lanes:
            c.set_profiling(not a.no_kernel_stats)
        res, t_span = pipelined(q, ctx, solver, pts, geom, a, cheb, prec, V, a.steps, lanes=lanes)
        ks = lanes[0][0].kernel_stats()
        for c, _ in lanes:
            c.set_profiling(False)
        runs[prec] = (res, t_span, ks)
        print(f"# {prec} path: {t_span / a.steps:.3f}s per window ({a.steps} windows, "
              f"{len(lanes)} in flight)", file=sys.stderr, flush=True)
    ref = runs["fp64"][0][0][0] if "fp64" in runs else None

    def summary(prec):
        res, t_span, ks = runs[prec]
        lat, counts, cands, worst = [], [], [], 0.0
        for s in range(a.steps):
            lam, rk, t_start, t_end, t_dev, t_host, st = res[s]
            lat.append(t_end - t_start)
            nin = int(np.count_nonzero(np.abs(lam - a.k0) <= a.R))
            if ref is not None:
                n, wv, _ = match_count(lam, ref, a.k0, a.R, real_only=True)
            else:
                n, wv = int(np.count_nonzero((np.abs(lam - a.k0) <= a.R)
                                             & (np.abs(lam.imag) <= REAL_TOL * np.abs(lam)))), 0.0
            counts.append(n)
            cands.append(nin)
            worst = max(worst, wv)
            print(f"# {prec} step {s}: latency {t_end - t_start:.3f}s (device {t_dev:.3f}s, "
                  f"host {t_host:.3f}s) eig {n}/{nin} worst {wv:.2e} rk={rk} stats={st}",
                  file=sys.stderr, flush=True)
        return {"value": float(np.sum(counts) / t_span), "window_s": t_span / a.steps,
                "p50_window_s": float(np.percentile(lat, 50)),
                "p99_window_s": float(np.percentile(lat, 99)),
                "eigenvalues_per_window": int(np.median(counts)),
                "candidates_in_disk_per_window": int(np.median(cands)),
                "max_rel_eig_err_vs_fp64": worst if ref is not None else None,
                "refine_resid_max": max(float(res[s][6].get("refine_resid_max", 0.0))
                                        for s in range(a.steps)),
                "kernels": {k: {"ms": round(v["ms"], 3), "launches": v["launches"]}
                            for k, v in ks.items()}}

    sums = {p_: summary(p_) for p_ in runs}
    best = max(sums, key=lambda p_: sums[p_]["value"])
    hs = sums[best]
    ks = runs[best][2]
    kind, ty = ("gemm_c128", "c128") if best == "fp64" else ("gemm_c64", "c64")
    g = ks[kind]
    if best == "mixed" and ks["gemm_c64_bf16"]["ms"] > 0:
        # the bf16-split tiles do complex64 work too: the LU's GEMM rate counts both
        gb = ks["gemm_c64_bf16"]
        g = {k_: g[k_] + gb[k_] for k_ in ("ms", "launches", "flops", "bytes", "issued")}
    avg_ms = g["ms"] / max(g["launches"], 1)
    achieved = g["flops"] / (g["ms"] * 1e-3) / 1e12 if g["ms"] > 0 else 0.0
    issued = g["issued"] / (g["ms"] * 1e-3) / 1e12 if g["ms"] > 0 else 0.0
    default_workload = (a.N, a.nq, a.k0, a.R, r_used) == (8192, 48, 800.0, 0.5, 768)
    traffic = TRAFFIC_PER_LAUNCH.get(ty) if default_workload else None
    out = {
        "metric": "eigenvalues/sec + p99 window latency, Beyn CFIE N=8192 at 1e-10 vs FP64 path",
        "value": hs["value"], "unit": "eigenvalues/s", "n_gpus": 1, "steps": a.steps,
        "warmup": a.warmup, "ms_per_step": hs["window_s"] * 1e3, "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None,
        "dtype": "c128" if best == "fp64" else "c64+c128-refine",
        "data": "synthetic (seeded probes)",
        "config": {"workload": "beyn-cfie-kress star(1,0.2,5) k0=%g R=%g" % (a.k0, a.R),
                   "path": best, "N": a.N, "nq": a.nq, "r": r_used, "r0": a.r0,
                   "svd_tol": a.svd_tol, "cheb": cheb, "cheb_tol": a.cheb_tol,
                   "refine_tol": a.refine_tol, "inflight": len(lanes)},
        "p50_window_s": hs["p50_window_s"], "p99_window_s": hs["p99_window_s"],
        "pipeline": ("device windows back to back; host SVD/eig of window s overlaps window s+1"
                     if len(lanes) == 1 else
                     f"{len(lanes)} windows in flight on separate device contexts; host SVD/eig "
                     "of each window overlaps the device work"),
        "eigenvalues_per_window": hs["eigenvalues_per_window"],
        "counted": ("real roots inside the disk (|Im k| <= 1e-8 |k|) matching a real root of "
                    "the complex128 path within 1e-10"),
        "candidates_in_disk_per_window": hs["candidates_in_disk_per_window"],
        "residual_filter_on_warmup_window": filt,
        "paths": {p_: {k_: v_ for k_, v_ in sums[p_].items() if k_ != "kernels"} for p_ in sums},
        "mixed_vs_fp64": (sums["fp64"]["window_s"] / sums["mixed"]["window_s"]
                          if len(sums) == 2 else None),
        "kernels": hs["kernels"],
        "gemm_autotune": [l for l in rep.splitlines() if l],
        "roofline": {"kernel": ("k_gemm_sub<complex128>, every launch of the window "
                                "(panels, triangular solves, QR; FP64 MFMA; the LU's "
                                "int8 updates are kernels.gemm_c128_i8)"
                                if best == "fp64" else
                                "k_gemm_sub<complex64> + k_gemm_bf6, every launch of the "
                                "window (LU updates, triangular solves; MFMA)"),
                     "bound": "mfma", "achieved": achieved, "peak": PEAK[ty], "unit": "TFLOP/s",
                     "frac": achieved / PEAK[ty], "avg_launch_ms": avg_ms,
                     "traffic": traffic,
                     "alg_bytes_per_launch": g["bytes"] / max(g["launches"], 1),
                     "flops_per_launch": g["flops"] / max(g["launches"], 1),
                     "issued_tflops": issued, "issued_frac": issued / PEAK[ty]},
    }
    if not a.no_cpu:
        try:
            out["cpu_baseline"] = cpu_baseline(a, cheb, r_used, hs["eigenvalues_per_window"])
        except Exception as e:  # the baseline must not hide the GPU result
            out["cpu_baseline"] = {"error": repr(e)}
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
