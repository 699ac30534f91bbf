"""Benchmark of the sparse solve path on one MI355X.

Workload: 3-D 7-point variable-coefficient diffusion on a 128^3 grid
(n = 2,097,152, nnz = 14,581,760; log-normal face coefficients, sigma 1.5,
10:1 z anisotropy, unit diagonal), RHS N(0,1).  A step is one complete solve
from x = 0 to an FP64 true relative residual <= 1e-6 with FP32 SpMV and
vectors, FP64 dot products, FP64-accumulated residual refresh every 50
iterations, and FP64 outer refinement.  Two preconditioners are timed:
Jacobi, and the learned factor G (M^-1 = G^T G) whose network inference on
this matrix runs inside the timed solve.  The headline value is the learned
solve (graph build, inference and factored PCG), or the Jacobi solve when
the learned one is not faster or misses the residual (the fallback rule).  Inputs are resident in HBM before the timed
region.

Also measured: the CSR SpMV kernel's HBM bandwidth, rotating over four copies
of the matrix (4 x 125 MB, more than the 256 MB Infinity Cache) so the
bandwidth is HBM's, and the oracle's single-core FP64 Jacobi-PCG time on a
bounded sample of the same system.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
METRIC = "PCG time-to-solve at relres 1e-6 (learned vs Jacobi); SpMV HBM GB/s"


def spmv_bytes(n: int, nnz: int, value_bytes: int = 4, index_bytes: int = 4) -> int:
    """Algorithmic bytes of one CSR SpMV: values + columns, row offsets, x and y."""
    return nnz * (value_bytes + index_bytes) + (n + 1) * index_bytes + 2 * n * value_bytes


def pcg_iteration_bytes(n: int, nnz: int, value_bytes: int = 4, index_bytes: int = 4, diagonals: int = 0,
                        unit_diagonal: bool = False, form: int = 3, value_streams: int = 0) -> int:
    """Algorithmic bytes of one CG / Jacobi-PCG iteration.  The matrix: CSR
    values, columns and offsets, or on the diagonal layout `value_streams`
    value arrays (default: one per diagonal) and a 2-byte mask per row.  The
    vectors, per row, by form (kernels per iteration):
    3  direction reads z, p, writes p; SpMV reads p, writes q; update reads
       x, p, r, q, M^-1, writes x, r, z                        (13 vectors)
    2  step reads r, u, p, s, w, x, M^-1, writes p, s, x, r, u; SpMV reads r,
       u, s, writes w                                          (16 vectors)
    1  one kernel reads r, u, w, s, p, x, M^-1, writes p, x, s, r, u, w
                                                               (13 vectors)
    With a unit diagonal (every Jacobi inverse exactly 1) u is r: no M^-1
    read and no u write or second read (11, 12, 10 vectors).  Gathers of
    neighbouring rows are counted once, with the row's own read.  These are the
    bytes of the per-kernel forms: a solve that runs in one launch keeps the
    matrix and vectors on the CUs and moves the exchanged words only, so its
    figure can pass what memory delivers."""
    vectors = {3: (13, 11), 2: (16, 12), 1: (13, 10)}[form][1 if unit_diagonal else 0]
    if diagonals:
        return (value_streams or diagonals) * n * value_bytes + 2 * n + vectors * n * value_bytes
    return nnz * (value_bytes + index_bytes) + (n + 1) * index_bytes + vectors * n * value_bytes


def factored_iteration_bytes(n: int, form: int, value_streams: int, g_diagonals: int = 4, value_bytes: int = 4):
    """Algorithmic bytes of one single-reduction factored iteration with A, G
    and G^T on the diagonal layout (2-byte masks per row, neighbours counted
    once), or None for another form.
    4  step + G r reads G, r, w, s, p, x, u, writes p, x, s, r, t; G^T t reads
       G^T, t, writes u; SpMV reads A's value arrays, u, r, s, writes w
    5  step + G r + G^T t reads G, r, w, s, p, x, u, writes p, x, s, r, u
       (t is recomputed, G^T not read); SpMV as in 4"""
    g = g_diagonals * value_bytes + 2
    spmv = value_streams * value_bytes + 2 + 4 * value_bytes
    if form == 5:
        return n * (g + 11 * value_bytes + spmv)
    if form == 4:
        return n * (g + 11 * value_bytes + g + 2 * value_bytes + spmv)
    return None


TRAFFIC_SUMMARY = os.path.join(ROOT, "profiles", "k_spmv_diffusion128_traffic.txt")


def committed_traffic(kernel: str):
    """HBM bytes per launch of `kernel` from the committed rocprofv3 FETCH_SIZE /
    WRITE_SIZE summary (already scaled by the copy-kernel calibration), or None."""
    try:
        with open(TRAFFIC_SUMMARY) as fh:
            for line in fh:
                parts = line.split()
                if len(parts) >= 3 and parts[0] == "traffic_bytes_per_launch" and parts[1] == kernel:
                    return int(parts[2])
    except OSError:
        pass
    return None


WORKLOADS = ("diffusion128", "poisson256", "lm-schur", "lm-schur-dense", "batch512", "learned-eval", "spmm8")


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--workload", default="diffusion128", choices=WORKLOADS,
                    help="diffusion128 is the headline; the others measure the remaining solve-path workloads")
    ap.add_argument("--grid", type=int, default=128)
    ap.add_argument("--spmv-rounds", type=int, default=50)
    ap.add_argument("--cpu-iterations", type=int, default=5000,
                    help="iteration cap of the CPU baseline's FP64 solve (it stops at relres 1e-6 first)")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--graph", type=int, default=-1, help="1: chunks as HIP graphs, 0: direct launches, "
                    "-1: the library's default (graphs below 262,144 rows)")
    ap.add_argument("--chunk", type=int, default=0)
    ap.add_argument("--max-inner", type=int, default=100000)
    ap.add_argument("--inner-rel", type=float, default=1e-3,
                    help="relative tolerance of each FP32 inner solve of the refinement loop")
    ap.add_argument("--no-learned", action="store_true", help="skip the learned-preconditioner solve")
    ap.add_argument("--weights", default=os.path.join(ROOT, "plamatrix_amd", "fsai_weights.npy"),
                    help="trained network parameters (float32 .npy written by plamatrix_amd.train_fsai)")
    ap.add_argument("--eval-systems", type=int, default=256, help="learned-eval: held-out systems per kind")
    ap.add_argument("--profile", action="store_true",
                    help="short run for profilers: one solve capped at 2000 inner iterations, no CPU leg")
    args = ap.parse_args()
    if args.profile:
        args.steps, args.warmup, args.no_cpu, args.max_inner, args.spmv_rounds = 1, 0, True, 2000, 20
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py measures one GPU: the solve path runs one process per GPU and independent "
              "systems shard across GPUs without communication. Run with --gpus 1.", file=sys.stderr)
        return 2

    import torch

    from plamatrix_amd import capi, generators

    run = {"diffusion128": run_diffusion, "poisson256": run_poisson, "lm-schur": run_schur,
           "lm-schur-dense": run_schur_dense,
           "batch512": run_batch, "learned-eval": run_learned_eval, "spmm8": run_spmm}[args.workload]
    line = run(args, torch, capi, generators)
    print(json.dumps(line))
    return 0


def host_cpu() -> str:
    """CPU model, online CPUs and the CPUs this process may run on."""
    model = "unknown CPU"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    try:
        allowed = len(os.sched_getaffinity(0))
    except AttributeError:
        allowed = os.cpu_count()
    return f"{model}, nproc {os.cpu_count()}, {allowed} available to this process, 1 used"


def base_line(args, metric, value, unit, higher_is_better, dtype, config, roofline, cpu):
    return {"metric": metric, "value": value, "unit": unit, "n_gpus": 1, "steps": args.steps,
            "warmup": args.warmup, "ms_per_step": value if unit == "ms" else None,
            "higher_is_better": higher_is_better, "scaling": "weak", "vs_baseline": None, "dtype": dtype,
            "data": "synthetic", "config": config, "roofline": roofline, "cpu_baseline": cpu}


def run_diffusion(args, torch, capi, generators):
    dev = torch.device("cuda:0")
    t_gen = time.perf_counter()
    h = generators.diffusion3d_csr(args.grid)
    b_host = generators.rhs_normal(h.rows, seed=3).astype(np.float64)
    gen_s = time.perf_counter() - t_gen
    n, nnz = h.rows, h.nnz
    a = capi.to_device_csr(h, compact=True)
    b = torch.from_numpy(b_host).to(dev)
    ws = capi.Workspace()

    if args.profile:
        # a plain 512 MiB device copy: the calibration point for the profiler's
        # FETCH_SIZE / WRITE_SIZE counters (2^29 bytes read, 2^29 written)
        src = torch.ones(1 << 27, dtype=torch.float32, device=dev)
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        del src, dst

    # ---- SpMV: tune lanes on rotated copies, then measure HBM bandwidth ----
    copies = [a]
    for _ in range(3):
        copies.append(capi.DeviceCSR(n, n, None, None, a.values.clone(), a.row_offsets32.clone(),
                                     a.col_indices32.clone()))
    xs = [torch.randn(n, dtype=torch.float32, device=dev) for _ in copies]
    ys = [torch.empty(n, dtype=torch.float32, device=dev) for _ in copies]

    def time_spmv(lanes: int, rounds: int) -> float:
        for i in range(len(copies)):
            capi.spmv(copies[i], xs[i], ys[i], lanes=lanes)
        start = torch.cuda.Event(enable_timing=True)
        stop = torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        start.record()
        for _ in range(rounds):
            for i in range(len(copies)):
                capi.spmv(copies[i], xs[i], ys[i], lanes=lanes)
        stop.record()
        torch.cuda.synchronize()
        return start.elapsed_time(stop) / (rounds * len(copies))

    candidates = {lanes: time_spmv(lanes, 5) for lanes in (0, 4, 8)}
    lanes = min(candidates, key=candidates.get)
    capi.lib().pm_tune_record(capi.ctypes.byref(a.descriptor()), capi.ctypes.c_int32(lanes))
    spmv_ms = time_spmv(lanes, args.spmv_rounds)
    spmv_b = spmv_bytes(n, nnz)
    spmv_gbs = spmv_b / (spmv_ms * 1e-3) / 1e9
    del copies[1:], xs, ys

    # ---- time-to-solve ----------------------------------------------------------
    pol = capi.policy(refresh_interval=50, use_graph=args.graph, chunk_iterations=args.chunk)
    x = torch.zeros(n, dtype=torch.float64, device=dev)
    inner = dict(relative_tolerance=args.inner_rel, max_iterations=args.max_inner)

    def timed(run):
        for _ in range(args.warmup):
            run()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        reps = [run() for _ in range(args.steps)]
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) / args.steps * 1e3, reps[-1]

    def jacobi_solve():
        x.zero_()
        return capi.pcg_refine(a, b, x, ws, target=1e-6, max_outer=10, pol=pol, **inner)

    ms_per_solve, rep = timed(jacobi_solve)
    relres = capi.true_relres(a, b, x, ws)
    iterations = rep.inner_iterations
    diagonals = ws.solver_diagonals
    # the matrix is scaled to a unit diagonal: its Jacobi solve runs as the
    # identical unpreconditioned iteration (no M^-1 read, no z write)
    unit_diagonal = ws.solver_preconditioner == "none"
    form, streams = ws.solver_form, ws.solver_value_streams
    it_bytes = pcg_iteration_bytes(n, nnz, diagonals=diagonals, unit_diagonal=unit_diagonal, form=form,
                                   value_streams=streams)
    it_ms = ms_per_solve / max(iterations, 1)

    # ---- learned preconditioner: G inferred on this matrix inside the timed solve ----
    learned = None
    if not args.no_learned:
        net = capi.FsaiNet(seed=0)
        net.parameters = np.load(args.weights)
        torch.cuda.synchronize()
        f0 = time.perf_counter()
        fg = capi.FsaiGraph(a)  # features, couplings, lower/upper patterns: once per sparsity pattern
        torch.cuda.synchronize()
        graph_ms = (time.perf_counter() - f0) * 1e3

        def learned_solve():
            x.zero_()
            capi.fsai_forward(net, fg)
            return capi.pcg_refine_factored(a, b, x, fg, ws, target=1e-6, max_outer=10, pol=pol, **inner)

        l_ms, l_rep = timed(learned_solve)
        l_form = ws.solver_form
        l_bytes = factored_iteration_bytes(n, l_form, ws.solver_value_streams)
        l_relres = capi.true_relres(a, b, x, ws)
        torch.cuda.synchronize()
        f0 = time.perf_counter()
        for _ in range(3):
            capi.fsai_forward(net, fg)
        torch.cuda.synchronize()
        fwd_ms = (time.perf_counter() - f0) / 3 * 1e3
        # one-off solve: the per-pattern graph build, network inference and the
        # factored solve; with a reused pattern only the last two recur
        total_ms = graph_ms + l_ms
        fallback = not (l_rep.converged and l_relres <= 1e-6 and total_ms < ms_per_solve)
        learned = {"ms": round(total_ms, 3), "solve_ms_pattern_reused": round(l_ms, 3),
                   "converged": l_rep.converged, "outer": l_rep.outer_iterations,
                   "inner_iterations": l_rep.inner_iterations, "true_relres": l_relres,
                   "forward_ms": round(fwd_ms, 3), "graph_build_ms": round(graph_ms, 3),
                   "ms_per_iteration": round((l_ms - fwd_ms) / max(l_rep.inner_iterations, 1), 4),
                   "kernels_per_iteration": {5: 2, 4: 3, 3: 4}.get(l_form),
                   "iteration_bytes": l_bytes,
                   "time_ratio_vs_jacobi": round(total_ms / ms_per_solve, 4),
                   "iteration_ratio_vs_jacobi": round(l_rep.inner_iterations / max(iterations, 1), 4),
                   "fewer_iterations_than_jacobi": l_rep.inner_iterations < iterations,
                   "fallback_to_jacobi": fallback, "weights": os.path.relpath(args.weights, ROOT)}
        del net, fg

    # to 1e-8 as well (refinement) - reported, not the headline
    x.zero_()
    torch.cuda.synchronize()
    t8 = time.perf_counter()
    rep8 = capi.pcg_refine(a, b, x, ws, target=1e-8, max_outer=1 if args.profile else 20, pol=pol, **inner)
    torch.cuda.synchronize()
    ms_1e8 = (time.perf_counter() - t8) * 1e3

    # ---- CPU baseline: the reference's FP64 Jacobi-PCG, one core, one full solve ----
    cpu = None
    if not args.no_cpu:
        import oracle

        use_ref = oracle.ref_available()
        ref = oracle.CSR(n, n, h.row_offsets, h.col_indices, h.values.astype(np.float64))
        c0 = time.perf_counter()
        cx, crep = oracle.pcg(ref, b_host, relative_tolerance=1e-6, max_iterations=args.cpu_iterations,
                              use_ref=use_ref)
        cpu_s = time.perf_counter() - c0
        import scipy.sparse as sp

        A64 = sp.csr_matrix((h.values.astype(np.float64), h.col_indices, h.row_offsets), shape=(n, n))
        cpu_relres = float(np.linalg.norm(b_host - A64 @ cx) / np.linalg.norm(b_host))
        who = ("the reference's own CPU pcg (iterative_solver_cpu.cpp built from source, serial, FP64 vectors)"
               if use_ref else "the oracle's restatement of iterative_solver_cpu.cpp (oracle/sparse.c, serial)")
        cpu = {"value": round(cpu_s * 1e3, 1), "unit": "ms", "cores": 1,
               "kind": "reference" if use_ref else "port",
               "sample": f"one full solve of the 128^3 system (FP64 values and rhs, x0 = 0) by {who} to its "
                         f"relative tolerance 1e-6: {crep.iterations} iterations, converged={crep.converged}, "
                         f"FP64 true relres {cpu_relres:.3e}; host {host_cpu()}",
               "iterations": crep.iterations, "true_relres": cpu_relres}

    kernel = "k_spmv<float,int>" if lanes == 0 else f"k_spmv_lanes<float,int,{lanes}>"
    # headline: learned preconditioner with its Jacobi fallback (taken when the
    # learned solve, graph build included, is not faster or misses the residual)
    if learned is not None and not learned["fallback_to_jacobi"]:
        value = learned["ms"]
    else:
        value = ms_per_solve
    line = {
        "metric": METRIC,
        "value": round(value, 3),
        "unit": "ms",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(value, 3),
        "higher_is_better": False,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {
            "workload": f"3-D 7-point variable-coefficient diffusion {args.grid}^3 (n={n}, nnz={nnz}), "
                        "solve from x=0 to FP64 true relres 1e-6: learned G^T G preconditioner (G inferred inside "
                        "the timed solve) with Jacobi-PCG fallback; FP32 SpMV/vectors + FP64 dots, residual "
                        "refresh every 50, FP64 refinement",
            "headline": "jacobi (fallback)" if learned is None or learned["fallback_to_jacobi"] else "learned",
            "rows": n, "nnz": nnz, "index_bits": 32, "lanes_per_row": lanes, "graph": {-1: "library default (direct launches at this size)", 0: False, 1: True}[args.graph],
        },
        "roofline": {"bound": "hbm", "achieved": round(spmv_gbs, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": round(spmv_gbs / HBM_PEAK_GBS, 4), "traffic": committed_traffic(kernel),
                     "traffic_source": "read from the committed rocprofv3 --pmc summary "
                                       "profiles/k_spmv_diffusion128_traffic.txt, not measured in this run",
                     "kernel": kernel, "bytes_per_launch": spmv_b,
                     "ms_per_launch": round(spmv_ms, 5)},
        "cpu_baseline": cpu,
        "learned": learned,
        "solve": {"preconditioner": "jacobi", "jacobi_kernels": "unit diagonal: z = r" if unit_diagonal else "z = M^-1 r", "ms": round(ms_per_solve, 3), "converged": rep.converged, "outer": rep.outer_iterations, "inner_iterations": iterations,
                  "true_relres": relres, "ms_per_iteration": round(it_ms, 4),
                  "matrix_layout": (f"diagonal ({diagonals} diagonals, {streams} value arrays read)" if diagonals
                                    else "csr"),
                  "kernels_per_iteration": form,
                  "iteration_bytes": it_bytes, "iteration_gbs": round(it_bytes / (it_ms * 1e-3) / 1e9, 1),
                  "to_1e8": {"ms": round(ms_1e8, 2), "outer": rep8.outer_iterations,
                             "inner_iterations": rep8.inner_iterations, "relres": rep8.final_relres}},
        "spmv": {"gbs": round(spmv_gbs, 1), "ms": round(spmv_ms, 5), "lanes_candidates_ms": candidates},
        "setup_s": round(gen_s, 2),
    }
    return line



def _median_ms(fn, repeats):
    """Median wall time of fn() in ms, device-synchronised around each call."""
    import torch

    times = []
    out = None
    for _ in range(repeats):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        out = fn()
        torch.cuda.synchronize()
        times.append((time.perf_counter() - t0) * 1e3)
    times.sort()
    return times[len(times) // 2], out


def _event_ms(torch, fn, repeats):
    """Mean device time of fn() in ms from HIP events on the current stream."""
    fn()
    start = torch.cuda.Event(enable_timing=True)
    stop = torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    start.record()
    for _ in range(repeats):
        fn()
    stop.record()
    torch.cuda.synchronize()
    return start.elapsed_time(stop) / repeats


def _cpu_median_s(fn, repeats):
    times = []
    out = None
    for _ in range(repeats):
        t0 = time.perf_counter()
        out = fn()
        times.append(time.perf_counter() - t0)
    times.sort()
    return times[len(times) // 2], out


def run_poisson(args, torch, capi, generators):
    """2-D 5-point Poisson 256^2 from shuffled COO triplets with 10% split
    duplicates: device COO->CSR (steady state, output preallocated) and FP64
    Jacobi-PCG to relative 1e-8 (max 2000) from x = 0, RHS U[-1,1] seed 1."""
    dev = torch.device("cuda:0")
    coo = generators.poisson2d_coo(256)
    n, t_count = coo.rows, len(coo.values)
    r = torch.from_numpy(coo.row_indices).to(dev)
    c = torch.from_numpy(coo.col_indices).to(dev)
    v = torch.from_numpy(coo.values).to(dev)
    ws = capi.Workspace()
    a = capi.coo_to_csr(n, n, r, c, v, ws)
    nnz = a.nnz
    def convert():
        # a workspace's deferred status must be read before its next conversion
        capi.coo_to_csr_async(n, n, r, c, v, a, ws)
        torch.cuda.synchronize()
        ws.check_status()

    conv_ms, _ = _median_ms(convert, 20)
    conv_bytes = t_count * (8 + 8 + 8) + nnz * (8 + 8) + (n + 1) * 8
    sync_ms, _ = _median_ms(lambda: capi.coo_to_csr(n, n, r, c, v, ws), 5)
    rhs = generators.rhs_uniform(n, seed=1)
    b = torch.from_numpy(rhs).to(dev)
    x = torch.zeros(n, dtype=torch.float64, device=dev)

    def solve():
        x.zero_()
        return capi.pcg(a, b, x, ws, capi.policy(chunk_iterations=args.chunk, use_graph=args.graph),
                        relative_tolerance=1e-8, max_iterations=2000)

    for _ in range(args.warmup):
        solve()
    solve_ms, rep = _median_ms(solve, max(args.steps, 3))
    form = ws.solver_form
    one_launch = ws.solver_one_launch == 1
    kernels = {1: "k_cg_fused_dia", 2: "k_cg_step + k_cg_spmv", 3: "k_direction + k_spmv_den + k_update"}[form]
    if one_launch:
        kernels = {1: "k_cg_persist", 2: "k_cg_csr"}[form] + ", one launch per solve"
    relres = capi.true_relres(a, b, x, ws)
    it_bytes = pcg_iteration_bytes(n, nnz, value_bytes=8, index_bytes=4 if a.row_offsets32 is not None else 8,
                                   form=form)
    it_ms = solve_ms / max(rep.iterations, 1)
    cpu = None
    if not args.no_cpu:
        import oracle

        use_ref = oracle.ref_available()
        c_conv, ref_csr = _cpu_median_s(lambda: oracle.coo_to_csr(n, n, coo.row_indices, coo.col_indices,
                                                                   coo.values, use_ref=use_ref), 5)
        c_solve, (_, crep) = _cpu_median_s(lambda: oracle.pcg(ref_csr, rhs, relative_tolerance=1e-8,
                                                               max_iterations=2000, use_ref=use_ref), 3)
        who = "the reference's own CPU cooToCsr and pcg (built from source)" if use_ref else "the oracle"
        cpu = {"value": round(c_solve * 1e3, 2), "unit": "ms", "cores": 1, "kind": "reference" if use_ref else "port",
               "sample": f"full workload, serial, median of 3 ({who}): PCG {crep.iterations} iterations "
                         f"{c_solve * 1e3:.1f} ms; COO->CSR median of 5: {c_conv * 1e3:.2f} ms"}
    line = base_line(args, "FP64 Jacobi-PCG time-to-solve at relres 1e-8, 2-D Poisson 256^2", round(solve_ms, 3),
                     "ms", False, "f64",
                     {"workload": f"2-D 5-point Poisson 256^2 (n={n}, nnz={nnz}) from {t_count} shuffled COO "
                                  "triplets with 10% split duplicates; device COO->CSR, FP64 Jacobi-PCG from x=0 "
                                  "to relres 1e-8, max 2000", "rows": n, "nnz": nnz, "triplets": t_count},
                     {"bound": "hbm", "achieved": round(it_bytes / (it_ms * 1e-3) / 1e9, 1), "peak": HBM_PEAK_GBS,
                      "unit": "GB/s", "frac": round(it_bytes / (it_ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
                      "traffic": None, "kernel": f"PCG iteration ({kernels})",
                      "bytes_per_launch": it_bytes, "ms_per_launch": round(it_ms, 5),
                      "note": f"latency-bound: {it_bytes / 1e6:.1f} MB per iteration in the per-kernel form"
                              + ("; one launch per solve keeps them on the CUs" if one_launch else "")},
                     cpu)
    line["solve"] = {"converged": rep.converged, "iterations": rep.iterations, "true_relres": relres}
    line["coo_to_csr"] = {"ms_steady": round(conv_ms, 4), "ms_synchronous": round(sync_ms, 4),
                          "bytes": conv_bytes, "gbs": round(conv_bytes / (conv_ms * 1e-3) / 1e9, 1)}
    return line


def _schur_assembly_bytes(inst, slots, values, terms):
    """Algorithmic bytes of the Schur numeric assembly: W, C, B read, the reduced
    values written, three int64 indices per term."""
    w_count = len(inst.primary)
    return (w_count * 18 * 8 + inst.eliminated_count * 9 * 8 + inst.primary_count * 36 * 8 + values * 8
            + terms * 3 * 8)


def run_schur(args, torch, capi, generators):
    """Synthetic LM / Schur system (2,000 primaries x 6, 200,000 secondaries x 3,
    1.2M residuals of dimension 2, Huber delta 1, lambda 1e-3): device normal
    equations from the Jacobians, reduced Schur assembly over the reused
    pattern, FP64 block-Jacobi PCG to relative 1e-6, back-substitution."""
    dev = torch.device("cuda:0")
    inst = generators.lm_schur_instance()
    t = lambda arr, dt: torch.from_numpy(np.ascontiguousarray(arr, dtype=dt)).to(dev)
    batch = dict(primary=t(inst.primary, np.int64), eliminated=t(inst.eliminated, np.int64),
                 primary_jacobians=t(inst.primary_jacobians, np.float64),
                 eliminated_jacobians=t(inst.eliminated_jacobians, np.float64),
                 residuals=t(inst.residuals, np.float64))
    pc, ec = inst.primary_count, inst.eliminated_count
    sw = capi.SchurWorkspace()
    ws = capi.Workspace()
    dp = torch.zeros(pc * 6, dtype=torch.float64, device=dev)
    de = torch.zeros(ec * 3, dtype=torch.float64, device=dev)

    def step():
        ne = capi.assemble_normal_equations(sw, pc, ec, 6, 3, **batch, weights=None, huber_delta=inst.huber_delta)
        rep = capi.schur_solve(sw, ne, inst.damping, dp, de, ws, max_iterations=2000, relative_tolerance=1e-6,
                               absolute_tolerance=0.0)
        return ne, rep

    torch.cuda.synchronize()
    t0 = time.perf_counter()
    ne, first = step()  # builds the pattern
    torch.cuda.synchronize()
    first_ms = (time.perf_counter() - t0) * 1e3
    for _ in range(args.warmup):
        step()
    ms, (ne, rep) = _median_ms(step, max(args.steps, 3))
    if not rep.converged:
        raise RuntimeError(rep.message)
    slots, values, terms = sw.pattern_size()
    ne_ms = _event_ms(torch, lambda: capi.assemble_normal_equations(
        sw, pc, ec, 6, 3, **batch, weights=None, huber_delta=inst.huber_delta), 5)
    asm_ms = _event_ms(torch, lambda: capi.schur_assemble(sw, ne, inst.damping), 5)
    asm_bytes = _schur_assembly_bytes(inst, slots, values, terms)
    r_count = len(inst.primary)
    ne_bytes = r_count * (12 + 6 + 2) * 8 + r_count * 2 * 8
    cpu = None
    if not args.no_cpu:
        import oracle

        if oracle.ref_available():
            w = generators.huber_weights(inst.residuals, inst.huber_delta)
            c_s, (_, _, crep) = _cpu_median_s(lambda: oracle.ref_schur_solve_batch(
                pc, ec, 6, 3, inst.primary, inst.eliminated, inst.primary_jacobians, inst.eliminated_jacobians,
                inst.residuals, w, inst.damping, backend=0, max_iterations=2000, relative_tolerance=1e-6,
                absolute_tolerance=0.0), 3)
            cpu = {"value": round(c_s * 1e3, 1), "unit": "ms", "cores": 1, "kind": "reference",
                   "sample": f"full workload, median of 3: the reference's own solveDampedSchurComplement with "
                             f"the CPU linear backend (built from source, serial) from the same residual batch "
                             f"and Huber weights, {crep.iterations} block-Jacobi PCG iterations"}
    line = base_line(args, "LM Schur step time (device normal equations + reduced Schur assembly + block-Jacobi "
                           "PCG to relres 1e-6 + back-substitution)", round(ms, 3), "ms", False, "f64",
                     {"workload": f"LM/Schur: {pc} primaries x 6, {ec} secondaries x 3, {r_count} residuals x 2, "
                                  "Huber delta 1, lambda 1e-3; reduced 12,000 x 12,000 system in 6x6 blocks, "
                                  "pattern reused", "slots": slots, "values": values, "terms": terms},
                     {"bound": "hbm", "achieved": round(asm_bytes / (asm_ms * 1e-3) / 1e9, 1), "peak": HBM_PEAK_GBS,
                      "unit": "GB/s", "frac": round(asm_bytes / (asm_ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
                      "traffic": None, "kernel": "reduced Schur numeric assembly (pm_schur_assemble)",
                      "bytes_per_launch": asm_bytes, "ms_per_launch": round(asm_ms, 4)},
                     cpu)
    line["solve"] = {"converged": rep.converged, "iterations": rep.iterations,
                     "final_residual_norm": rep.final_residual_norm, "initial_residual_norm": rep.initial_residual_norm,
                     "first_call_ms_with_pattern_build": round(first_ms, 2)}
    line["normal_equations"] = {"ms": round(ne_ms, 4), "bytes_read": ne_bytes,
                                "gbs": round(ne_bytes / (ne_ms * 1e-3) / 1e9, 1)}
    return line


def run_schur_dense(args, torch, capi, generators):
    """The LM / Schur step of run_schur with the dense backend (the reference's
    DenseCpu): device normal equations, reduced assembly, dense FP64 Cholesky
    of the 12,000 x 12,000 reduced system, triangular solves, residual check
    and back-substitution."""
    dev = torch.device("cuda:0")
    inst = generators.lm_schur_instance()
    t = lambda arr, dt: torch.from_numpy(np.ascontiguousarray(arr, dtype=dt)).to(dev)
    batch = dict(primary=t(inst.primary, np.int64), eliminated=t(inst.eliminated, np.int64),
                 primary_jacobians=t(inst.primary_jacobians, np.float64),
                 eliminated_jacobians=t(inst.eliminated_jacobians, np.float64),
                 residuals=t(inst.residuals, np.float64))
    pc, ec = inst.primary_count, inst.eliminated_count
    sw = capi.SchurWorkspace()
    ws = capi.Workspace()
    dp = torch.zeros(pc * 6, dtype=torch.float64, device=dev)
    de = torch.zeros(ec * 3, dtype=torch.float64, device=dev)

    def step():
        ne = capi.assemble_normal_equations(sw, pc, ec, 6, 3, **batch, weights=None, huber_delta=inst.huber_delta)
        rep = capi.schur_solve(sw, ne, inst.damping, dp, de, ws, relative_tolerance=1e-10, absolute_tolerance=0.0,
                               dense=True)
        return ne, rep

    step()
    for _ in range(args.warmup):
        step()
    ms, (ne, rep) = _median_ms(step, max(args.steps, 3))
    if not rep.converged:
        raise RuntimeError(rep.message)
    # the dense solve alone on the assembled reduced system, timed with HIP
    # events on the stream it runs on
    a, rhs_ptr, _ = capi.schur_system(sw)
    n = a.rows
    x = torch.empty(n, dtype=torch.float64, device=dev)
    solve_ms = _event_ms(torch, lambda: capi.dense_cholesky_solve(a, rhs_ptr, x.data_ptr(), ws), 3)
    flops = n ** 3 / 3 + 2 * n ** 2  # factorization + two triangular solves
    tflops = flops / (solve_ms * 1e-3) / 1e12
    cpu = None
    if not args.no_cpu:
        import oracle

        if oracle.ref_available():
            # bounded sample: the same generator at half the primaries (a 6,000 x
            # 6,000 reduced system), scaled by 8 = 2^3 for the cubic factorization
            half = generators.lm_schur_instance(primary_count=pc // 2, eliminated_count=ec // 2)
            w = generators.huber_weights(half.residuals, half.huber_delta)
            c_s, (_, _, crep) = _cpu_median_s(lambda: oracle.ref_schur_solve_batch(
                pc // 2, ec // 2, 6, 3, half.primary, half.eliminated, half.primary_jacobians,
                half.eliminated_jacobians, half.residuals, w, half.damping, backend=1, relative_tolerance=1e-10,
                absolute_tolerance=0.0), 1)
            threads = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))
            cpu = {"value": round(c_s * 8e3, 1), "unit": "ms", "cores": threads, "kind": "reference",
                   "sample": f"the reference's own solveDampedSchurComplement with the DenseCpu backend (built "
                             f"from source, OpenMP, {threads} threads) on the same generator at {pc // 2} "
                             f"primaries x {ec // 2} secondaries (6,000 x 6,000 reduced system): "
                             f"{c_s * 1e3:.0f} ms, scaled by 8 for the cubic factorization"}
    line = base_line(args, "LM Schur step time with the dense Cholesky backend (device normal equations + reduced "
                           "Schur assembly + dense FP64 Cholesky + triangular solves + residual check + "
                           "back-substitution)", round(ms, 3), "ms", False, "f64",
                     {"workload": f"LM/Schur: {pc} primaries x 6, {ec} secondaries x 3, {len(inst.primary)} "
                                  "residuals x 2, Huber delta 1, lambda 1e-3; reduced 12,000 x 12,000 system "
                                  "factored densely", "rows": n},
                     {"bound": "mfma", "achieved": round(tflops, 2), "peak": 78.6, "unit": "TFLOP/s",
                      "frac": round(tflops / 78.6, 4), "traffic": None,
                      "kernel": "pm_dense_cholesky_solve (k_dc_potrf + k_dc_gemm FP64 MFMA + triangular solves)",
                      "flops_per_launch": int(flops), "ms_per_launch": round(solve_ms, 3)},
                     cpu)
    line["solve"] = {"converged": rep.converged, "final_residual_norm": rep.final_residual_norm,
                     "initial_residual_norm": rep.initial_residual_norm}
    return line


def run_batch(args, torch, capi, generators):
    """512 uneven SPD systems in one batched solve: per-system FP32 SpMV with
    FP64 dots, per-system relative tolerance 1e-6, device-side convergence
    flags and graph-replayed iterations."""
    dev = torch.device("cuda:0")
    t0 = time.perf_counter()
    from plamatrix_amd import workloads

    batch = workloads.batch_systems(capi, generators, torch)
    a, begin, end, kinds, lens, nnzs, members = (batch.a, batch.begin, batch.end, batch.kinds, batch.lens,
                                                 batch.nnzs, batch.members)
    gen_s = time.perf_counter() - t0
    total = a.rows
    rng = np.random.default_rng(7)
    b_host = np.zeros(total, dtype=np.float64)
    for b0, ln in zip(begin, lens):
        b_host[b0:b0 + ln] = rng.standard_normal(ln)
    b = torch.from_numpy(b_host).to(dev)
    x = torch.zeros(total, dtype=torch.float64, device=dev)
    ws = capi.Workspace()
    pol = capi.policy(refresh_interval=50, use_graph=args.graph)
    # the reduced Schur members (6x6-block systems, as in the single LM solve)
    # take 6x6 block-Jacobi, the Laplacian and diffusion members Jacobi
    blocks = [6 if k == "schur" else 1 for k in kinds]

    def solve():
        x.zero_()
        return capi.batch_block_pcg_refine(a, begin, end, blocks, b, x, ws, target=1e-6, max_outer=10, pol=pol,
                                           relative_tolerance=args.inner_rel, max_iterations=20000)

    def solve_jacobi():
        x.zero_()
        return capi.batch_pcg_refine(a, begin, end, b, x, ws, target=1e-6, max_outer=10, pol=pol,
                                     relative_tolerance=args.inner_rel, max_iterations=20000)

    solve_jacobi()
    jacobi_ms, reps_j = _median_ms(solve_jacobi, 3)
    its_j = np.array([r.inner_iterations for r in reps_j])
    for _ in range(args.warmup):
        solve()
    ms, reps = _median_ms(solve, max(args.steps, 3))
    its = np.array([r.inner_iterations for r in reps])
    outer = np.array([r.outer_iterations for r in reps])
    conv = sum(r.converged for r in reps)
    # per-system FP64 true residuals (host, FP64) of the last solve
    xh = x.cpu().numpy()
    import scipy.sparse as sp

    worst = 0.0
    for (where, m), b0, ln in zip(members, begin, lens):
        if where == "host":
            A = sp.csr_matrix((m.values.astype(np.float64), m.col_indices, m.row_offsets), shape=(ln, ln))
        else:
            # the FP32-rounded values the batch solves
            _, ro, ci, va = m
            A = sp.csr_matrix((va.float().double().cpu().numpy(), ci.cpu().numpy(), ro.cpu().numpy()),
                              shape=(ln, ln))
        bb = b_host[b0:b0 + ln]
        worst = max(worst, float(np.linalg.norm(bb - A @ xh[b0:b0 + ln]) / np.linalg.norm(bb)))
    # algorithmic bytes of the per-kernel form (systems held on the CUs move fewer):
    # each system's iteration traffic times its iterations (a block-Jacobi row also reads its 6-value inverse row)
    streamed = sum((pcg_iteration_bytes(ln, z) + (6 * 4 * ln if bs > 1 else 0)) * int(it)
                   for ln, z, it, bs in zip(lens, nnzs, its, blocks))
    gbs = streamed / (ms * 1e-3) / 1e9
    cpu = None
    if not args.no_cpu:
        import oracle

        use_ref = oracle.ref_available()
        sample = list(range(0, len(lens), 32))
        c_s = 0.0
        work_sample = 0.0
        cpu_its = []
        for i in sample:
            where, m = members[i]
            if where == "host":
                csr = oracle.CSR(lens[i], lens[i], m.row_offsets, m.col_indices, m.values.astype(np.float64))
            else:
                _, ro, ci, va = m
                csr = oracle.CSR(lens[i], lens[i], ro.cpu().numpy(), ci.cpu().numpy(),
                                 va.float().double().cpu().numpy())
            rhs = b_host[begin[i]:begin[i] + lens[i]]
            c0 = time.perf_counter()
            _, crep = oracle.pcg(csr, rhs, relative_tolerance=1e-6, max_iterations=20000, use_ref=use_ref)
            c_s += time.perf_counter() - c0
            cpu_its.append(int(crep.iterations))
            work_sample += nnzs[i] * max(int(crep.iterations), 1)
        # the other systems' Jacobi iteration counts from the batched Jacobi solve
        work_all = float(sum(z * max(int(it), 1) for z, it in zip(nnzs, its_j)))
        who = "the reference's own CPU pcg (built from source)" if use_ref else "the oracle's CPU pcg"
        cpu = {"value": round(c_s * work_all / work_sample * 1e3, 1), "unit": "ms", "cores": 1,
               "kind": "reference" if use_ref else "port",
               "sample": f"{len(sample)} of the 512 systems (every 32nd) solved one by one, serial FP64 Jacobi-PCG "
                         f"to 1e-6 by {who}, {c_s:.1f} s ({sum(cpu_its)} iterations); scaled to all systems by "
                         "sum(nnz x Jacobi iterations), the other systems' counts from the batched Jacobi solve"}
    line = base_line(args, "Batched PCG time-to-solve, 512 uneven systems at per-system relres 1e-6", round(ms, 3),
                     "ms", False, "f32",
                     {"workload": f"512 systems, n log-uniform in [1e3, 2e5] (seed 4), cycling 2-D Laplacian / 3-D "
                                  f"diffusion / reduced LM Schur; {total} rows (64-aligned), {int(sum(nnzs))} nnz; "
                                  "batched PCG (6x6 block-Jacobi on the Schur members, Jacobi on the others) with "
                                  "FP32 SpMV/vectors + FP64 dots, residual refresh every 50, batched FP64 refinement "
                                  "to per-system true relres 1e-6",
                      "rows": int(sum(lens)), "nnz": int(sum(nnzs)), "systems": len(lens)},
                     {"bound": "hbm", "achieved": round(gbs, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                      "frac": round(gbs / HBM_PEAK_GBS, 4), "traffic": None,
                      "kernel": "batched PCG iteration (sum over systems of iteration bytes x iterations / solve time)",
                      "bytes_per_launch": int(streamed), "ms_per_launch": round(ms, 3)},
                     cpu)
    line["solve"] = {"converged": int(conv), "systems": len(reps), "inner_iterations_max": int(its.max()),
                     "inner_iterations_mean": round(float(its.mean()), 1), "outer_max": int(outer.max()),
                     "worst_true_relres": worst, "worst_reported_relres": max(r.final_relres for r in reps),
                     "setup_s": round(gen_s, 1)}
    schur = [i for i, k in enumerate(kinds) if k == "schur"]
    line["jacobi_only"] = {"ms": round(jacobi_ms, 3), "converged": int(sum(r.converged for r in reps_j)),
                           "inner_iterations_max": int(its_j.max()),
                           "schur_inner_iterations_mean": round(float(its_j[schur].mean()), 1)}
    line["solve"]["schur_inner_iterations_mean"] = round(float(its[schur].mean()), 1)
    return line


def run_learned_eval(args, torch, capi, generators):
    """Held-out evaluation of the trained network on scaled-down 3-D diffusion
    boxes and reduced LM Schur systems (eval seeds 2*10^6 + i), all systems of
    both kinds in one batch: one batched learned solve (graph build over the
    block-diagonal matrix, inference, the per-system Jacobi fallback chosen on
    the device by probe loss, batched factored PCG) against one batched
    Jacobi-PCG solve of the same systems, FP32 inner solves refined in FP64 to a
    true relres of 1e-6 per system.  Also timed: plain Jacobi-PCG one system per
    call (the reference's shape), on the same GPU."""
    from plamatrix_amd import train_fsai, workloads

    dev = torch.device("cuda:0")
    net = capi.FsaiNet(seed=0)
    net.parameters = np.load(args.weights)
    count = args.eval_systems
    t0 = time.perf_counter()
    hosts = [train_fsai.make_system("diffusion", 2_000_000 + i) for i in range(count)]
    hosts += [train_fsai.make_system("schur", 2_050_000 + i) for i in range(count)]
    kinds = ["diffusion"] * count + ["schur"] * count
    a, begin, end, lens, nnzs = workloads.pack_members(capi, torch, [("host", h) for h in hosts], dev,
                                                       pad_identity=True)
    gen_s = time.perf_counter() - t0
    rng = np.random.default_rng(11)
    b_host = np.zeros(a.rows)
    for b0, ln in zip(begin, lens):
        b_host[b0:b0 + ln] = rng.standard_normal(ln)
    b = torch.from_numpy(b_host).to(dev)
    x = torch.zeros_like(b)
    ws = capi.Workspace()
    pol = capi.policy(refresh_interval=50, use_graph=args.graph)
    inner = dict(relative_tolerance=args.inner_rel, max_iterations=20000)
    state = {}

    def jacobi():
        x.zero_()
        return capi.batch_pcg_refine(a, begin, end, b, x, ws, target=1e-6, max_outer=10, pol=pol, **inner)

    def learned():
        graph = capi.FsaiGraph(a)
        capi.fsai_forward(net, graph)
        flags, losses = capi.fsai_batch_select(graph, begin, end, probes=8, seed=1)
        x.zero_()
        reps = capi.batch_pcg_refine_factored(a, begin, end, b, x, graph, ws, jacobi=flags, target=1e-6,
                                              max_outer=10, pol=pol, **inner)
        state.update(flags=flags, losses=losses, graph=graph)
        return reps

    def learned_pattern_reused():
        graph = state["graph"]
        capi.fsai_forward(net, graph)
        flags, _ = capi.fsai_batch_select(graph, begin, end, probes=8, seed=1)
        x.zero_()
        return capi.batch_pcg_refine_factored(a, begin, end, b, x, graph, ws, jacobi=flags, target=1e-6,
                                              max_outer=10, pol=pol, **inner)

    for _ in range(args.warmup):
        jacobi()
        learned()
    j_ms, jreps = _median_ms(jacobi, max(args.steps, 3))
    xj = x.cpu().numpy()
    l_ms, lreps = _median_ms(learned, max(args.steps, 3))
    xl = x.cpu().numpy()
    r_ms, _ = _median_ms(learned_pattern_reused, max(args.steps, 3))
    flags = state["flags"].cpu().numpy()
    import scipy.sparse as sp

    worst = {"jacobi": 0.0, "learned": 0.0}
    per_kind = {}
    for kind in ("diffusion", "schur"):
        idx = [i for i in range(len(hosts)) if kinds[i] == kind]
        ji = np.array([jreps[i].inner_iterations for i in idx])
        li = np.array([lreps[i].inner_iterations for i in idx])
        kept = np.array([flags[i] == 0 for i in idx])
        per_kind[kind] = {"systems": len(idx), "learned_kept": int(kept.sum()),
                          "jacobi_iterations_mean": round(float(ji.mean()), 2),
                          "learned_iterations_mean": round(float(li.mean()), 2),
                          "iteration_ratio": round(float(li.sum() / ji.sum()), 4),
                          "kept_with_more_iterations": int(((li >= ji) & kept).sum())}
    for i, (h, b0, e0) in enumerate(zip(hosts, begin, end)):
        A = sp.csr_matrix((h.values.astype(np.float64), h.col_indices, h.row_offsets), shape=(h.rows, h.rows))
        bb = b_host[b0:e0]
        for name, xs in (("jacobi", xj), ("learned", xl)):
            worst[name] = max(worst[name], float(np.linalg.norm(bb - A @ xs[b0:e0]) / np.linalg.norm(bb)))
    # plain Jacobi-PCG one system per call (FP64 refinement, same target)
    sample = list(range(0, len(hosts), 8))
    dev_csrs = [capi.to_device_csr(hosts[i], compact=True) for i in sample]
    rhs = [torch.from_numpy(b_host[begin[i]:end[i]].copy()).to(dev) for i in sample]

    def per_system():
        for d, bb in zip(dev_csrs, rhs):
            xx = torch.zeros_like(bb)
            capi.pcg_refine(d, bb, xx, ws, target=1e-6, max_outer=10, pol=pol, **inner)

    per_system()
    s_ms, _ = _median_ms(per_system, 3)
    seq_ms = s_ms * len(hosts) / len(sample)
    conv = all(r.converged for r in jreps) and all(r.converged for r in lreps)
    line = base_line(args, "Batched learned vs batched Jacobi PCG wall-time ratio on held-out systems at relres 1e-6",
                     round(l_ms / j_ms, 4), "ratio", False, "f32",
                     {"workload": f"{count} held-out scaled-down 3-D diffusion boxes (16..33 per side) and {count} "
                                  "reduced LM Schur systems (300 primaries, 6,000 secondaries), eval seeds 2*10^6+i, "
                                  f"in one batch ({a.rows} rows, {sum(nnzs)} nnz); FP32 inner batched PCG with FP64 "
                                  "refinement to a per-system FP64 true relres of 1e-6",
                      "weights": os.path.relpath(args.weights, ROOT)},
                     None, None)
    line["batched"] = {"jacobi_ms": round(j_ms, 3), "learned_ms": round(l_ms, 3),
                       "learned_ms_pattern_reused": round(r_ms, 3),
                       "learned_includes": "graph build, inference, per-system selection, batched factored solve",
                       "all_converged": conv, "worst_true_relres": worst}
    line["one_system_per_call"] = {"jacobi_ms": round(seq_ms, 3),
                                   "sample": f"{len(sample)} of {len(hosts)} systems (every 8th) solved one per call "
                                             "by pm_pcg_refine, scaled by the system count",
                                   "batched_learned_ratio": round(l_ms / seq_ms, 4),
                                   "batched_jacobi_ratio": round(j_ms / seq_ms, 4)}
    line["per_kind"] = per_kind
    line["setup_s"] = round(gen_s, 1)
    return line


def run_spmm(args, torch, capi, generators):
    """Y = A B with 8 column-major right-hand sides on the 128^3 diffusion
    matrix (FP32, int32 indices), rotating over four copies of the matrix as
    the SpMV measurement does, against eight separate SpMVs."""
    dev = torch.device("cuda:0")
    k = 8
    h = generators.diffusion3d_csr(args.grid)
    n, nnz = h.rows, h.nnz
    a = capi.to_device_csr(h, compact=True)
    copies = [a] + [capi.DeviceCSR(n, n, None, None, a.values.clone(), a.row_offsets32.clone(),
                                   a.col_indices32.clone()) for _ in range(3)]
    bs = [torch.randn((k, n), dtype=torch.float32, device=dev) for _ in copies]
    ys = [torch.empty((k, n), dtype=torch.float32, device=dev) for _ in copies]
    ws = capi.Workspace()
    rounds = 20

    def spmm_all():
        for i in range(len(copies)):
            capi.spmm(copies[i], bs[i], ys[i], ws)

    def spmv_all():
        for i in range(len(copies)):
            for j in range(k):
                capi.spmv(copies[i], bs[i][j], ys[i][j], ws)

    spmm_ms = _event_ms(torch, spmm_all, rounds) / len(copies)
    spmv_ms = _event_ms(torch, spmv_all, 5) / len(copies)
    byts = nnz * 8 + (n + 1) * 4 + 2 * k * n * 4
    gbs = byts / (spmm_ms * 1e-3) / 1e9
    cpu = None
    if not args.no_cpu:
        import oracle

        use_ref = oracle.ref_available()
        csr = oracle.CSR(n, n, h.row_offsets, h.col_indices, h.values)
        bh = np.asfortranarray(bs[0].cpu().numpy().T)
        c_s, _ = _cpu_median_s(lambda: oracle.spmm(csr, bh, use_ref=use_ref), 3)
        cpu = {"value": round(c_s * 1e3, 1), "unit": "ms", "cores": 1, "kind": "reference" if use_ref else "port",
               "sample": "full workload, median of 3: the reference's own CPU spmm (built from source, serial)"
                         if use_ref else "full workload, median of 3: the oracle's CPU spmm"}
    line = base_line(args, "CSR SpMM time, 8 right-hand sides, 3-D 7-point diffusion 128^3", round(spmm_ms, 4), "ms",
                     False, "f32",
                     {"workload": f"Y = A B, A 3-D 7-point diffusion {args.grid}^3 (n={n}, nnz={nnz}) FP32/int32, "
                                  "B and Y 8 column-major columns; four rotated matrix copies", "rows": n, "nnz": nnz,
                      "columns": k},
                     {"bound": "hbm", "achieved": round(gbs, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                      "frac": round(gbs / HBM_PEAK_GBS, 4), "traffic": None,
                      "kernel": "k_spmm_pack<float> + k_spmm_tile<float,int> (one 8-column tile)",
                      "bytes_per_launch": byts, "ms_per_launch": round(spmm_ms, 5)},
                     cpu)
    line["eight_spmv_ms"] = round(spmv_ms, 4)
    line["speedup_vs_eight_spmv"] = round(spmv_ms / spmm_ms, 2)
    return line

if __name__ == "__main__":
    sys.exit(main())
