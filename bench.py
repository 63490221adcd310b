"""Benchmark: pressure solves/s to 1e-8 relative residual on one MI355X.

Workload (one step = one pressure solve from x0 = 0): the 128^3 jittered hex box
(2,097,152 cells, interior vertices moved by +-20% of the spacing), pressure Poisson system with
coefficients |S_f| / |C_N - C_P|, zero-gradient walls, pressure pinned at cell 0, seeded
zero-mean right-hand side; smoothed-aggregation AMG (threshold 0.08 halved per level) built once
on the host; solved to |b - A x| <= 1e-8 |b| with
  * value: mixed precision - FP32 Jacobi V-cycle inside FP64 flexible CG (the metric's "mixed"),
  * beside it: the plain FP64 AMG-PCG (the reference algorithm) and the FP64 Jacobi-BiCGStab
    momentum system of the same mesh.
Inputs are resident in HBM before the timed region. The CPU baseline is the reference's own host
AMG-PCG (solve_amg_cg_host, compiled from the reference sources into oracle/_ref) on the same
hierarchy and right-hand side, timed on this machine's host cores for a bounded sample.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--size 128] [--skip-cpu]
"""
from __future__ import annotations

import argparse
import gc
import json
import os
import sys
import time
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

METRIC = "pressure solves/s @1e-8 rel-res, mixed vs FP64 AMG-PCG; HBM GB/s; p99 ms"
HBM_PEAK_GBS = 8000.0
# Kernel names as rocprofv3 reports them (profiles/ and profiles/traffic.json are keyed by these).
K_SPMV_MIXED = "k_spmv_pz<float, 1, 2>"
K_SPMV_FP64 = "k_spmv_pz<double, 1, 1>"
K_SWEEP_MIXED = "k_l0_jacobi<float, 1, 2, true>"
K_SWEEP_FP64 = "k_l0_jacobi<double, 1, 1, false>"


def _traffic() -> dict:
    """HBM bytes per launch measured by rocprofv3 --pmc (FETCH_SIZE, WRITE_SIZE) for this
    workload, keyed by kernel@cube side."""
    path = ROOT / "profiles" / "traffic.json"
    return json.loads(path.read_text())["hbm_bytes_per_launch"] if path.exists() else {}


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def cpu_model() -> str:
    try:
        for line in Path("/proc/cpuinfo").read_text().splitlines():
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def host_cores() -> int:
    """CPUs this process may run on (the GPU host's share), not the machine's count."""
    try:
        return len(os.sched_getaffinity(0))
    except AttributeError:
        return os.cpu_count() or 1


def _oracle_lists(hier_view):
    from oracle import bind as ob

    levels = hier_view.levels
    a_l = [ob.Csr(lv.a.n, lv.a.n, lv.a.row_ptr, lv.a.col, lv.a.val) for lv in levels]
    p_l = [None if lv.p is None else ob.Csr(lv.p.n, lv.p.n_cols, lv.p.row_ptr, lv.p.col, lv.p.val)
           for lv in levels]
    r_l = [None if lv.r is None else ob.Csr(lv.r.n, lv.r.n_cols, lv.r.row_ptr, lv.r.col, lv.r.val)
           for lv in levels]
    return a_l, p_l, r_l


def _ref_amg_cg(hier_view, b, tol, threads, budget_s, max_solves=1000):
    """Times the reference's solve_amg_cg_host (oracle/_ref) or, where that library was not
    built, the oracle's restatement, on `threads` host threads for about budget_s seconds;
    returns (median seconds, iterations, solves, kind, last solution)."""
    from oracle import bind as ob

    a_l, p_l, r_l = _oracle_lists(hier_view)
    ci = hier_view.coarse_inverse
    ob.set_threads(threads)
    kind = "reference" if ob.ref_available() else "port"
    times, iters = [], []
    t_start = time.perf_counter()
    x = None
    while True:
        x = np.zeros(b.shape[0])
        t0 = time.perf_counter()
        if kind == "reference":
            st = ob.ref_solve_amg_cg_host(a_l, p_l, r_l, ci, b, x, tol, 1000)
        else:
            st = ob.amg_cg_lists(a_l, p_l, r_l, ci, b, x, tol, 1000)
        times.append(time.perf_counter() - t0)
        iters.append(st.iterations)
        if time.perf_counter() - t_start > budget_s or len(times) >= max_solves:
            break
    ob.set_threads(1)
    return float(np.median(times)), int(np.median(iters)), len(times), kind, x


def _sgs_pcg(a_csr, b, tol, decay, budget_s):
    """The reference's device: "cpu" path restated by the oracle (single thread): SGS V-cycle
    AMG-PCG (amg.cpp:94-118, 192-225, 253-285) on the oracle's own hierarchy of the matrix."""
    from oracle import bind as ob

    oh = ob.Hierarchy(ob.Csr(a_csr.n, a_csr.n, a_csr.row_ptr, a_csr.col, a_csr.val), decay=decay)
    times, iters = [], []
    t_start = time.perf_counter()
    while True:
        x = np.zeros(b.shape[0])
        t0 = time.perf_counter()
        st = oh.sgs_pcg(b, x, tol, 1000)
        times.append(time.perf_counter() - t0)
        iters.append(st.iterations)
        if time.perf_counter() - t_start > budget_s:
            break
    return float(np.median(times)), int(np.median(iters)), len(times)


def cpu_baseline(hier_view, a_csr, b, tol, budget_s, label):
    """The reference's host AMG-PCG on the same hierarchy and right-hand side, on every host core
    (the primary baseline) and on one core, and the reference's CPU path (SGS V-cycle, oracle
    port) on one core, each on a bounded sample."""
    cores = host_cores()
    med, its, k, kind, _ = _ref_amg_cg(hier_view, b, tol, cores, budget_s)
    med1, its1, k1, _, _ = _ref_amg_cg(hier_view, b, tol, 1, budget_s / 3, max_solves=3)
    sgs_med, sgs_its, sgs_k = _sgs_pcg(a_csr, b, tol, 0.5, budget_s / 3)
    return {"value": 1.0 / med, "unit": "solves/s", "cores": cores, "kind": kind,
            "cpu_model": cpu_model(),
            "sample": f"{k} FP64 Jacobi-V-cycle AMG-PCG solves (solve_amg_cg_host) of {label} "
                      f"(same hierarchy, x0 = 0, 1e-8) on {cores} threads, median {med * 1e3:.1f} ms, "
                      f"{its} iterations; the reference threads loops with n > 20000",
            "one_core": {"value": 1.0 / med1, "unit": "solves/s", "cores": 1, "kind": kind,
                         "sample": f"{k1} solves, median {med1 * 1e3:.1f} ms, {its1} iterations"},
            "sgs_pcg_port": {"value": 1.0 / sgs_med, "unit": "solves/s", "cores": 1, "kind": "port",
                             "sample": f"{sgs_k} SGS-V-cycle AMG-PCG solves (the reference's device "
                                       f"\"cpu\" algorithm, amg.cpp:253-285, restated by the oracle) on "
                                       f"the oracle's hierarchy of the same matrix, median "
                                       f"{sgs_med * 1e3:.1f} ms, {sgs_its} iterations"}}


def config1_section(steps: int, cpu: bool, budget_s: float) -> dict:
    """The reference's own CPU-runnable case: 32^3 uniform box, the reference's hierarchy
    (threshold 0.08 on every level, amg.hpp:18), FP64 AMG-PCG to 1e-8 on the GPU against the
    reference's host AMG-PCG on the same hierarchy (all host cores and one core)."""
    import cfd_amd
    from cfd_amd import AmgHierarchy, DeviceSolver, Method, Precision, SolveControl, cases

    _, s = cases.config1()
    pat = cases.csr_pattern(s.n, s.owner, s.neighbour)
    a = cases.ldu_to_csr(pat, s.diag, s.upper, s.lower)
    h = AmgHierarchy(a)  # strength_decay 1.0: the reference's fixed threshold
    dev = DeviceSolver(pat)
    dev.assemble(s.diag, s.upper, s.lower)
    dev.set_amg(h.view())
    dev.set_rhs(s.source)
    tol = 1e-8 * float(np.linalg.norm(s.source))
    out = {"workload": f"32^3 uniform box ({s.n} cells), reference hierarchy (threshold 0.08 on "
                       f"every level): levels {h.level_sizes()}, operator complexity "
                       f"{h.operator_complexity():.2f}, FP64 AMG-PCG to 1e-8 from x0 = 0",
           "setup_ms_host": round(h.setup_ms, 1)}
    for prec in (Precision.FP64, Precision.MIXED_FP32):
        for _ in range(2):
            dev.set_x(None)
            dev.solve_resident(Method.Cg, True, prec, SolveControl(tol, 500))
        t = time.perf_counter()
        for _ in range(steps):
            dev.set_x(None)
            st = dev.solve_resident(Method.Cg, True, prec, SolveControl(tol, 500))
        dt = (time.perf_counter() - t) / steps
        out[prec.name.lower()] = {"solves_per_s": round(1.0 / dt, 2), "iterations": st.iterations,
                                  "converged": st.converged,
                                  "true_rel_residual": st.true_residual / st.rhs_norm}
    x_gpu = None
    dev.set_x(None)
    dev.solve_resident(Method.Cg, True, Precision.FP64, SolveControl(tol, 500))
    x_gpu = dev.get_x()
    dev.close()
    if cpu:
        cores = host_cores()
        med, its, k, kind, x_ref = _ref_amg_cg(h.view(), s.source, tol, cores, budget_s)
        med1, its1, k1, _, _ = _ref_amg_cg(h.view(), s.source, tol, 1, budget_s / 2)
        out["cpu_baseline"] = {"value": 1.0 / med, "unit": "solves/s", "cores": cores, "kind": kind,
                               "sample": f"{k} solves (solve_amg_cg_host, same hierarchy), median "
                                         f"{med * 1e3:.2f} ms, {its} iterations",
                               "one_core": {"value": 1.0 / med1, "cores": 1,
                                            "sample": f"{k1} solves, median {med1 * 1e3:.2f} ms"},
                               "gpu_fp64_rel_error_vs_reference":
                                   float(np.linalg.norm(x_gpu - x_ref) / np.linalg.norm(x_ref))}
        out["speedup_gpu_fp64_vs_cpu_all_cores"] = round(out["fp64"]["solves_per_s"] * med, 2)
    return out


def batched(steps: int, count: int = 256) -> dict:
    """Config of 256 independent pressure systems (cell counts log-uniform in [4096, 500000],
    half uniform and half jittered boxes, cell aspect 1:1:1 to 1:1:8, seeded zero-mean right-hand
    sides) solved together to 1e-8: one launch per solver stage covers every system. Reported:
    solves/s of the mixed (FP32 V-cycle, FP64 flexible CG) batch, of the FP64 batch, and of the
    plain FP64 path solving the same systems one after another; the largest relative difference
    between each mixed solution and its FP64 solution."""
    import cfd_amd
    from cfd_amd import AmgHierarchy, AmgSettings, DeviceSolver, Method, Precision, SolveControl, cases

    t0 = time.perf_counter()
    members, ctls = [], []
    cells = 0
    for s in cases.batch_shapes(count):
        mesh = cases.box_mesh(s["nx"], s["ny"], s["nz"], hi=(1.0, 1.0, s["lz"]),
                              jitter=s["jitter"], seed=s["seed"])
        p = cases.pressure_system(mesh, rhs_seed=s["seed"] + 1)
        pat = cases.csr_pattern(p.n, p.owner, p.neighbour)
        a = cases.ldu_to_csr(pat, p.diag, p.upper, p.lower)
        dev = DeviceSolver(pat)
        dev.assemble(p.diag, p.upper, p.lower)
        dev.set_amg(AmgHierarchy(a, AmgSettings(strength_decay=0.5)).view())
        dev.set_rhs(p.source)
        members.append(dev)
        ctls.append(SolveControl(1e-8 * float(np.linalg.norm(p.source)), 500))
        cells += p.n
    log(f"batch: {count} systems, {cells} cells, set up in {time.perf_counter() - t0:.1f} s")

    def timed_batch(prec):
        batch = cfd_amd.Batch(members, Method.Cg, True, prec)
        for rep in range(1 + steps):  # one untimed solve (graph capture), then the timed ones
            if rep == 1:
                t = time.perf_counter()
            batch.zero_x()  # x0 = 0 for every member, one launch
            st = batch.solve(ctls)
        dt = time.perf_counter() - t
        if not all(x.converged for x in st):
            raise RuntimeError(f"batched {prec.name}: a system did not converge")
        xs = [d.get_x() for d in members]
        batch.close()
        return count * steps / dt, dt / steps, st, xs

    sps_m, t_m, st_m, x_m = timed_batch(Precision.MIXED_FP32)
    sps_d, t_d, st_d, x_d = timed_batch(Precision.FP64)
    sps_b, t_b, st_b, x_b = timed_batch(Precision.MIXED_BF16)
    # Plain FP64 path: the same systems, one resident solve after another.
    for d, c in zip(members, ctls):
        d.set_x(None)
        d.solve_resident(Method.Cg, True, Precision.FP64, c)
    t = time.perf_counter()
    for d, c in zip(members, ctls):
        d.set_x(None)
        d.solve_resident(Method.Cg, True, Precision.FP64, c)
    t_seq = time.perf_counter() - t
    err = max(float(np.linalg.norm(a - b) / np.linalg.norm(b)) for a, b in zip(x_m, x_d))
    err_b = max(float(np.linalg.norm(a - b) / np.linalg.norm(b)) for a, b in zip(x_b, x_d))
    footprint = sum(d.footprint() for d in members)
    for d in members:
        d.close()
    its = lambda st: [int(min(x.iterations for x in st)), int(max(x.iterations for x in st))]
    return {
        "workload": f"{count} pressure systems, {cells} cells in all, log-uniform 4096..500000 "
                    "cells, SA-AMG-PCG to 1e-8 rel. residual from x0 = 0",
        "mixed_solves_per_s": round(sps_m, 2),
        "fp64_batched_solves_per_s": round(sps_d, 2),
        "fp64_one_by_one_solves_per_s": round(count / t_seq, 2),
        "bf16_batched_solves_per_s": round(sps_b, 2),
        "speedup_mixed_vs_fp64_batched": round(sps_m / sps_d, 3),
        "speedup_mixed_vs_fp64_one_by_one": round(sps_m * t_seq / count, 3),
        "ms_per_batch_mixed": round(1e3 * t_m, 2),
        "ms_per_batch_fp64": round(1e3 * t_d, 2),
        "iterations_mixed_min_max": its(st_m),
        "iterations_fp64_min_max": its(st_d),
        "max_true_rel_residual_mixed": max(x.true_residual / x.rhs_norm for x in st_m),
        "max_rel_error_mixed_vs_fp64": err,
        "max_rel_error_bf16_vs_fp64": err_b,
        "footprint_bytes": footprint,
    }


def stored_values(a) -> int:
    """Value slots the library stores for the level-0 operator of CSR matrix a when it is
    exactly symmetric (the pressure systems): the symmetric stencil storage keeps the entries
    with offset >= 0 only, one slot per stencil offset >= 0 for every row padded to 64; a matrix
    whose offsets form no small symmetric stencil keeps its nnz values."""
    rows = np.repeat(np.arange(a.n, dtype=np.int64), np.diff(a.row_ptr))
    off = np.unique(a.col.astype(np.int64) - rows)
    if len(off) > 16 or not np.array_equal(np.sort(-off), off):
        return int(a.nnz)
    return int(-(-a.n // 64) * 64 * int(np.count_nonzero(off >= 0)))


def roofline(probe, kernel, nnz, traffic=None, working_set=None, values=None, vbytes=8):
    """Roofline entry of one probed kernel: algorithmic bytes per launch under the 4-byte
    column-index convention (every stored entry counted with a 4-byte index, vectors once) over
    the HIP-event average duration, and the same on the bytes the layout stores (the level-0
    stencil layout keeps one offset table per 64-row slice and no per-entry index; with
    symmetric storage `values` value slots of vbytes each instead of nnz)."""
    ms, launches, nbytes = probe
    gbs = nbytes / (ms * 1e-3) / 1e9 if ms > 0 else 0.0
    stored = nbytes - 4.0 * nnz - (0 if values is None else vbytes * (nnz - values))
    gbs_stored = stored / (ms * 1e-3) / 1e9 if ms > 0 else 0.0
    out = {"bound": "hbm", "achieved": round(gbs, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
           "frac": round(gbs / HBM_PEAK_GBS, 4), "traffic": traffic, "kernel": kernel,
           "bytes_per_launch": int(nbytes), "avg_us": round(ms * 1e3, 3), "launches": int(launches),
           "achieved_stored": round(gbs_stored, 1), "frac_stored": round(gbs_stored / HBM_PEAK_GBS, 4),
           "stored_bytes_per_launch": int(stored)}
    if working_set is not None:
        out["working_set_mb"] = round(working_set / 1e6, 1)
    return out


def stress(n_side: int = 160, reps: int = 5) -> dict:
    """Precision stress: 160^3 jittered box, rho = 1000 inside a seeded sphere of radius 0.2 and
    1 outside (face coefficients with harmonic averaging), solved to 1e-10 relative residual by
    the FP64 AMG-PCG and by the mixed solvers (FP32 V-cycle, optionally BF16 level-0
    off-diagonals, inside FP64 flexible CG). Reported per solver: iterations, true residual,
    relative error against the FP64 solution, solves/s."""
    import cfd_amd
    from cfd_amd import AmgHierarchy, AmgSettings, DeviceSolver, Method, Precision, SolveControl, cases

    t0 = time.perf_counter()
    mesh, p = cases.config3(n_side)
    pat = cases.csr_pattern(p.n, p.owner, p.neighbour)
    a = cases.ldu_to_csr(pat, p.diag, p.upper, p.lower)
    h = AmgHierarchy(a, AmgSettings(strength_decay=0.5))
    dev = DeviceSolver(pat)
    dev.assemble(p.diag, p.upper, p.lower)
    dev.set_amg(h.view())
    dev.set_rhs(p.source)
    log(f"stress: {p.n} cells, levels {h.level_sizes()}, set up in {time.perf_counter() - t0:.1f} s")
    bnorm = float(np.linalg.norm(p.source))
    ctl = SolveControl(1e-10 * bnorm, 1000)
    out, x64, xs = {}, None, {}
    for prec in (Precision.FP64, Precision.MIXED_FP32, Precision.MIXED_BF16):
        times = []
        gc.collect()
        gc.disable()
        for _ in range(reps + 2):  # the first two solve eagerly and capture the graphs
            dev.set_x(None)
            t = time.perf_counter()
            st = dev.solve_resident(Method.Cg, True, prec, ctl)
            times.append(time.perf_counter() - t)
        gc.enable()
        x = dev.get_x()
        if prec == Precision.FP64:
            x64 = x
        xs[prec.name.lower()] = x
        out[prec.name.lower()] = {
            "iterations": st.iterations, "converged": st.converged,
            "true_rel_residual": st.true_residual / bnorm,
            "rel_error_vs_fp64": float(np.linalg.norm(x - x64) / np.linalg.norm(x64)),
            "solves_per_s": round(1.0 / float(np.median(times[2:])), 3)}
    # The mixed solve's two heaviest level-0 kernels at a working set larger than the 256 MB
    # Infinity Cache (the FP64 operator alone is 228 MB of values).
    traffic = _traffic()
    probes = {}
    for kind in (2, 1):
        dev.probe(kind)
        for _ in range(2):
            dev.set_x(None)
            dev.solve_resident(Method.Cg, True, Precision.MIXED_FP32, ctl)
        probes[kind] = dev.probe_read(Precision.MIXED_FP32)
    dev.probe(0)
    sv = stored_values(a)
    out["roofline_outer_spmv"] = roofline(probes[2], K_SPMV_MIXED, a.nnz, traffic.get(f"{K_SPMV_MIXED}@{n_side}"),
                                          dev.footprint(), sv, 8)
    out["roofline_l0_fp32_sweep"] = roofline(probes[1], K_SWEEP_MIXED, a.nnz,
                                             traffic.get(f"{K_SWEEP_MIXED}@{n_side}"), dev.footprint(), sv, 4)
    out["_solutions"] = xs  # for the CPU reference comparison; removed before printing
    out["_hierarchy"] = (h.view(), p.source, 1e-10 * bnorm)
    out["workload"] = (f"{n_side}^3 jittered box ({p.n} cells), rho 1000 in a sphere of radius "
                       "0.2 / 1 outside, harmonic faces, SA-AMG-PCG to 1e-10")
    return out


def served(count: int = 24, rate: float = 200.0, seed: int = 20240607) -> dict:
    """Serving workload: requests with Poisson arrivals (rate per second, seeded), each a
    jittered box of log-uniform 10,000..4,000,000 cells with a run of 1..20 time-step right-hand
    sides (each the previous one plus 5% seeded noise), solved to 1e-8 from the previous step's
    solution with the hierarchy kept resident. The same arrival sequence is replayed against
    the mixed-precision server (continuous batching), the FP64 server, and the plain FP64 path
    (one solve at a time); then the mixed server again with a device-memory budget of a third of
    its unconstrained peak, so that admission by footprint holds requests back, and with each
    request's hierarchy built when it arrives (setup with its sparse products on the GPU, four
    requests at a time), so that request latency includes hierarchy construction. Reported:
    solves/s over the makespan and p50 / p99 latencies."""
    import threading

    import cfd_amd
    from cfd_amd import AmgHierarchy, AmgSettings, Precision, cases

    t0 = time.perf_counter()
    gen, arrivals = cases.serving_requests(count, rate=rate, seed=seed)
    reqs, csrs, cells, solves = [], [], 0, 0
    for g in gen:
        s = g["system"]
        view = AmgHierarchy(g["csr"], AmgSettings(strength_decay=0.5)).view()
        reqs.append(dict(pattern=g["pattern"], diag=s.diag, upper=s.upper, lower=s.lower, amg=view,
                         rhs=g["rhs"]))
        csrs.append(g["csr"])
        cells += s.n
        solves += len(g["rhs"])
    log(f"serve: {count} requests, {cells} cells, {solves} solves, set up in "
        f"{time.perf_counter() - t0:.1f} s")

    def replay(prec, slots, budget=0, build_at_arrival=False):
        from concurrent.futures import ThreadPoolExecutor

        with cfd_amd.Server(max_active_solves=slots, precision=prec, memory_budget_bytes=budget) as srv:
            handles = [None] * count
            arrived = [0.0] * count
            submitted = [0.0] * count
            pool = ThreadPoolExecutor(4) if build_at_arrival else None

            def submit(i, q):
                if build_at_arrival:  # the request's hierarchy is built when it arrives (products on the GPU)
                    q = dict(q, amg=AmgHierarchy(csrs[i], AmgSettings(strength_decay=0.5), device=True).view())
                submitted[i] = time.perf_counter()
                handles[i] = srv.submit(**q, keep_solutions=False)

            def submitter():
                start = time.perf_counter()
                futures = []
                for i, q in enumerate(reqs):
                    delay = arrivals[i] - (time.perf_counter() - start)
                    if delay > 0:
                        time.sleep(delay)
                    arrived[i] = time.perf_counter()
                    if pool is not None:
                        futures.append(pool.submit(submit, i, q))
                    else:
                        submit(i, q)
                for f in futures:
                    f.result()

            t = time.perf_counter()
            th = threading.Thread(target=submitter)
            th.start()
            th.join()
            done = [srv.wait(h) for h in handles]
            span = time.perf_counter() - t
            c = srv.counters()
            if pool is not None:
                pool.shutdown()
        lat = np.concatenate([d.step_latency_ms for d in done])
        req_lat = np.array([d.latency_ms for d in done])
        if build_at_arrival:  # from arrival (before the setup) to the request's last result
            req_lat = req_lat + 1e3 * (np.array(submitted) - np.array(arrived))
        ok = all(st.converged for d in done for st in d.stats)
        worst = max(st.true_residual / st.rhs_norm for d in done for st in d.stats)
        return {"solves_per_s": round(solves / span, 2), "makespan_s": round(span, 3),
                "p50_solve_ms": round(float(np.percentile(lat, 50)), 3),
                "p99_solve_ms": round(float(np.percentile(lat, 99)), 3),
                "p50_request_ms": round(float(np.percentile(req_lat, 50)), 3),
                "p99_request_ms": round(float(np.percentile(req_lat, 99)), 3),
                "all_converged": ok, "max_true_rel_residual": worst,
                "peak_active_solves": c.peak_active_solves,
                "peak_resident_gb": round(c.peak_resident_bytes / 1e9, 2),
                "budget_gb": round(c.budget_bytes / 1e9, 2),
                "staging_thread_s": round(c.staging_ms / 1e3, 3), "retiring_thread_s": round(c.retiring_ms / 1e3, 3),
                "engine_busy_s": round(c.engine_busy_ms / 1e3, 3)}

    mixed = replay(Precision.MIXED_FP32, 64)
    fp64 = replay(Precision.FP64, 64)
    plain = replay(Precision.FP64, 1)
    budget = int(mixed["peak_resident_gb"] * 1e9 / 3)
    gated = replay(Precision.MIXED_FP32, 64, budget=budget)
    with_setup = replay(Precision.MIXED_FP32, 64, build_at_arrival=True)
    return {"workload": f"{count} requests, Poisson arrivals at {rate:g}/s, {cells} cells, "
                        f"{solves} time-step solves to 1e-8",
            "mixed_served": mixed, "fp64_served": fp64, "fp64_one_at_a_time": plain,
            "mixed_served_memory_gated": gated,
            "mixed_served_with_setup_at_arrival": with_setup,
            "speedup_mixed_vs_fp64_served": round(mixed["solves_per_s"] / fp64["solves_per_s"], 3),
            "speedup_mixed_vs_fp64_one_at_a_time":
                round(mixed["solves_per_s"] / plain["solves_per_s"], 3)}


def fv_bytes(m, op: str) -> float:
    """Algorithmic bytes of one finite-volume operation: every array element it needs, read or
    written once (the neighbour values a cell gathers are counted once, with their array)."""
    nc, nif, nf = m.n_cells, m.n_internal_faces, m.n_faces
    nb = nf - nif
    lists = 4 * (nc + 1) + 4 * (2 * nif + nb)          # cell_offsets + cell_faces
    inner = 4 * (nc + 1) + 4 * (2 * nif + nc)          # lists read up to the first boundary face
    own_nei = 8 * nif

    def gauss(k):                                        # k components
        return lists + own_nei + 8 * nif + 24 * nf + 8 * k * (nc + nb) + 8 * nc + 24 * k * nc

    def lsq(k):
        return lists + own_nei + 24 * nf + 8 * k * (nc + nb) + 72 * nc + 24 * k * nc

    def corrected(k):
        second = lists + own_nei + 8 * nif + 24 * nf + 24 * nif + 24 * nc + 8 * k * (nc + nb) + 24 * k * nc \
            + 8 * nc + 24 * k * nc
        return lsq(k) + second

    grad = {"gradient_gauss": gauss(1), "gradient_least_squares": lsq(1), "gradient_corrected": corrected(1),
            "vector_gradient_least_squares": lsq(3), "vector_gradient_corrected": corrected(3)}
    if op in grad:
        return float(grad[op])
    if op == "scalar_corrections":
        corr = inner + own_nei + 8 * nif + 24 * nif + 24 * nc + 24 * nc + 8 * nif + 8 * nif + 24 * nif + 16 * nc
        return float(lsq(1) + corr)
    if op == "momentum_corrections":
        limiter = lists + own_nei + 24 * nc + 24 * nb + 72 * nc + 24 * nf + 24 * nc + 24 * nc
        mom = inner + own_nei + 8 * nif + 24 * nif + 24 * nc + 72 * nc + 24 * nc + 24 * nc + 8 * nif + 8 * nif \
            + 24 * nif + 24 * nif + 48 * nc
        return float(limiter + mom)
    if op == "pressure_equation":  # with the relaxation-independent flux term
        hbya = inner + own_nei + 16 * nif + 24 * nc + 48 * nc + 8 * nc + 32 * nc
        press = lists + own_nei + 8 * nif + 24 * nf + 8 * nf + 32 * nc + 36 * nb + 24 * nc + 8 * nf + 16 * nf \
            + 16 * nif + 16 * nc
        return float(hbya + press)
    raise KeyError(op)


def fv_section(n_side: int = 128, reps: int = 10, cpu: bool = True) -> dict:
    """Finite-volume cell kernels (cfdg_fv_*) on an n_side^3 jittered hex box: device time of each
    operation's kernels (HIP events in the library), algorithmic GB/s against the 8 TB/s HBM
    roofline, the PCIe-inclusive time of the call, and the reference's gpu::DeviceFv host path on
    the same mesh (oracle/_ref, all host cores) as the CPU baseline."""
    from cfd_amd.fv import DeviceFv, fv_box, synthetic_pressure_inputs

    t0 = time.perf_counter()
    mesh = fv_box(n_side, n_side, n_side, jitter=0.2, seed=11)
    rng = np.random.default_rng(5)
    nc, nb, nif = mesh.n_cells, mesh.n_boundary, mesh.n_internal_faces
    phi, bv = rng.standard_normal(nc), rng.standard_normal(nb)
    u, ub = rng.standard_normal((nc, 3)), rng.standard_normal((nb, 3))
    flux, nu = rng.standard_normal(nif), rng.uniform(0.01, 0.2, nif)
    src, src3 = np.zeros(nc), np.zeros((nc, 3))
    eps2 = np.array([1e-3, 1e-3, 1e-3])
    log(f"fv: {nc} cells, {mesh.n_faces} faces, mesh built in {time.perf_counter() - t0:.1f} s")
    ops = {
        "gradient_gauss": lambda d: d.gradient(phi, bv, 0),
        "gradient_least_squares": lambda d: d.gradient(phi, bv, 1),
        "gradient_corrected": lambda d: d.gradient(phi, bv, 2),
        "vector_gradient_least_squares": lambda d: d.vector_gradient(u, ub, 1),
        "vector_gradient_corrected": lambda d: d.vector_gradient(u, ub, 2),
        "scalar_corrections": lambda d: d.scalar_corrections(phi, bv, 1, flux, nu, True, src),
        "momentum_corrections": lambda d: d.momentum_corrections(flux, nu, True, True, False, eps2, 0.0, True, src3),
    }
    pin = synthetic_pressure_inputs(mesh, 21, relax=True)
    ops["pressure_equation"] = lambda d: d.pressure_equation(pin)
    out = {"workload": f"{n_side}^3 jittered hex box ({nc} cells, {mesh.n_faces} faces), FP64",
           "roofline_peak_gbs": 8000.0, "ops": {}}
    with DeviceFv(mesh) as dev:
        dev.vector_gradient(u, ub, 1)
        for name, f in ops.items():
            f(dev)  # warm-up
            dev.timing(True)
            dms = []
            for _ in range(reps):
                f(dev)
                dms.append(dev.last_kernel_ms())
            dev.timing(False)
            t = time.perf_counter()
            for _ in range(reps):
                f(dev)
            wall = (time.perf_counter() - t) / reps
            ms = float(np.median(dms))
            nbytes = fv_bytes(mesh, name)
            gbs = nbytes / (ms * 1e-3) / 1e9
            out["ops"][name] = {"device_ms": round(ms, 4), "bytes": int(nbytes), "achieved_gbs": round(gbs, 1),
                                "frac": round(gbs / 8000.0, 4), "call_ms_with_pcie": round(1e3 * wall, 2)}
            log(f"fv {name}: {ms:.3f} ms device, {gbs:.0f} GB/s ({gbs / 80.0:.1f}% of HBM), "
                f"{1e3 * wall:.1f} ms with PCIe")
        out["pressure_handover"] = pressure_handover(mesh, dev, reps)
    dom = max(out["ops"], key=lambda k: out["ops"][k]["device_ms"])
    out["roofline"] = {"bound": "hbm", "kernel": dom, "achieved": out["ops"][dom]["achieved_gbs"], "peak": 8000.0,
                       "unit": "GB/s", "frac": out["ops"][dom]["frac"]}
    if cpu:
        out["cpu_baseline"] = fv_cpu_baseline(mesh, ops)
    return out


def pressure_handover(mesh, dev, reps: int) -> dict:
    """A solver system takes the pressure equation the DeviceFv object assembled, within HBM
    (cfdg_system_assemble_pressure), against the same equation as host arrays (assemble +
    set_rhs over PCIe): wall ms per hand-over."""
    import cfd_amd
    from cfd_amd import cases
    from cfd_amd.fv import synthetic_pressure_inputs

    nif = mesh.n_internal_faces
    pat = cases.csr_pattern(mesh.n_cells, mesh.owner[:nif].astype(np.int32), mesh.neighbour.astype(np.int32))
    eq = dev.pressure_equation(synthetic_pressure_inputs(mesh, 21, relax=True))
    sysd = cfd_amd.DeviceSolver(pat)
    try:
        res = {}
        for name, f in (("resident_ms", lambda: sysd.assemble_pressure(dev)),
                        ("host_arrays_ms", lambda: (sysd.assemble(eq.diag, eq.upper, eq.lower),
                                                    sysd.set_rhs(eq.source)))):
            f()
            t = time.perf_counter()
            for _ in range(reps):
                f()
            res[name] = round(1e3 * (time.perf_counter() - t) / reps, 3)
        res["host_bytes"] = int(8 * (2 * mesh.n_cells + 2 * nif))
    finally:
        sysd.close()
    log(f"pressure hand-over: resident {res['resident_ms']} ms, host arrays {res['host_arrays_ms']} ms")
    return res


def fv_cpu_baseline(mesh, ops) -> dict:
    """The reference's gpu::DeviceFv on host threads (oracle/_ref), one call of each operation on
    the same mesh and fields, in the same order (the momentum corrections use the vector gradient
    of the call before them)."""
    from oracle import bind as ob

    kind = "reference" if ob.ref_available() else "port"
    host = ob.FvReference(mesh) if kind == "reference" else None
    res = {}
    for name, f in ops.items():
        if host is None or name == "pressure_equation":
            continue
        t = time.perf_counter()
        f(host)
        res[name] = round(1e3 * (time.perf_counter() - t), 2)
    cores = os.cpu_count() or 1
    out = {"unit": "ms per call", "ms": res, "cores": int(os.environ.get("OMP_NUM_THREADS", cores)), "kind": kind,
           "sample": "one call of each operation on the same mesh (host arrays, no transfers)"}
    if "pressure_equation" in ops:
        # The reference's flow solver needs Eigen (absent): its face loops are timed as the
        # oracle's single-threaded C restatement.
        port = ob.FvOracle(mesh)
        t = time.perf_counter()
        ops["pressure_equation"](_OracleAsDevice(port))
        out["pressure_equation"] = {"ms": round(1e3 * (time.perf_counter() - t), 2), "cores": 1, "kind": "port"}
    return out


class _OracleAsDevice:
    """Lets the pressure-equation op run on the oracle (same call shape as DeviceFv)."""

    def __init__(self, port):
        self.port = port

    def pressure_equation(self, inp):
        return self.port.pressure_equation(inp)


def main(argv=None) -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--size", type=int, default=128)
    ap.add_argument("--skip-cpu", action="store_true")
    ap.add_argument("--cpu-seconds", type=float, default=15.0)
    ap.add_argument("--skip-batch", action="store_true")
    ap.add_argument("--skip-serve", action="store_true")
    ap.add_argument("--skip-stress", action="store_true")
    ap.add_argument("--skip-fv", action="store_true")
    ap.add_argument("--fv-only", action="store_true", help="only the finite-volume kernel section")
    ap.add_argument("--solves-only", action="store_true",
                    help="only the mixed and FP64 solves of the single system (for profiler runs)")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="only run 10 device copies of 256 MiB (HBM counter calibration)")
    args = ap.parse_args(argv)
    if args.copy_calibration:
        import torch

        src = torch.ones(32 * 2 ** 20, dtype=torch.float64, device="cuda")
        dst = torch.empty_like(src)
        for _ in range(10):
            dst.copy_(src)
        torch.cuda.synchronize()
        print(json.dumps({"copy_bytes_read": src.numel() * 8, "copy_bytes_written": dst.numel() * 8,
                          "copies": 10}))
        return 0
    if args.fv_only:
        print(json.dumps({"fv": fv_section(cpu=not args.skip_cpu)}), flush=True)
        return 0
    if args.gpus != 1:
        print(json.dumps({"error": "this build runs on one GPU only; --gpus must be 1 "
                                   "(batched and served systems shard across GPUs by system)"}))
        return 2

    import cfd_amd
    from cfd_amd import AmgHierarchy, AmgSettings, DeviceSolver, Method, Precision, SolveControl, cases

    if not cfd_amd.device_available():
        raise RuntimeError("no HIP device visible")
    log(cfd_amd.device_description())
    t0 = time.perf_counter()
    mesh, p_sys, m_sys = cases.config2(args.size)
    pat = cases.csr_pattern(p_sys.n, p_sys.owner, p_sys.neighbour)
    a = cases.ldu_to_csr(pat, p_sys.diag, p_sys.upper, p_sys.lower)
    sv0 = stored_values(a)  # level-0 value slots of the symmetric stencil storage
    log(f"generated {p_sys.n} cells / {p_sys.n_faces} faces in {time.perf_counter() - t0:.1f} s")
    hier = AmgHierarchy(a, AmgSettings(strength_decay=0.5))
    # the same setup with its sparse products on the GPU (second build: the first call in a
    # process also loads the sort kernels); the hierarchy is bit-identical
    AmgHierarchy(a, AmgSettings(strength_decay=0.5), device=True)
    setup_dev_ms = AmgHierarchy(a, AmgSettings(strength_decay=0.5), device=True).setup_ms
    log(f"AMG setup {hier.setup_ms:.0f} ms (host), {setup_dev_ms:.0f} ms (products on the GPU), "
        f"levels {hier.level_sizes()}, operator complexity {hier.operator_complexity():.3f}")
    view = hier.view()
    dev = DeviceSolver(pat)
    dev.assemble(p_sys.diag, p_sys.upper, p_sys.lower)
    sizes = hier.level_sizes()
    # the FP32 cycle's dense tail: the first level below the finest, not the coarsest, of <= 512 rows,
    # or <= 2048 rows with n^2 at most a tenth of the finest operator's entries
    tail_m = next((l for l in range(1, len(sizes) - 1)
                   if sizes[l] <= 512 or (sizes[l] <= 2048 and 10 * sizes[l] ** 2 <= a.nnz)), 0)
    if os.environ.get("CFDG_DENSE_TAIL") == "0":
        tail_m = 0
    t_set = time.perf_counter()
    dev.set_amg(view)  # uploads the levels, estimates the FP32 weights, forms the fused restrictions
    set_amg_ms = 1e3 * (time.perf_counter() - t_set)
    log(f"set_amg {set_amg_ms:.0f} ms")
    b = p_sys.source
    dev.set_rhs(b)
    bnorm = float(np.linalg.norm(b))
    tol = 1e-8 * bnorm
    ctl = SolveControl(tol, 500)

    def run(prec, k):
        lat, dev_ms, its = [], [], []
        for _ in range(k):
            t = time.perf_counter()
            dev.set_x(None)
            st = dev.solve_resident(Method.Cg, True, prec, ctl)
            lat.append(time.perf_counter() - t)
            dev_ms.append(st.solve_ms)
            its.append(st.iterations)
            if not st.converged:
                raise RuntimeError(f"{prec.name} solve did not converge: {st}")
        return np.array(lat), np.array(dev_ms), its, st

    run(Precision.MIXED_FP32, args.warmup)
    run(Precision.FP64, max(2, args.warmup))
    if args.solves_only:
        _, dm, im, _ = run(Precision.MIXED_FP32, args.steps)
        _, dd, idd, _ = run(Precision.FP64, args.steps)
        log("mixed solves (device ms): " + " ".join(f"{v:.3f}" for v in dm))
        log("FP64 solves (device ms): " + " ".join(f"{v:.3f}" for v in dd))
        print(json.dumps({"cells": p_sys.n, "mixed_device_ms": float(np.median(dm)), "mixed_iterations": im[-1],
                          "fp64_device_ms": float(np.median(dd)), "fp64_iterations": idd[-1],
                          "set_amg_ms": round(set_amg_ms, 1)}), flush=True)
        return 0
    # Timed region (the value): HIP-graph solves, no instrumentation.
    # Python's cyclic collector stays off inside the timed solves (its pauses are host time of
    # the harness, not of the library).
    gc.collect()
    gc.disable()
    t_mixed = time.perf_counter()
    lat_m, dms_m, its_m, st_m = run(Precision.MIXED_FP32, args.steps)
    t_mixed = time.perf_counter() - t_mixed
    x_mixed = dev.get_x()
    t_fp64 = time.perf_counter()
    lat_d, dms_d, its_d, st_d = run(Precision.FP64, args.steps)
    t_fp64 = time.perf_counter() - t_fp64
    x_fp64 = dev.get_x()
    run(Precision.MIXED_BF16, max(2, args.warmup))
    t_bf16 = time.perf_counter()
    lat_b, dms_b, its_b, st_b = run(Precision.MIXED_BF16, args.steps)
    t_bf16 = time.perf_counter() - t_bf16
    gc.enable()
    log("mixed solve wall ms: " + " ".join(f"{1e3 * v:.2f}" for v in lat_m))
    log("fp64 solve wall ms: " + " ".join(f"{1e3 * v:.2f}" for v in lat_d))
    x_bf16 = dev.get_x()
    log(f"bf16: {args.steps / t_bf16:.2f} solves/s, it {its_b[-1]}, true rel res "
        f"{st_b.true_residual / bnorm:.2e}")
    # Instrumented pass over the same solves: HIP events on the solve stream bracket every
    # launch of one kernel (kernel-by-kernel launches, same kernels): the mixed solve's longest
    # launch per iteration, the outer FP64 q = A p (probe 2), is the roofline kernel; beside it the
    # last level-0 Jacobi sweep of each V-cycle (probe 1) and the FP64 solve's two.
    k_probe = max(2, args.steps // 2)
    probes = {}
    for prec in (Precision.MIXED_FP32, Precision.FP64):
        for kind in (2, 1):
            dev.probe(kind)
            run(prec, k_probe)
            probes[(prec, kind)] = dev.probe_read(prec)
    dev.probe(0)
    traffic = _traffic()
    side = args.size

    # The same comparison with the same smoother: the mixed V-cycle with the reference's
    # 2 + 2 sweeps at w = 0.7 (cfdg_set_mixed_smoother ratio 0), so the ratio to the FP64
    # solve shows the precision's own gain.
    from cfd_amd import _lib as L
    tuned = json.loads((ROOT / "cfd_amd" / "tuning.json").read_text()).get("mixed_smoother", {})
    sweeps_m, ratio_m = int(tuned.get("sweeps", 1)), float(tuned.get("ratio", 6.0))
    L.call("cfdg_set_mixed_smoother", 2, 0.0)
    dev_ref = DeviceSolver(pat)
    dev_ref.assemble(p_sys.diag, p_sys.upper, p_sys.lower)
    dev_ref.set_amg(view)
    dev_ref.set_rhs(b)
    for _ in range(max(2, args.warmup)):
        dev_ref.set_x(None)
        dev_ref.solve_resident(Method.Cg, True, Precision.MIXED_FP32, ctl)
    t_same = time.perf_counter()
    for _ in range(args.steps):
        dev_ref.set_x(None)
        st_same = dev_ref.solve_resident(Method.Cg, True, Precision.MIXED_FP32, ctl)
    t_same = time.perf_counter() - t_same
    dev_ref.close()
    L.call("cfdg_set_mixed_smoother", sweeps_m, ratio_m)

    log(f"mixed: {args.steps / t_mixed:.2f} solves/s, it {its_m[-1]}, true rel res "
        f"{st_m.true_residual / bnorm:.2e}; fp64: {args.steps / t_fp64:.2f} solves/s, it {its_d[-1]}, "
        f"true rel res {st_d.true_residual / bnorm:.2e}")

    # Momentum system of the same mesh: Jacobi-BiCGStab in FP64 (config 2b).
    mdev = DeviceSolver(pat)
    mdev.assemble(m_sys.diag, m_sys.upper, m_sys.lower)
    mdev.set_rhs(m_sys.source)
    mtol = 1e-8 * float(np.linalg.norm(m_sys.source))
    # the first solve launches kernel by kernel, the second captures the graphs; the first few
    # solves after the system is built run ~1.75x slower (measured: 9.0 against 5.1 ms) and are
    # warm-up too
    for _ in range(max(8, args.warmup)):
        mdev.set_x(None)
        mdev.solve_resident(Method.BiCgStab, False, Precision.FP64, SolveControl(mtol, 2000))
    k_mom = max(1, args.steps)
    lat_mom = []
    gc.collect()
    gc.disable()
    t_mom = time.perf_counter()
    for _ in range(k_mom):
        t = time.perf_counter()
        mdev.set_x(None)
        st_mom = mdev.solve_resident(Method.BiCgStab, False, Precision.FP64, SolveControl(mtol, 2000))
        lat_mom.append(time.perf_counter() - t)
    t_mom = time.perf_counter() - t_mom
    gc.enable()
    log("momentum solve wall ms: " + " ".join(f"{1e3 * v:.2f}" for v in lat_mom))

    err = float(np.linalg.norm(x_mixed - x_fp64) / np.linalg.norm(x_fp64))
    value = args.steps / t_mixed
    fp64_value = args.steps / t_fp64
    out = {
        "metric": METRIC,
        "value": round(value, 3),
        "unit": "solves/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(1e3 * t_mixed / args.steps, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32+f64",
        "data": "synthetic",
        "config": {
            "workload": f"pressure Poisson, {args.size}^3 jittered hex box ({p_sys.n} cells), "
                        "SA-AMG-PCG to 1e-8 rel. residual from x0 = 0",
            "cells": p_sys.n,
            "nnz": int(a.nnz),
            "amg_levels": hier.level_sizes(),
            "operator_complexity": round(hier.operator_complexity(), 4),
            "strength_threshold": "0.08 * 0.5^level",
            "vcycle_mixed": f"FP32 V-cycle, {sweeps_m}+{sweeps_m} damped-Jacobi sweeps per level with "
                            f"w_l = 2 / (h_l (1 + 1/{ratio_m:g})) (degree-1 Chebyshev, h_l the top of the "
                            "D^-1 A spectrum); levels 1..L-2 of at most 65536 rows restrict with the "
                            "fused product R (I - A W); " + (
                                f"ends at level {tail_m} ({hier.level_sizes()[tail_m]} rows) with its dense "
                                "FP64 inverse (the FP32 cycle's dense tail)" if tail_m else
                                "dense FP64 coarsest inverse") + ", in FP64 flexible CG",
            "vcycle_fp64": "FP64 V-cycle, 2+2 damped-Jacobi sweeps at w = 0.7 (the reference), dense "
                           "FP64 coarsest inverse, in standard PCG",
        },
        "iterations_mixed": int(its_m[-1]),
        "iterations_fp64": int(its_d[-1]),
        "fp64_solves_per_s": round(fp64_value, 3),
        "speedup_vs_fp64": round(value / fp64_value, 3),
        "p50_ms": round(1e3 * float(np.percentile(lat_m, 50)), 3),
        "p99_ms": round(1e3 * float(np.percentile(lat_m, 99)), 3),
        "fp64_p99_ms": round(1e3 * float(np.percentile(lat_d, 99)), 3),
        "device_ms_mixed": round(float(np.median(dms_m)), 3),
        "device_ms_fp64": round(float(np.median(dms_d)), 3),
        "true_rel_residual_mixed": st_m.true_residual / bnorm,
        "true_rel_residual_fp64": st_d.true_residual / bnorm,
        "mixed_vs_fp64_rel_error": err,
        "mixed_bf16": {"solves_per_s": round(args.steps / t_bf16, 3), "iterations": int(its_b[-1]),
                       "device_ms": round(float(np.median(dms_b)), 3),
                       "p99_ms": round(1e3 * float(np.percentile(lat_b, 99)), 3),
                       "true_rel_residual": st_b.true_residual / bnorm,
                       "rel_error_vs_fp64": float(np.linalg.norm(x_bf16 - x_fp64) / np.linalg.norm(x_fp64))},
        "momentum_bicgstab_fp64": {"solves_per_s": round(k_mom / t_mom, 3),
                                   "iterations": st_mom.iterations,
                                   "true_rel_residual": st_mom.true_residual / np.linalg.norm(m_sys.source)},
        "setup_ms": round(hier.setup_ms, 1),
        "set_amg_ms": round(set_amg_ms, 1),
        "setup_ms_device_products": round(setup_dev_ms, 1),
        "footprint_bytes": dev.footprint(),
        "same_smoother": {"mixed_solves_per_s": round(args.steps / t_same, 3),
                          "iterations": st_same.iterations,
                          "true_rel_residual": st_same.true_residual / bnorm,
                          "speedup_vs_fp64": round(args.steps / t_same / fp64_value, 3),
                          "vcycle": "FP32 V-cycle with the FP64 path's smoother (2+2 sweeps, w = 0.7)"},
        "roofline": roofline(probes[(Precision.MIXED_FP32, 2)],
                             f"{K_SPMV_MIXED}: outer FP64 q = A p_new, p_new = z + beta p_old (z FP32), p.q; "
                             "the mixed solve's longest launch per iteration", a.nnz,
                             traffic.get(f"{K_SPMV_MIXED}@{side}"), None, sv0, 8),
        "roofline_l0_sweep_mixed": roofline(probes[(Precision.MIXED_FP32, 1)],
                                            f"{K_SWEEP_MIXED}: last level-0 FP32 Jacobi sweep + r.z, z.q",
                                            a.nnz, traffic.get(f"{K_SWEEP_MIXED}@{side}"), None, sv0, 4),
        "roofline_fp64_spmv": roofline(probes[(Precision.FP64, 2)],
                                       f"{K_SPMV_FP64}: FP64 q = A p_new, p_new = z + beta p_old, p.q",
                                       a.nnz, traffic.get(f"{K_SPMV_FP64}@{side}"), None, sv0, 8),
        "roofline_fp64_sweep": roofline(probes[(Precision.FP64, 1)],
                                        f"{K_SWEEP_FP64}: last level-0 FP64 Jacobi sweep + r.z", a.nnz,
                                        traffic.get(f"{K_SWEEP_FP64}@{side}"), None, sv0, 8),
        "stored_value_slots_level0": sv0,
        "working_set_mb": round(dev.footprint() / 1e6, 1),
        "roofline_note": (f"at {side}^3 the level-0 FP64 values fit the 256 MB Infinity Cache, so these "
                          "rates are not HBM evidence; precision_stress reports the same kernels at 160^3, "
                          "beyond it. frac follows the 4-byte-index convention (every entry counted with "
                          "its value and a 4-byte index); the library stores the symmetric operator's "
                          f"{sv0} value slots ({sv0 / a.nnz:.2f} per entry) and no indices, so frac can "
                          "exceed 1; frac_stored is on the stored bytes"),
        "cpu_baseline": None,
    }
    if not args.skip_batch:
        del dev, mdev
        out["batched"] = batched(max(2, args.steps // 4))
    if not args.skip_serve:
        out["served"] = served()
    stress_x, stress_h = None, None
    if not args.skip_stress:
        out["precision_stress"] = stress()
        stress_x = out["precision_stress"].pop("_solutions")
        stress_h = out["precision_stress"].pop("_hierarchy")
    if not args.skip_fv:
        out["fv"] = fv_section(cpu=not args.skip_cpu)
    out["config1"] = config1_section(max(4, args.steps // 2), not args.skip_cpu, args.cpu_seconds / 3)
    if not args.skip_cpu:
        out["cpu_baseline"] = cpu_baseline(view, a, b, tol, args.cpu_seconds,
                                           f"the same {side}^3 system")
        if stress_h is not None:
            # The precision stress against the reference's FP64 host AMG-PCG on the same
            # hierarchy (all host cores, one solve).
            hv, bs, tols = stress_h
            med, its, _, kind, x_ref = _ref_amg_cg(hv, bs, tols, host_cores(), 0.0, max_solves=1)
            ps = out["precision_stress"]
            ps["cpu_reference_fp64"] = {"kind": kind, "iterations": its, "seconds": round(med, 2),
                                        "cores": host_cores()}
            for name, x in stress_x.items():
                ps[name]["rel_error_vs_cpu_reference_fp64"] = float(np.linalg.norm(x - x_ref) /
                                                                    np.linalg.norm(x_ref))
    print(json.dumps(out), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
