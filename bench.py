#!/usr/bin/env python3
"""Benchmark of the CCSD amplitude-residual hot path on one MI355X.

Default workload (one "step" = one CCSD iteration over resident data):
  ccsd-h2o8  (H2O)8 on a 2x2x2 lattice (O-O 2.8 A, seeded 0.1 A jitter, random
             orientations), cc-pVDZ, o=40, v=152: RHF and AO->MO on the host,
             then the converged solve to 1e-8 and K timed iterations
             (update + tau + residual + energy/error) in FP64 and in each
             mixed-precision form; the headline is the fastest form within
             1 uEh of FP64.

Prints ONE JSON line with the metric, the roofline of the dominant kernel (the
V+ GEMM of the pair-symmetric pp-ladder contraction, 2 (v(v+1)/2)^2 o^2 FLOPs
per launch; the full contraction's 2 o^2 v^4 where that form runs) and the CPU
baseline (one oracle residual on the host cores).

Other workloads: pp-ladder (R[a,b,i,j] += sum_cd tau[c,d,i,j] V[a,b,c,d],
o=32, v=256, FP64, ccsd_r1_r2.h:275; V ~ N(0, 0.05) symmetrised to the 8-fold
(ac|bd) symmetry, tau ~ N(0, 1e-2) / (e_c + e_d - e_i - e_j)); ccsd-h2o6
(o=30, v=114); ccsd-h20 (H20 chain, o=10, v=90); copy (counter calibration);
batched-hchains; adjoint-h2o6; df-h2o8 (density-fitted residual, method df);
transform-h2o8 (AO->MO integral transform on the device); triples-h2o6 / triples-h2o8 (CCSD(T)).
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

# TFLOP/s dense MFMA, MI355X, of the unit each form's contractions run on
PEAK = {"f64": 78.6, "f32": 157.3, "bf16x3": 2500.0, "f16x3": 2500.0, "bf16x6": 2500.0}
MFMA_PRODUCTS = {"f64": 1, "f32": 1, "bf16x3": 3, "f16x3": 3, "bf16x6": 6}
DTYPE = {"f64": "f64",
         "f32": "f32-mfma contractions / f64 update, DIIS, energy",
         "bf16x3": "bf16 hi+lo split contractions (3 products) / f64 update, DIIS, energy",
         "f16x3": "fp16 hi+lo split contractions (3 products) / f64 update, DIIS, energy",
         "bf16x6": "bf16 hi+mid+lo split contractions (6 products) / f64 update, DIIS, energy"}


def _args():
    p = argparse.ArgumentParser()
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--steps", type=int, default=5)
    p.add_argument("--warmup", type=int, default=2)
    p.add_argument("--workload", default="ccsd-h2o8",
                   choices=["ccsd-h2o8", "ccsd-h2o6", "ccsd-h20", "pp-ladder", "copy",
                            "batched-hchains", "adjoint-h2o6", "df-h2o8", "transform-h2o8",
                            "triples-h2o6", "triples-h2o8", "eom-h2o6", "direct-h2o8"])
    p.add_argument("--forms", default="f64,f16x3,bf16x3",
                   help="contraction precisions to run for the CCSD workloads (first = reference)")
    p.add_argument("--max-iter", type=int, default=40)
    p.add_argument("--copy-gib", type=float, default=4.0,
                   help="size of the plain copy used to calibrate rocprofv3 byte counters")
    p.add_argument("--precision", default="f64", choices=["f64", "f32", "bf16x3"])
    p.add_argument("--o", type=int, default=32)
    p.add_argument("--v", type=int, default=256)
    p.add_argument("--no-cpu-baseline", action="store_true")
    p.add_argument("--no-small-system", action="store_true",
                   help="skip the H20-chain FP64 iteration the (H2O)8 line also reports")
    p.add_argument("--batch-count", type=int, default=256, help="chains in the batched workload")
    p.add_argument("--batch-mem-gib", type=float, default=150.0,
                   help="HBM budget per group of chains in the batched workload")
    p.add_argument("--batch-precision", default="f64", choices=["f64", "f32"])
    p.add_argument("--cpu-sample-rows", type=int, default=8192)
    return p.parse_args()


def make_pp_ladder_inputs(o, v, seed=2):
    """Synthetic pp-ladder operands, generated on the GPU (V) / host (tau)."""
    import numpy as np
    import torch
    rng = np.random.default_rng(seed)
    e_occ = rng.uniform(-1.5, -0.3, o)
    e_vir = rng.uniform(0.1, 3.0, v)
    tau = rng.normal(0.0, 1e-2, (v, v, o, o))
    tau /= (e_vir[:, None, None, None] + e_vir[None, :, None, None]
            - e_occ[None, None, :, None] - e_occ[None, None, None, :])
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    # X[p,q,r,s] = (pq|rs) ~ N(0, 0.05), symmetrised over the 8 real-orbital
    # permutations; V[a,b,c,d] = (ac|bd)
    X = torch.empty((v, v, v, v), dtype=torch.float64, device="cuda")
    X.normal_(0.0, 0.05, generator=g)
    S = X.clone()
    for perm in [(1, 0, 2, 3), (0, 1, 3, 2), (1, 0, 3, 2), (2, 3, 0, 1), (3, 2, 0, 1),
                 (2, 3, 1, 0), (3, 2, 1, 0)]:
        S.add_(X.permute(*perm))
    del X
    S.mul_(0.125)
    V = S.permute(0, 2, 1, 3).contiguous()
    del S
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return V, torch.from_numpy(tau).to("cuda"), e_occ, e_vir, tau


def cpu_baseline_pp(V, tau_np, rows):
    """The oracle's pp-ladder contraction (oracle.ccsd.pp_ladder, a BLAS dgemm
    through numpy) on a bounded sample of rows (a,b) of V."""
    import numpy as np
    from oracle import ccsd as O  # noqa: F401  (the oracle defines the contraction)
    v = tau_np.shape[0]
    o = tau_np.shape[2]
    rows = min(rows, v * v)
    Vs = V.reshape(v * v, v * v)[:rows].cpu().numpy()
    T = tau_np.reshape(v * v, o * o)
    Vs @ T[:, :8]  # warm the BLAS pool
    t0 = time.perf_counter()
    R = Vs @ T
    dt = time.perf_counter() - t0
    flops = 2.0 * rows * v * v * o * o
    threads = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))
    return {"value": flops / dt / 1e12, "unit": "TFLOP/s", "cores": threads, "kind": "port",
            "seconds": dt,
            "sample": f"oracle pp-ladder GEMM on rows 0..{rows - 1} of V ({rows}x{v * v} @ "
                      f"{v * v}x{o * o}, {flops:.3e} FLOPs, numpy/OpenBLAS fp64)",
            "full_kernel_seconds_extrapolated": dt * (v * v) / rows}, R


def uneven_hashmarks(n, rng, lo=20, hi=64):
    """TiledRange1 hashmarks with tile sizes drawn uniformly from {lo..hi}; the
    last tile is clipped into [lo, hi] by merging or splitting with its
    predecessor."""
    hm = [0]
    while n - hm[-1] > hi:
        hm.append(hm[-1] + int(rng.integers(lo, hi + 1)))
    if n - hm[-1] < lo and len(hm) > 1:
        hm.pop()
        rest = n - hm[-1]
        if rest > hi:
            hm.append(hm[-1] + rest // 2)
    hm.append(n)
    return hm


def pp_ladder_tile_boundary(V, o, v, seed=2):
    """The pp-ladder workload's operands arrive as TiledArray tiles of uneven
    sizes 20-64: the seeded tiling is applied to V, the tiled buffer is handed to
    a context through mpqc_ccsd_set_integral (device memory, TA layout), and the
    gathered dense Gabcd is read back and compared with V.  Returns the tilings
    and the gather time (not part of the contraction's timed region)."""
    import ctypes
    import numpy as np
    import torch
    from mpqc_amd import _lib as L
    rng = np.random.default_rng(seed)
    occ_hm = uneven_hashmarks(o, rng) if o > 64 else [0, o]
    vir_hm = uneven_hashmarks(v, rng)
    ho = (ctypes.c_int64 * len(occ_hm))(*occ_hm)
    hv = (ctypes.c_int64 * len(vir_hm))(*vir_hm)
    lib = L.load()
    ctx = ctypes.c_void_p()
    L.check(lib.mpqc_ccsd_ctx_create(o, v, ho, len(occ_hm) - 1, hv, len(vir_hm) - 1, L.PREC_F64,
                                     ctypes.byref(ctx)), None)
    try:
        tiled = torch.empty_like(V)
        # dense -> tiles through the context (set dense, read back in tile layout)
        L.check(lib.mpqc_ccsd_set_integral(ctx, L.INT_GABCD, ctypes.c_void_p(V.data_ptr()), L.LAYOUT_DENSE,
                                           L.MEM_DEVICE), ctx)
        L.check(lib.mpqc_ccsd_get_integral(ctx, L.INT_GABCD, ctypes.c_void_p(tiled.data_ptr()),
                                           L.LAYOUT_TA_TILES, L.MEM_DEVICE), ctx)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        L.check(lib.mpqc_ccsd_set_integral(ctx, L.INT_GABCD, ctypes.c_void_p(tiled.data_ptr()),
                                           L.LAYOUT_TA_TILES, L.MEM_DEVICE), ctx)
        gather_s = time.perf_counter() - t0
        back = torch.empty_like(V)
        L.check(lib.mpqc_ccsd_get_integral(ctx, L.INT_GABCD, ctypes.c_void_p(back.data_ptr()), L.LAYOUT_DENSE,
                                           L.MEM_DEVICE), ctx)
        torch.cuda.synchronize()
        same = bool(torch.equal(back, V))
        moved = not bool(torch.equal(tiled.reshape(-1)[:4096], V.reshape(-1)[:4096]))
        del tiled, back
    finally:
        lib.mpqc_ccsd_ctx_destroy(ctx)
    torch.cuda.empty_cache()
    sizes = [b - a for a, b in zip(vir_hm[:-1], vir_hm[1:])]
    log(f"uneven tiles: vir {sizes}; TA-tile gather of V {gather_s * 1e3:.1f} ms, round trip exact: {same}")
    return {"occ_hashmarks": occ_hm, "vir_hashmarks": vir_hm, "vir_tile_sizes": sizes,
            "gather_ms": round(gather_s * 1e3, 3), "round_trip_exact": same and moved,
            "note": "tiles are gathered into the dense GEMM layout once at the boundary"}


def bench_pp_ladder(args):
    import numpy as np
    import torch
    from mpqc_amd.ccsd import pp_ladder
    o, v = args.o, args.v
    V, tau, e_occ, e_vir, tau_np = make_pp_ladder_inputs(o, v)
    R = torch.zeros((v, v, o, o), dtype=torch.float64, device="cuda")
    stream = torch.cuda.current_stream()
    sptr = stream.cuda_stream

    def step():
        pp_ladder(V.data_ptr(), tau.data_ptr(), R.data_ptr(), o, v, 1.0, 0.0, args.precision,
                  stream=sptr)

    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    starts = [torch.cuda.Event(enable_timing=True) for _ in range(args.steps)]
    ends = [torch.cuda.Event(enable_timing=True) for _ in range(args.steps)]
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for k in range(args.steps):
        starts[k].record(stream)
        step()
        ends[k].record(stream)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    kms = [s.elapsed_time(e) for s, e in zip(starts, ends)]
    ms = sum(kms) / len(kms)
    flops = 2.0 * o * o * float(v) ** 4
    tflops = flops / (ms * 1e-3) / 1e12
    # parity spot check against float64 host products on a few rows
    rows = np.random.default_rng(5).choice(v * v, 16, replace=False)
    Vr = V.reshape(v * v, v * v)[torch.from_numpy(rows).to("cuda")].cpu().numpy()
    ref = Vr @ tau_np.reshape(v * v, o * o)
    got = R.reshape(v * v, o * o)[torch.from_numpy(rows).to("cuda")].cpu().numpy()
    max_rel = float(np.abs(got - ref).max() / np.abs(ref).max())
    tiles = pp_ladder_tile_boundary(V, o, v) if args.precision == "f64" else None
    cpu = None
    if not args.no_cpu_baseline:
        cpu, _ = cpu_baseline_pp(V, tau_np, args.cpu_sample_rows)
    line = {
        "metric": "CCSD iter wall-time + TFLOP/s (frac MFMA peak), mixed vs FP64 at <=1 uEh",
        "value": round(tflops, 3),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms, 3),
        "wall_s_timed_region": round(wall, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": {"f64": "f64", "f32": "f32-mfma", "bf16x3": "bf16x3-split"}[args.precision],
        "data": "synthetic (seeded: V torch CUDA generator seed 2, tau numpy PCG64 seed 2)",
        "config": {"workload": f"pp-ladder R[ab,ij]+=sum_cd tau[cd,ij] V[ab,cd] o={o} v={v}",
                   "o": o, "v": v, "flops_per_step": flops, "precision": args.precision,
                   "parallelism": "single-gpu"},
        "roofline": {"bound": "mfma", "achieved": round(tflops, 3),
                     "peak": PEAK[args.precision], "unit": "TFLOP/s",
                     "frac": round(tflops / PEAK[args.precision], 4),
                     "traffic": profiled_traffic("pp-ladder", args.precision, "pp_ladder")[0],
                     "kernel": "dgemm_f64_kernel (pp-ladder GEMM M=v^2 N=o^2 K=v^2)"},
        "parity_max_rel_err_vs_fp64_host": max_rel,
        "ta_tiles": tiles,
        "cpu_baseline": cpu,
    }
    if cpu:
        line["cpu_baseline"]["gpu_speedup"] = round(tflops / cpu["value"], 1)
    return line


SYSTEMS = {
    # name: (description, builder)
    "ccsd-h2o8": "(H2O)8 on a 2x2x2 cubic lattice, O-O 2.8 A +- U[0.1] A jitter, random "
                 "orientations (seed 4), cc-pVDZ, all electrons (o=40, v=152)",
    "ccsd-h2o6": "(H2O)6 on a 3x2x1 lattice, same generator (seed 5), cc-pVDZ, all electrons "
                 "(o=30, v=114)",
    "ccsd-h20": "linear H20 chain, 1.8 bohr spacing, cc-pVDZ, all electrons (o=10, v=90)",
}


def profiled_traffic(workload, form, kernel):
    """HBM bytes per launch of `kernel` measured with rocprofv3 FETCH_SIZE /
    WRITE_SIZE (calibrated against a device copy), read from the summaries under
    profiles/ (lines 'bench-traffic: workload=... form=... kernel=... bytes=...')."""
    import glob
    import re
    for path in sorted(glob.glob(os.path.join(ROOT, "profiles", "*.md"))):
        with open(path) as fh:
            for line in fh:
                m = re.match(r"\s*bench-traffic: workload=(\S+) form=(\S+) kernel=(\S+) bytes=(\S+)", line)
                if m and m.group(1) == workload and m.group(2) == form and m.group(3) == kernel:
                    return float(m.group(4)), os.path.relpath(path, ROOT)
    return None, None


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def build_system(name):
    from mpqc_amd.chem.molecule import h_chain, water_cluster
    from mpqc_amd.chem.scf import rhf
    from mpqc_amd.chem.mo import ccsd_integrals
    if name == "ccsd-h2o8":
        mol = water_cluster((2, 2, 2), seed=4)
    elif name == "ccsd-h2o6":
        mol = water_cluster((3, 2, 1), seed=5)
    else:
        mol = h_chain(20, 1.8)
    log(f"{name}: {len(mol.symbols)} atoms, RHF/cc-pVDZ")
    t0 = time.perf_counter()
    scf = rhf(mol, "cc-pVDZ")
    t1 = time.perf_counter()
    log(f"RHF E={scf.energy:.10f} in {t1 - t0:.1f}s; AO->MO")
    inp = ccsd_integrals(scf, frozen_core=False)
    t2 = time.perf_counter()
    log(f"MO integrals o={inp.o} v={inp.v} in {t2 - t1:.1f}s")
    del scf
    return inp, {"rhf_s": round(t1 - t0, 2), "ao2mo_s": round(t2 - t1, 2)}


def host_info():
    """CPU model, usable cores and the BLAS numpy runs on (for the CPU baseline)."""
    import numpy as np  # noqa: F401  (loads the BLAS so threadpoolctl sees it)
    model = "unknown"
    try:
        with open("/proc/cpuinfo") as fh:
            for line in fh:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    blas = "unknown"
    try:
        import threadpoolctl
        for lib in threadpoolctl.threadpool_info():
            if lib.get("user_api") == "blas":
                blas = f"{lib.get('internal_api')} {lib.get('version')} ({lib.get('architecture')}, " \
                       f"{lib.get('num_threads')} threads)"
                break
    except ImportError:
        pass
    try:
        cores = len(os.sched_getaffinity(0))
    except AttributeError:
        cores = os.cpu_count() or 1
    return {"cpu_model": model, "blas": blas, "host_cores_visible": cores}


def _blas_threads():
    try:
        import threadpoolctl
        for lib in threadpoolctl.threadpool_info():
            if lib.get("user_api") == "blas":
                return int(lib.get("num_threads"))
    except ImportError:
        pass
    return int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))


def cpu_baseline_ccsd(inp, n_iter=2):
    """The oracle's solver loop (oracle.ccsd.compute_ccsd: Jacobi + DIIS update,
    tau, cs_ccsd_r1 + cs_ccsd_r2, error and energy, as ccsd.h:367-468) on the
    host cores from the initial guess, timed per full iteration between
    successive energy evaluations; plus the dominant contraction (the pp-ladder
    GEMM of ccsd_r1_r2.h:275) on a bounded sample of V's rows at one BLAS thread
    and at all of them."""
    import numpy as np
    from oracle import ccsd as O
    ints = O.Integrals(**inp.blocks)
    stamps = []
    O.compute_ccsd(ints, inp.eps_occ, inp.eps_vir, max_iter=n_iter + 1, target_precision=1e-30,
                   callback=lambda *a: stamps.append(time.perf_counter()))
    per_it = [b - a for a, b in zip(stamps[:-1], stamps[1:])]
    dt = sum(per_it) / len(per_it)
    flops = O.ccsd_flops(inp.o, inp.v)
    threads = _blas_threads()
    # one-core sample: rows of the ladder GEMM, V (v^2 x v^2) @ tau (v^2 x o^2)
    o, v = inp.o, inp.v
    rows = min(v * v, 1536)
    Vs = np.ascontiguousarray(inp.blocks["Gabcd"].reshape(v * v, v * v)[:rows])
    T = np.random.default_rng(0).normal(0, 1e-2, (v * v, o * o))
    import contextlib
    try:
        import threadpoolctl
    except ImportError:
        threadpoolctl = None
    rates = {}
    for label, nt in [("one_core", 1), ("all_cores", threads)]:
        if threadpoolctl is None and nt != threads:
            continue
        lim = (threadpoolctl.threadpool_limits(limits=nt, user_api="blas") if threadpoolctl
               else contextlib.nullcontext())
        with lim:
            Vs[:64] @ T  # warm the pool
            t0 = time.perf_counter()
            Vs @ T
            rates[label] = 2.0 * rows * v * v * o * o / (time.perf_counter() - t0) / 1e9
    one_core_it = flops / (rates["one_core"] * 1e9) if "one_core" in rates else None
    return {"value": flops / dt / 1e12, "unit": "TFLOP/s", "cores": threads, "kind": "port",
            "seconds_per_iteration": round(dt, 3),
            "iterations_timed": len(per_it),
            "sample": f"oracle solver loop (numpy fp64, einsum on BLAS), {len(per_it)} full iterations "
                      f"(update+tau+residual+energy) at o={o} v={v}, {flops:.3e} FLOPs each",
            "one_core": {"gflops": round(rates.get("one_core", float("nan")), 2),
                         "all_cores_gflops": round(rates["all_cores"], 2),
                         "sample": f"pp-ladder GEMM rows 0..{rows - 1} ({rows}x{v * v} @ {v * v}x{o * o})",
                         "iteration_s_at_that_rate": round(one_core_it, 1) if one_core_it else None},
            **host_info()}


def _timed_iterations(c, args, label):
    """W untimed, then K timed iterations from the initial guess; one iteration
    = Jacobi/DIIS update + tau + residual + energy/error (the last call
    synchronises).  Then the same iterations again with per-contraction HIP-event
    timing.  Returns (ms per iteration, kernel times per iteration)."""
    c.init_guess()
    c.energy_error()
    for _ in range(args.warmup):
        c.update()
        c.residual()
        c.energy_error()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        c.update()
        c.residual()
        c.energy_error()
    ms = (time.perf_counter() - t0) * 1e3 / args.steps
    c.set_option("kernel_timing", 1)
    c.init_guess()
    c.energy_error()
    for _ in range(args.warmup + args.steps):
        c.update()
        c.residual()
        c.energy_error()
    kt = c.kernel_times()
    c.set_option("kernel_timing", 0)
    n_it = args.warmup + args.steps
    tot = sum(x["ms"] for x in kt.values()) / n_it
    log(f"{label}: {ms:.2f} ms/iteration; event-timed phases sum to {tot:.2f} ms/iteration")
    for k, x in sorted(kt.items(), key=lambda kv: -kv[1]["ms"])[:70]:
        log(f"   {k:24s} {x['ms'] / n_it:8.3f} ms/it  {x['calls'] / n_it:5.1f} calls/it"
            + (f"  {x['flops'] / max(1e-12, x['ms'] * 1e-3) / 1e12:7.2f} TF" if x["flops"] else ""))
    return ms, kt


def bench_ccsd(args):
    import numpy as np
    from mpqc_amd.ccsd import CCSD, Integrals
    from oracle.ccsd import ccsd_flops
    inp, setup = build_system(args.workload)
    o, v = inp.o, inp.v
    flops = ccsd_flops(o, v)
    ints = Integrals(**inp.blocks)
    forms = {}
    for prec in args.forms.split(","):
        c = CCSD(o, v, precision=prec, max_iter=args.max_iter)
        c.set_integrals(ints)
        c.set_orbital_energies(inp.eps_occ, inp.eps_vir)
        # converged solve (target precision 1e-8, as the workload specifies)
        E = c.compute_ccsd(target_precision=1e-8)
        rows = c.trace()
        log(f"{prec}: E_corr={E:.12f} after {len(rows)} iterations")
        ms, kt = _timed_iterations(c, args, prec)
        c.close()
        forms[prec] = {"E_corr": E, "iterations": len(rows), "ms_per_iteration": ms,
                       "tflops": flops / (ms * 1e-3) / 1e12,
                       "solve_iteration_ms": [round(r.seconds * 1e3, 3) for r in rows],
                       "kernels": {k: {"calls": x["calls"], "avg_ms": x["ms"] / max(1, x["calls"]),
                                       "tflops": x["flops"] / max(1e-12, x["ms"] * 1e-3) / 1e12}
                                   for k, x in kt.items()}}
    ref = forms[args.forms.split(",")[0]]
    for prec, f in forms.items():
        f["dE_vs_f64"] = f["E_corr"] - ref["E_corr"]
        f["speedup_vs_f64"] = ref["ms_per_iteration"] / f["ms_per_iteration"]
    # headline form: the fastest per iteration among those within 1 uEh of FP64 that
    # converge in at most 25% more iterations (a form that needs many more iterations
    # is not faster to the answer)
    it_ref = ref["iterations"]
    ok = [p for p, f in forms.items()
          if abs(f["dE_vs_f64"]) <= 1e-6 and f["iterations"] <= 1.25 * it_ref]
    head = min(ok, key=lambda p: forms[p]["ms_per_iteration"])
    hf = forms[head]
    nvs, nva = v * (v + 1) // 2, v * (v - 1) // 2
    if "r2:pp_ladder_sym" in hf["kernels"]:
        # the split forms run the ladder on pair-symmetric blocks: two GEMMs with half
        # the FLOPs of the full contraction; the roofline is the larger (V+) one's
        pp_tag = "r2:pp_ladder_sym"
        pp = hf["kernels"][pp_tag]
        pp_flops = 2.0 * nvs * o * o * nvs
        pp_desc = (f"pair-symmetric pp-ladder GEMM, V+ half (M=v(v+1)/2={nvs}, N=o^2={o * o}, "
                   f"K=v(v+1)/2) avg {pp['avg_ms']:.3f} ms")
        executed = flops - 2.0 * o * o * v ** 4 + 2.0 * o * o * (nvs * nvs + nva * nva)
    else:
        pp_tag = "r2:pp_ladder"
        pp = hf["kernels"].get(pp_tag, {"avg_ms": float("nan")})
        pp_flops = 2.0 * o * o * v ** 4
        pp_desc = f"pp-ladder GEMM (M=v^2, N=o^2, K=v^2) avg {pp['avg_ms']:.3f} ms"
        executed = flops
    pp_tf = pp_flops / (pp["avg_ms"] * 1e-3) / 1e12
    traffic, traffic_src = profiled_traffic(args.workload, head, pp_tag)
    log("CPU baseline (oracle residual)" if not args.no_cpu_baseline else "no CPU baseline")
    cpu = None if args.no_cpu_baseline else cpu_baseline_ccsd(inp)
    line = {
        "metric": "CCSD iter wall-time + TFLOP/s (frac MFMA peak), mixed vs FP64 at <=1 uEh",
        "value": round(hf["tflops"], 3),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(hf["ms_per_iteration"], 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": DTYPE[head],
        "data": "synthetic molecule (seeded geometry), RHF + AO->MO on the host",
        "config": {"workload": SYSTEMS[args.workload], "o": o, "v": v,
                   "algorithmic_flops_per_iteration": flops, "form": head,
                   # value = the reference's contraction FLOPs per second of wall time; the
                   # pair-symmetric ladder executes fewer
                   "executed_flops_per_iteration": executed,
                   "parallelism": "single-gpu"},
        "roofline": {"bound": "mfma", "achieved": round(pp_tf, 3),
                     "peak": PEAK[head], "unit": "TFLOP/s",
                     "frac": round(pp_tf / PEAK[head], 4), "traffic": traffic,
                     "traffic_source": traffic_src,
                     "kernel": pp_desc,
                     # the split forms issue MFMA_PRODUCTS matrix-core products per algorithmic FLOP
                     "mfma_products_per_flop": MFMA_PRODUCTS.get(head, 1),
                     "mfma_work_frac": round(pp_tf * MFMA_PRODUCTS.get(head, 1) / PEAK[head], 4),
                     "algorithmic_flops_per_launch": pp_flops},
        # per form: the figures north_star asks for each result (kernel tables go to stderr)
        "forms": {p: {"ms_per_iteration": round(f["ms_per_iteration"], 3),
                      "iterations": f["iterations"],
                      "tflops": round(f["tflops"], 2),
                      "E_corr": "%.12f" % f["E_corr"],
                      "dE_vs_f64": "%.3e" % f["dE_vs_f64"],
                      "speedup_vs_f64": round(f["speedup_vs_f64"], 3)}
                  for p, f in forms.items()},
        "setup": setup,
        "cpu_baseline": cpu,
    }
    if cpu:
        line["cpu_baseline"]["gpu_speedup"] = round(hf["tflops"] / cpu["value"], 1)
    if args.workload == "ccsd-h2o8" and not args.no_small_system:
        line["small_system"] = small_system_iteration(args)
    return line


def small_system_iteration(args):
    """The small-system configuration (H20 chain, o=10, v=90) in FP64: its
    iteration time beside the headline, since at that size launch count and
    small-tile efficiency, not the matrix cores, set the time."""
    from mpqc_amd.ccsd import CCSD, Integrals
    inp, _ = build_system("ccsd-h20")
    c = CCSD(inp.o, inp.v, precision="f64", max_iter=args.max_iter)
    c.set_integrals(Integrals(**inp.blocks))
    c.set_orbital_energies(inp.eps_occ, inp.eps_vir)
    E = c.compute_ccsd(target_precision=1e-8)
    n = len(c.trace())
    ms, _ = _timed_iterations(c, args, "h20 f64")
    c.close()
    return {"workload": SYSTEMS["ccsd-h20"], "form": "f64", "ms_per_iteration": round(ms, 3),
            "iterations": n, "E_corr": "%.12f" % E, "residual": "HIP graph replay"}


def bench_copy(args):
    """A plain device copy of known size: the reference point for scaling the
    rocprofv3 FETCH_SIZE / WRITE_SIZE counters to bytes."""
    import torch
    n = int(args.copy_gib * (1 << 30) / 8)
    x = torch.ones(n, dtype=torch.float64, device="cuda")
    y = torch.empty_like(x)
    for _ in range(args.warmup):
        y.copy_(x)
    torch.cuda.synchronize()
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    s.record()
    for _ in range(args.steps):
        y.copy_(x)
    e.record()
    torch.cuda.synchronize()
    ms = s.elapsed_time(e) / args.steps
    nbytes = 2 * n * 8
    return {"metric": "device copy bandwidth (counter calibration)", "value": nbytes / ms / 1e6,
            "unit": "GB/s", "ms_per_step": ms, "bytes_read_per_step": n * 8,
            "bytes_written_per_step": n * 8, "steps": args.steps, "warmup": args.warmup}


def _chain_sizes(count):
    """(o, v) of the seeded H-chain batch: n even uniform in [8, 32], spacing
    U[1.6, 2.0] bohr, cc-pVDZ (5 functions per H): o = n/2, v = 4.5 n."""
    from mpqc_amd.chem.molecule import h_chain_batch
    return [(len(m.symbols) // 2, 9 * len(m.symbols) // 2) for m in h_chain_batch(count=count, seed=3)]


def _context_doubles(o, v):
    """Device doubles one residual context holds (integrals, derived layouts,
    amplitudes, intermediates)."""
    ov, oo, vv = o * v, o * o, v * v
    return vv * vv + 3 * ov * vv + 35 * ov * ov + 10 * oo * ov + 3 * oo * oo + 64 * max(vv, ov, oo * oo, 4096)


def _synthetic_blocks(o, v, gen):
    """Seeded random integral blocks of the reference shapes on the device
    (Fock diagonals e_occ in [-1.5, -0.3], e_vir in [0.1, 3.0])."""
    import torch
    dev = "cuda"
    shapes = {"Fia": (o, v), "Fij": (o, o), "Fab": (v, v), "Gijab": (o, o, v, v),
              "Gijkl": (o, o, o, o), "Giajb": (o, v, o, v), "Giabc": (o, v, v, v),
              "Gijka": (o, o, o, v), "Gabcd": (v, v, v, v)}
    out = {}
    for name, shp in shapes.items():
        out[name] = 0.01 * torch.randn(shp, dtype=torch.float64, device=dev, generator=gen)
    eo = -0.3 - 1.2 * torch.rand(o, dtype=torch.float64, device=dev, generator=gen)
    ev = 0.1 + 2.9 * torch.rand(v, dtype=torch.float64, device=dev, generator=gen)
    out["Fij"] += torch.diag(eo)
    out["Fab"] += torch.diag(ev)
    return out


def bench_batched(args):
    """One residual for each of the seeded H chains, all molecules of a group in
    grouped launches (one hipGraph), groups sized to the HBM budget."""
    import ctypes
    import torch
    from mpqc_amd import _lib as L
    from mpqc_amd.batch import CCSDBatch
    from oracle.ccsd import ccsd_flops
    sizes = _chain_sizes(args.batch_count)
    budget = args.batch_mem_gib * (1 << 30) / 8
    order = sorted(range(len(sizes)), key=lambda k: sizes[k])
    groups, cur, cur_mem = [], [], 0.0
    for k in order:
        need = _context_doubles(*sizes[k])
        if cur and cur_mem + need > budget:
            groups.append(cur)
            cur, cur_mem = [], 0.0
        cur.append(k)
        cur_mem += need
    groups.append(cur)
    log(f"batched: {len(sizes)} chains (o {min(s[0] for s in sizes)}-{max(s[0] for s in sizes)}, "
        f"v {min(s[1] for s in sizes)}-{max(s[1] for s in sizes)}) in {len(groups)} groups")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    total_ms, total_flops, tune_s = 0.0, 0.0, 0.0
    stage_totals = {}
    for gi, grp in enumerate(groups):
        os_ = [sizes[k][0] for k in grp]
        vs_ = [sizes[k][1] for k in grp]
        with CCSDBatch(os_, vs_, precision=args.batch_precision) as B:
            for j, k in enumerate(grp):
                o, v = sizes[k]
                blocks = _synthetic_blocks(o, v, gen)
                for name, idx in L.INTEGRAL_IDS.items():
                    t = blocks[name].contiguous()
                    B._check(B.lib.mpqc_ccsd_batch_set_integral(B.h, j, idx, ctypes.c_void_p(t.data_ptr()),
                                                                L.LAYOUT_DENSE, L.MEM_DEVICE))
                t1 = 0.01 * torch.randn((v, o), dtype=torch.float64, device="cuda", generator=gen)
                t2 = 0.01 * torch.randn((v, v, o, o), dtype=torch.float64, device="cuda", generator=gen)
                B._check(B.lib.mpqc_ccsd_batch_set_amplitudes(B.h, j, ctypes.c_void_p(t1.data_ptr()),
                                                              ctypes.c_void_p(t2.data_ptr()),
                                                              L.LAYOUT_DENSE, L.MEM_DEVICE))
                del blocks, t1, t2
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            B.tune(reps=1)
            tune_s += time.perf_counter() - t0
            ms = B.time(reps=args.steps)
            B.time_stages(reps=1)
            for st in B.stages():
                agg = stage_totals.setdefault(st["tag"], {"ms": 0.0, "flops": 0.0, "kind": st["kind"]})
                agg["ms"] += st["ms"]
                agg["flops"] += st["flops"]
            fl = sum(ccsd_flops(o, v) for o, v in zip(os_, vs_))
            log(f"group {gi}: {len(grp)} chains, {ms:.2f} ms per batched residual, "
                f"{fl / (ms * 1e-3) / 1e12:.2f} TFLOP/s")
            total_ms += ms
            total_flops += fl
        torch.cuda.empty_cache()
    tflops = total_flops / (total_ms * 1e-3) / 1e12
    pp = stage_totals.get("r2:pp_ladder", {"ms": float("nan"), "flops": float("nan")})
    pp_tf = pp["flops"] / (pp["ms"] * 1e-3) / 1e12
    top = sorted(stage_totals.items(), key=lambda kv: -kv[1]["ms"])[:12]
    cpu = None
    if not args.no_cpu_baseline:
        cpu = cpu_baseline_batched(sizes)
    peak = PEAK[args.batch_precision]
    line = {
        "metric": "batched CCSD residuals: wall time + TFLOP/s (frac MFMA peak)",
        "value": round(tflops, 3), "unit": "TFLOP/s", "n_gpus": 1, "steps": args.steps,
        "warmup": 1, "ms_per_step": round(total_ms, 3), "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": args.batch_precision,
        "data": "synthetic integrals of the chains' shapes (torch CUDA generator seed 3); "
                "chain sizes from the seeded generator (numpy PCG64 seed 3)",
        "config": {"workload": f"{len(sizes)} H chains n=8..32 cc-pVDZ (o=n/2, v=4.5n), one residual each",
                   "groups": len(groups), "algorithmic_flops": total_flops, "parallelism": "single-gpu",
                   "graph": "one hipGraph per group", "autotune_s": round(tune_s, 2)},
        "roofline": {"bound": "mfma", "achieved": round(pp_tf, 3), "peak": peak, "unit": "TFLOP/s",
                     "frac": round(pp_tf / peak, 4), "traffic": None,
                     "kernel": "grouped pp-ladder contraction over all chains"},
        "stages_top": {k: {"ms": round(v_["ms"], 3), "kind": v_["kind"],
                           "tflops": round(v_["flops"] / max(v_["ms"], 1e-9) / 1e9, 2)}
                       for k, v_ in top},
        "cpu_baseline": cpu,
    }
    return line


def cpu_baseline_batched(sizes, budget_s=10.0):
    """Oracle residuals (numpy/OpenBLAS) of the smallest chains of the batch, as
    many as fit in about budget_s seconds."""
    import numpy as np
    from oracle import ccsd as O
    rng = np.random.default_rng(3)
    done, flops, t_used = 0, 0.0, 0.0
    for o, v in sorted(sizes):
        blocks = {"Fia": (o, v), "Fij": (o, o), "Fab": (v, v), "Gijab": (o, o, v, v), "Gijkl": (o, o, o, o),
                  "Giajb": (o, v, o, v), "Giabc": (o, v, v, v), "Gijka": (o, o, o, v), "Gabcd": (v, v, v, v)}
        b = {k: 0.01 * rng.normal(size=s) for k, s in blocks.items()}
        ints = O.Integrals(**b)
        t1 = 0.01 * rng.normal(size=(v, o))
        t2 = 0.01 * rng.normal(size=(v, v, o, o))
        t0 = time.perf_counter()
        tau = O.make_tau(t1, t2)
        O.cs_ccsd_r1(t1, t2, tau, ints)
        O.cs_ccsd_r2(t1, t2, tau, ints)
        t_used += time.perf_counter() - t0
        flops += O.ccsd_flops(o, v)
        done += 1
        if t_used > budget_s:
            break
    threads = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))
    return {"value": flops / t_used / 1e12, "unit": "TFLOP/s", "cores": threads, "kind": "port",
            "sample": f"oracle residuals of the {done} smallest chains ({flops:.3e} FLOPs in {t_used:.1f} s)"}


def bench_adjoint(args):
    """(H2O)6 cc-pVDZ: converged CCSD, Lambda equations and dE/dF for a field
    along z (f + F mu, F = 1e-4 a.u., fixed orbitals), checked against a
    four-point central difference of the converged energy."""
    import numpy as np
    import torch
    from mpqc_amd.adjoint import ccsd_energy, mo_dipole_blocks
    from mpqc_amd.ccsd import CCSD, Integrals
    from mpqc_amd.chem.molecule import water_cluster
    from mpqc_amd.chem.scf import rhf
    from mpqc_amd.chem.mo import ccsd_integrals
    from oracle.ccsd import ccsd_flops
    mol = water_cluster((3, 2, 1), seed=5)
    t0 = time.perf_counter()
    scf = rhf(mol, "cc-pVDZ")
    inp = ccsd_integrals(scf, frozen_core=False)
    mu = mo_dipole_blocks(scf, axis=2)
    log(f"adjoint (H2O)6: o={inp.o} v={inp.v}, set-up {time.perf_counter() - t0:.1f}s")
    from mpqc_amd.adjoint import last_info
    F0 = 1e-4
    # (amplitude, Lambda) targets in the solver's error measure |r| / (size1 + size2), which
    # divides by ~1e7 elements here: FP64 goes to 1e-14 / 1e-16 (per-element residuals
    # ~1e-11); the FP32 contractions' noise floor is near 1e-12 in this measure
    precs = {"f64": (1e-14, 1e-16), "f32": (1e-11, 1e-12)}

    def blocks_at(Fv):
        b = dict(inp.blocks)
        for n in ("Fia", "Fij", "Fab"):
            b[n] = inp.blocks[n] + Fv * mu[n]
        return b

    forms = {}
    fd_f64 = None
    for form in ("f64", "f32"):
        prec, lprec = precs[form]
        F = torch.tensor(F0, dtype=torch.float64, requires_grad=True)
        tb = {n: torch.from_numpy(np.array(a)) for n, a in inp.blocks.items()}
        for n in ("Fia", "Fij", "Fab"):
            tb[n] = tb[n] + F * torch.from_numpy(mu[n])
        torch.cuda.synchronize()
        t1 = time.perf_counter()
        E = ccsd_energy(tb, inp.eps_occ, inp.eps_vir, precision=form, target_precision=prec,
                        lambda_precision=lprec, max_iter=200)
        t2 = time.perf_counter()
        E.backward()
        t3 = time.perf_counter()
        grad = F.grad.item()

        def e_at(Fv):
            with CCSD(inp.o, inp.v, precision=form, max_iter=200) as c:
                c.set_integrals(Integrals(**blocks_at(Fv)))
                c.set_orbital_energies(inp.eps_occ, inp.eps_vir)
                return c.compute_ccsd(target_precision=prec)

        info = dict(last_info)
        h = 5e-4
        fd = (8 * (e_at(F0 + h) - e_at(F0 - h)) - (e_at(F0 + 2 * h) - e_at(F0 - 2 * h))) / (12 * h)
        if form == "f64":
            fd_f64 = fd
        forms[form] = {"E_corr": E.item(), "dE_dF_adjoint": grad, "dE_dF_central_difference": fd,
                       "rel_err": abs(grad - fd) / abs(fd),
                       "rel_err_vs_f64_difference": abs(grad - fd_f64) / abs(fd_f64),
                       "solve_s": round(t2 - t1, 3), "lambda_and_gradient_s": round(t3 - t2, 3), **info}
        log(f"{form}: dE/dF adjoint {grad:.10e} difference {fd:.10e} rel {abs(grad - fd) / abs(fd):.2e} "
            f"(vs f64 difference {abs(grad - fd_f64) / abs(fd_f64):.2e}); solve {t2 - t1:.2f}s "
            f"({info.get('ccsd_iterations')} it), Lambda + gradient {t3 - t2:.2f}s "
            f"({info.get('lambda_iterations')} it)")
    f = forms["f64"]
    line = {
        "metric": "adjoint dE/dF vs central differences (relative error) and Lambda time",
        "value": f["rel_err"], "unit": "relative error", "n_gpus": 1, "steps": 1, "warmup": 0,
        "ms_per_step": round(1e3 * f["lambda_and_gradient_s"], 3), "higher_is_better": False,
        "scaling": "weak", "vs_baseline": None, "dtype": "f64",
        "data": "(H2O)6 seeded geometry, RHF + AO->MO on the host, field along z",
        "config": {"workload": "(H2O)6 cc-pVDZ o=30 v=114, F_z = 1e-4 a.u.", "o": inp.o, "v": inp.v,
                   "algorithmic_flops_per_iteration": ccsd_flops(inp.o, inp.v),
                   "parallelism": "single-gpu"},
        "forms": forms,
        "roofline": None,
        "cpu_baseline": None,
    }
    return line


def bench_df(args):
    """Density-fitted CCSD (method "df", reduced_abcd_memory) on (H2O)8 with
    the cc-pVDZ orbital basis and cc-pVDZ as the fitting basis (the pairing of
    the reference's DF validation input, orbital basis 6-31G / fitting basis
    cc-pVDZ, moved up one orbital basis): RI-RHF and the DF MO factors on the
    host, then converged solves and K timed iterations in the forms of --forms
    (FP64 and the 16-bit split forms, whose (ab|cd) blocks go through planes),
    beside the standard FP64 residual on the same (DF four-index) integrals."""
    import numpy as np
    from mpqc_amd.ccsd import CCSD, Integrals
    from mpqc_amd.chem.df import df_ccsd_integrals, ri_rhf
    from mpqc_amd.chem.molecule import water_cluster
    from oracle.ccsd import ccsd_flops
    mol = water_cluster((2, 2, 2), seed=4)
    t0 = time.perf_counter()
    d = ri_rhf(mol, "cc-pVDZ", "cc-pVDZ")
    t1 = time.perf_counter()
    inp = df_ccsd_integrals(d, frozen_core=False)
    t2 = time.perf_counter()
    o, v, Q = inp.o, inp.v, inp.naux
    log(f"df-h2o8: RI-RHF E={d.scf.energy:.10f} ({t1 - t0:.1f}s), DF MO factors o={o} v={v} "
        f"naux={Q} ({t2 - t1:.1f}s)")
    del d
    forms = {}
    for prec in [p for p in args.forms.split(",") if p in ("f64", "f32", "f16x3", "bf16x3")] or ["f64"]:
        c = CCSD(o, v, precision=prec, max_iter=args.max_iter)
        c.set_df_basis(Q)
        c.set_integrals(inp.df_blocks())
        c.set_orbital_energies(inp.base.eps_occ, inp.base.eps_vir)
        E = c.compute_ccsd(target_precision=1e-8)
        n_rows = len(c.trace())
        log(f"df {prec}: E_corr={E:.12f} after {n_rows} iterations")
        ms, kt = _timed_iterations(c, args, f"df {prec}")
        c.close()
        n_it = args.warmup + args.steps
        exec_flops = sum(x["flops"] for x in kt.values()) / n_it
        forms[prec] = {"E_corr": E, "iterations": n_rows, "ms_per_iteration": ms,
                       "executed_contraction_flops": exec_flops,
                       "tflops_executed": exec_flops / (ms * 1e-3) / 1e12,
                       "kernels": {k: {"calls": x["calls"], "avg_ms": x["ms"] / max(1, x["calls"]),
                                       "tflops": x["flops"] / max(1e-12, x["ms"] * 1e-3) / 1e12}
                                   for k, x in kt.items()}}
    # the standard residual on the same integrals (Gabcd, Giabc from the same factors)
    c = CCSD(o, v, precision="f64", max_iter=args.max_iter)
    c.set_integrals(Integrals(**inp.base.blocks))
    c.set_orbital_energies(inp.base.eps_occ, inp.base.eps_vir)
    E_std = c.compute_ccsd(target_precision=1e-8)
    ms_std, _ = _timed_iterations(c, args, "standard f64 on the DF integrals")
    c.close()
    ref = forms.get("f64", next(iter(forms.values())))
    for f in forms.values():
        f["dE_vs_f64"] = f["E_corr"] - ref["E_corr"]
        f["solve_ms"] = f["iterations"] * f["ms_per_iteration"]
    # headline form: the shortest solve (iterations x time per iteration) within 1 uEh of FP64
    head = min([p for p, f in forms.items() if abs(f["dE_vs_f64"]) <= 1e-6],
               key=lambda p: forms[p]["solve_ms"])
    hf = forms[head]
    lad = hf["kernels"].get("r2:df_pp_ladder", {"avg_ms": float("nan"), "tflops": float("nan")})
    cpu = None
    if not args.no_cpu_baseline:
        from oracle import ccsd as O
        from oracle import ccsd_df as D
        ints = D.DFIntegrals(**inp.df_blocks())
        t1a = O.jacobi_update_t1(ints.Fia.T, inp.base.eps_occ, inp.base.eps_vir)
        t2a = O.jacobi_update_t2(ints.Gijab.transpose(2, 3, 0, 1), inp.base.eps_occ, inp.base.eps_vir)
        tau = O.make_tau(t1a, t2a)
        ta = time.perf_counter()
        D.cs_ccsd_r1_df(t1a, t2a, tau, ints)
        D.cs_ccsd_r2_df(t1a, t2a, tau, ints)
        dt = time.perf_counter() - ta
        threads = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))
        cpu = {"value": dt * 1e3, "unit": "ms per residual", "cores": threads, "kind": "port",
               "sample": f"one DF oracle residual (numpy/OpenBLAS fp64 einsum) at o={o} v={v} naux={Q}, "
                         "first-iteration amplitudes"}
    line = {
        "metric": "DF-CCSD iteration wall-time (method df, reduced_abcd_memory)",
        "value": round(hf["ms_per_iteration"], 3), "unit": "ms/iteration", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(hf["ms_per_iteration"], 3),
        "higher_is_better": False, "scaling": "weak", "vs_baseline": None,
        "dtype": DTYPE[head],
        "data": "synthetic molecule (seeded geometry), RI-RHF + DF MO factors on the host",
        "config": {"workload": "(H2O)8 cc-pVDZ orbitals, cc-pVDZ fitting basis, method df", "o": o,
                   "v": v, "naux": Q, "form": head, "parallelism": "single-gpu",
                   "standard_algorithmic_flops_per_iteration": ccsd_flops(o, v)},
        "roofline": {"bound": "mfma", "achieved": round(lad["tflops"], 3), "peak": PEAK[head],
                     "unit": "TFLOP/s", "frac": round(lad["tflops"] / PEAK[head], 4), "traffic": None,
                     "kernel": f"DF pp-ladder GEMM per (ab|cd) block (M=nb v, N=o^2, K=v^2) "
                               f"avg {lad['avg_ms']:.3f} ms",
                     "mfma_products_per_flop": MFMA_PRODUCTS.get(head, 1),
                     "mfma_work_frac": round(lad["tflops"] * MFMA_PRODUCTS.get(head, 1) / PEAK[head], 4)},
        "forms": {p: {"ms_per_iteration": round(f["ms_per_iteration"], 3), "iterations": f["iterations"],
                      "tflops_executed": round(f["tflops_executed"], 2), "E_corr": "%.12f" % f["E_corr"],
                      "dE_vs_f64": "%.3e" % f["dE_vs_f64"]} for p, f in forms.items()},
        "standard_f64_same_integrals": {"E_corr": E_std, "ms_per_iteration": round(ms_std, 3),
                                        "dE_vs_df_f64": E_std - ref["E_corr"]},
        "setup": {"ri_rhf_s": round(t1 - t0, 2), "df_factors_s": round(t2 - t1, 2)},
        "cpu_baseline": cpu,
    }
    return line


def _device_copy(hip, a):
    import ctypes
    import numpy as np
    a = np.ascontiguousarray(a, dtype=np.float64)
    p = ctypes.c_void_p()
    if hip.hipMalloc(ctypes.byref(p), a.nbytes) != 0:
        raise MemoryError("hipMalloc failed")
    if hip.hipMemcpy(p, a.ctypes.data_as(ctypes.c_void_p), a.nbytes, 1) != 0:
        raise RuntimeError("hipMemcpy failed")
    return p


def bench_transform(args):
    """AO -> MO transform on the device (LCAOFactory::compute4): (H2O)8 cc-pVDZ,
    nbf = 192, every orbital active (o=40, v=152).  The AO integrals, Fock matrix
    and coefficients are resident in HBM before the timed region; one step = one
    mpqc_ccsd_transform_ao call (four quarter-transform GEMMs, six block
    extractions, the Fock blocks).  The density-fitted transform (cc-pVDZ as the
    fitting basis, naux = 192) is timed the same way."""
    import ctypes
    import numpy as np
    from mpqc_amd import _lib as L
    from mpqc_amd.ccsd import CCSD
    from mpqc_amd.chem.basis import BasisSet
    from mpqc_amd.chem.df import inv_sqrt
    from mpqc_amd.chem.molecule import water_cluster
    from mpqc_amd.chem.scf import rhf
    mol = water_cluster((2, 2, 2), seed=4)
    t0 = time.perf_counter()
    scf = rhf(mol, "cc-pVDZ")
    log(f"transform-h2o8: RHF in {time.perf_counter() - t0:.1f}s")
    n = scf.F.shape[0]
    Ci, Ca = scf.C[:, :scf.ndocc], scf.C[:, scf.ndocc:]
    o, v = Ci.shape[1], Ca.shape[1]
    nmo = o + v
    L.load()
    hip = ctypes.CDLL("libamdhip64.so.7")
    hip.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    hip.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    hip.hipFree.argtypes = [ctypes.c_void_p]
    t0 = time.perf_counter()
    dev = [_device_copy(hip, a) for a in (scf.eri, scf.F, Ci, Ca)]
    h2d_s = time.perf_counter() - t0
    log(f"AO integrals to HBM: {scf.eri.nbytes / 2**30:.2f} GiB in {h2d_s:.2f}s (pageable host memory)")
    # quarter transforms of the occupied / virtual combinations that some block needs
    flops = 2.0 * (n**4 * nmo + n**3 * (o * nmo + v * v) + n**2 * (o * o * nmo + o * v * nmo + v**3)
                   + n * (o**3 * nmo + 2 * o * o * v * v + o * v**3 + v**4))
    res = {}
    with CCSD(o, v) as c:
        for _ in range(args.warmup):
            c._check(c.lib.mpqc_ccsd_transform_ao(c.ctx, n, *dev, L.MEM_DEVICE))
        t0 = time.perf_counter()
        for _ in range(args.steps):
            c._check(c.lib.mpqc_ccsd_transform_ao(c.ctx, n, *dev, L.MEM_DEVICE))
        ms = (time.perf_counter() - t0) * 1e3 / args.steps
        res["ao"] = {"ms": ms, "tflops": flops / (ms * 1e-3) / 1e12}
        log(f"transform_ao: {ms:.2f} ms per call, {flops / (ms * 1e-3) / 1e12:.1f} TFLOP/s")
        Gijab_gpu = c.get_integral("Gijab")
    for p in dev:
        hip.hipFree(p)
    # density-fitted transform
    dfbs = BasisSet("cc-pVDZ", mol)
    B = scf.basis.eri3(dfbs)
    Lm = inv_sqrt(dfbs.eri2())
    Q = B.shape[0]
    devd = [_device_copy(hip, a) for a in (B, Lm, scf.F, Ci, Ca)]
    dflops = 2.0 * (Q * Q * n * n + Q * n * n * nmo + Q * n * nmo * nmo
                    + Q * (o * v) ** 2 + Q * o**4 + 2 * Q * o**3 * v + Q * o * o * v * v)
    with CCSD(o, v) as c:
        c.set_df_basis(Q)
        for _ in range(args.warmup):
            c._check(c.lib.mpqc_ccsd_transform_df(c.ctx, n, *devd, L.MEM_DEVICE))
        t0 = time.perf_counter()
        for _ in range(args.steps):
            c._check(c.lib.mpqc_ccsd_transform_df(c.ctx, n, *devd, L.MEM_DEVICE))
        dms = (time.perf_counter() - t0) * 1e3 / args.steps
        res["df"] = {"ms": dms, "tflops": dflops / (dms * 1e-3) / 1e12, "naux": Q}
        log(f"transform_df: {dms:.2f} ms per call")
    for p in devd:
        hip.hipFree(p)
    cpu = None
    if not args.no_cpu_baseline:
        from oracle import ao2mo as A
        # bounded sample: the Gijab block alone (4 quarter transforms with o, v columns)
        ta = time.perf_counter()
        x = np.einsum("sp,sabc->pabc", Ci, scf.eri, optimize=True)
        x = np.einsum("ar,pabc->prbc", Ca, x, optimize=True)
        x = np.einsum("bq,prbc->prqc", Ci, x, optimize=True)
        x = np.einsum("cs,prqc->prqs", Ca, x, optimize=True)
        dt = time.perf_counter() - ta
        sflops = 2.0 * (n**4 * o + n**3 * o * v + n**2 * o * v * o + n * o * v * o * v)
        err = float(np.abs(x.transpose(0, 2, 1, 3) - Gijab_gpu).max())
        threads = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))
        cpu = {"value": sflops / dt / 1e12, "unit": "TFLOP/s", "cores": threads, "kind": "port",
               "seconds": round(dt, 3),
               "sample": f"the Gijab block by the oracle's quarter transforms (numpy einsum), "
                         f"{sflops:.3e} FLOPs; max |GPU - oracle| = {err:.1e}"}
        _ = A  # the oracle module restates the same four steps for all blocks
    line = {
        "metric": "AO->MO integral transform time (compute4) on one GPU",
        "value": round(res["ao"]["ms"], 3), "unit": "ms per transform", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(res["ao"]["ms"], 3),
        "higher_is_better": False, "scaling": "weak", "vs_baseline": None, "dtype": "f64",
        "data": "synthetic molecule (seeded geometry), RHF AO integrals resident in HBM",
        "config": {"workload": "(H2O)8 cc-pVDZ AO->MO, nbf=192, o=40, v=152 (all nine blocks + Fock)",
                   "nbf": n, "o": o, "v": v, "transform_flops": flops, "parallelism": "single-gpu",
                   "ao_h2d_seconds_pageable": round(h2d_s, 3)},
        "roofline": {"bound": "mfma", "achieved": round(res["ao"]["tflops"], 3), "peak": PEAK["f64"],
                     "unit": "TFLOP/s", "frac": round(res["ao"]["tflops"] / PEAK["f64"], 4), "traffic": None,
                     "kernel": "whole transform_ao call (quarter transforms of the occupied / virtual "
                               "combinations that the blocks need), their FLOPs"},
        "df_transform": {k: (round(x, 4) if isinstance(x, float) else x) for k, x in res["df"].items()},
        "cpu_baseline": cpu,
    }
    return line


def bench_triples(args):
    """CCSD(T) on one GPU: (H2O)6 or (H2O)8 cc-pVDZ, FP64 CCSD converged to 1e-8,
    then one (T) evaluation (mpqc_ccsd_triples) per step from the resident
    amplitudes and integrals."""
    from mpqc_amd.ccsd import CCSD, Integrals
    from oracle.ccsd_t import ccsd_t_flops
    name = "ccsd-h2o8" if args.workload == "triples-h2o8" else "ccsd-h2o6"
    inp, setup = build_system(name)
    o, v = inp.o, inp.v
    with CCSD(o, v, max_iter=args.max_iter) as c:
        c.set_integrals(Integrals(**inp.blocks))
        c.set_orbital_energies(inp.eps_occ, inp.eps_vir)
        E = c.compute_ccsd(target_precision=1e-8)
        log(f"{name}: E_CCSD={E:.12f}; (T)")
        for _ in range(args.warmup):
            c.triples()
        times, ets = [], []
        for _ in range(args.steps):
            t0 = time.perf_counter()
            et, dev_s = c.triples()
            times.append(time.perf_counter() - t0)
            ets.append(et)
            log(f"  (T) = {et:.12e} in {times[-1]:.3f}s (device {dev_s:.3f}s)")
        # the same (T) with the W GEMMs on fp16 hi+lo planes
        c.set_option("precision", 3)
        t0 = time.perf_counter()
        et16, _ = c.triples()
        sec16 = time.perf_counter() - t0
        log(f"  f16x3 (T) = {et16:.12e} in {sec16:.3f}s (vs f64 {et16 - ets[-1]:+.2e} Eh)")
    flops = ccsd_t_flops(o, v)
    sec = sum(times) / len(times)
    cpu = None
    if not args.no_cpu_baseline:
        import numpy as np
        from mpqc_amd.chem.mo import ccsd_integrals
        from mpqc_amd.chem.molecule import water_cluster
        from mpqc_amd.chem.scf import rhf
        from oracle import ccsd as O
        from oracle.ccsd_t import ccsd_t_straight
        # bounded sample: the oracle's straight (T) for one water monomer of the
        # same generator (its t3 fits in host memory), at MP2 amplitudes
        small = ccsd_integrals(rhf(water_cluster((1, 1, 1), seed=4), "cc-pVDZ"))
        b = small.blocks
        t1 = O.jacobi_update_t1(b["Fia"].T, small.eps_occ, small.eps_vir)
        t2 = O.jacobi_update_t2(b["Gijab"].transpose(2, 3, 0, 1), small.eps_occ, small.eps_vir)
        ta = time.perf_counter()
        ccsd_t_straight(t1, t2, b["Gijab"], b["Giabc"], b["Gijka"], small.eps_occ, small.eps_vir)
        dt = time.perf_counter() - ta
        sf = ccsd_t_flops(small.o, small.v)
        threads = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))
        cpu = {"value": sf / dt / 1e12, "unit": "TFLOP/s", "cores": threads, "kind": "port",
               "seconds": round(dt, 3),
               "sample": f"the oracle's straight (T) (numpy einsum, full t3 in memory) for one water "
                         f"(o={small.o}, v={small.v}), {sf:.3e} FLOPs"}
    line = {
        "metric": "CCSD(T) triples time on one GPU",
        "value": round(sec, 4), "unit": "s per (T)", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(sec * 1e3, 3), "higher_is_better": False,
        "scaling": "weak", "vs_baseline": None, "dtype": "f64",
        "data": "synthetic molecule (seeded geometry), RHF + AO->MO on the host, converged FP64 CCSD",
        "config": {"workload": f"(T) for {SYSTEMS[name]}", "o": o, "v": v, "triples_flops": flops,
                   "parallelism": "single-gpu", "E_CCSD": E, "E_T": ets[-1]},
        "roofline": {"bound": "mfma", "achieved": round(flops / sec / 1e12, 3), "peak": PEAK["f64"],
                     "unit": "TFLOP/s", "frac": round(flops / sec / 1e12 / PEAK["f64"], 4), "traffic": None,
                     "kernel": "whole (T): 2 o^3 v^4 + 2 o^4 v^3 GEMM FLOPs over the wall time"},
        "f16x3": {"seconds": round(sec16, 4), "E_T": et16, "dE_T_vs_f64": et16 - ets[-1],
                  "speedup_vs_f64": round(sec / sec16, 3)},
        "setup": setup,
        "cpu_baseline": cpu,
    }
    return line


def bench_eom(args):
    """EOM-EE-CCSD on one GPU: (H2O)6 cc-pVDZ, FP64 CCSD converged to 1e-10, then the
    four lowest singlets to 1e-9 (the settings of the reference's h2o-eom-ccsd
    inputs: property precision 1e-9, CCSD at 0.1 of it, 8 vectors per root)."""
    import numpy as np
    from mpqc_amd.ccsd import CCSD, Integrals
    name = "ccsd-h2o6"
    inp, setup = build_system(name)
    o, v = inp.o, inp.v
    n_roots, conv = 4, 1e-9
    with CCSD(o, v, precision="f64", max_iter=args.max_iter) as c:
        c.set_integrals(Integrals(**inp.blocks))
        c.set_orbital_energies(inp.eps_occ, inp.eps_vir)
        E = c.compute_ccsd(target_precision=0.1 * conv)
        log(f"{name}: E_CCSD={E:.12f}; EOM-EE-CCSD, {n_roots} singlets")
        for _ in range(args.warmup):
            c.eom_ee(n_roots, target_precision=conv, max_iter=100)
        times, roots = [], None
        for _ in range(args.steps):
            t0 = time.perf_counter()
            w, it = c.eom_ee(n_roots, target_precision=conv, max_iter=100)
            times.append(time.perf_counter() - t0)
            roots = w
            nprod, psec = c.eom_stats()
            log(f"  roots {np.array2string(w, precision=10)} in {times[-1]:.3f}s, {it} iterations, "
                f"{nprod} J^T products, {1e3 * psec / nprod:.2f} ms each")
    sec = sum(times) / len(times)
    # the sweep's products from o^4 v^2 up: the ladder on symmetric pairs, two adjoints of each ring and of
    # the hole-hole ladder, one of each contraction of amplitudes with integrals
    flops_product = 1.0 * o**2 * v**4 + 16.0 * o**3 * v**3 + 6.0 * o**4 * v**2
    per_product = psec / nprod
    cpu = None
    if not args.no_cpu_baseline:
        from oracle import ccsd as O
        ints = O.Integrals(**inp.blocks)
        t1 = O.jacobi_update_t1(ints.Fia.T, inp.eps_occ, inp.eps_vir)
        t2 = O.jacobi_update_t2(ints.Gijab.transpose(2, 3, 0, 1), inp.eps_occ, inp.eps_vir)
        rng = np.random.default_rng(0)
        d1, d2 = rng.normal(size=t1.shape), rng.normal(size=t2.shape)
        h = 1e-5
        ta = time.perf_counter()
        for sgn in (1.0, -1.0):  # one Jacobian-vector product by central differences
            a1, a2 = t1 + sgn * h * d1, t2 + sgn * h * d2
            tau = O.make_tau(a1, a2)
            O.cs_ccsd_r1(a1, a2, tau, ints)
            O.cs_ccsd_r2(a1, a2, tau, ints)
        dt = time.perf_counter() - ta
        threads = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))
        cpu = {"value": round(dt, 3), "unit": "s per Jacobian product", "cores": threads, "kind": "port",
               "gpu_seconds_per_product": round(per_product, 5),
               "sample": f"one Jacobian-vector product of the oracle residual by central differences "
                         f"(two numpy/OpenBLAS fp64 residuals) at o={o} v={v}"}
    line = {
        "metric": "EOM-EE-CCSD time (4 singlets) on one GPU",
        "value": round(sec, 4), "unit": "s per EOM-EE-CCSD", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(sec * 1e3, 3), "higher_is_better": False,
        "scaling": "weak", "vs_baseline": None, "dtype": "f64",
        "data": "synthetic molecule (seeded geometry), RHF + AO->MO on the host, converged FP64 CCSD",
        "config": {"workload": f"EOM-EE-CCSD singlets for {SYSTEMS[name]}", "o": o, "v": v,
                   "n_roots": n_roots, "convergence": conv, "max_vector": 8, "guess": "CIS",
                   "parallelism": "single-gpu",
                   "E_CCSD": E, "singlets": [float(x) for x in roots], "jt_products": nprod,
                   "jt_product_ms": round(1e3 * per_product, 3), "jt_product_flops": flops_product},
        "roofline": {"bound": "mfma", "achieved": round(flops_product / per_product / 1e12, 3),
                     "peak": PEAK["f64"], "unit": "TFLOP/s",
                     "frac": round(flops_product / per_product / 1e12 / PEAK["f64"], 4), "traffic": None,
                     "kernel": "whole J^T product (reverse sweep of the residual), FLOPs of its products from "
                               "o^4 v^2 up over its event-timed duration"},
        "setup": setup,
        "cpu_baseline": cpu,
    }
    return line


def bench_direct(args):
    """AO integral-direct CCSD (method "direct") on one GPU: (H2O)8 cc-pVDZ, FP64,
    AO integrals resident in HBM; a converged solve, then timed iterations with the
    U = (pq|rs) [Ca tau Ca^T] GEMM per iteration, beside the standard FP64 solve."""
    from mpqc_amd.ccsd import CCSD, Integrals
    from mpqc_amd.chem.molecule import water_cluster
    from mpqc_amd.chem.scf import rhf
    from mpqc_amd.chem.mo import ccsd_integrals
    from oracle.ccsd import ccsd_flops
    t0 = time.perf_counter()
    scf = rhf(water_cluster((2, 2, 2), seed=4), "cc-pVDZ")
    inp = ccsd_integrals(scf, frozen_core=False)
    nbf = scf.eri.shape[0]
    Ci, Ca = scf.C[:, :scf.ndocc], scf.C[:, scf.ndocc:]
    o, v = inp.o, inp.v
    log(f"direct (H2O)8: nbf={nbf} o={o} v={v}, set-up {time.perf_counter() - t0:.1f}s")
    blocks = {k: a for k, a in inp.blocks.items() if k != "Gabcd"}
    with CCSD(o, v, precision="f64", max_iter=args.max_iter) as c:
        c.set_integrals(blocks)
        ta = time.perf_counter()
        c.set_direct_ao(scf.eri, Ci, Ca)
        upload_s = time.perf_counter() - ta
        c.set_orbital_energies(inp.eps_occ, inp.eps_vir)
        E = c.compute_ccsd(target_precision=1e-8)
        n_it = len(c.trace())
        log(f"direct: E_corr={E:.12f} after {n_it} iterations")
        ms, kt = _timed_iterations(c, args, "direct f64")
    with CCSD(o, v, precision="f64", max_iter=args.max_iter) as c:
        c.set_integrals(Integrals(**inp.blocks))
        c.set_orbital_energies(inp.eps_occ, inp.eps_vir)
        E_std = c.compute_ccsd(target_precision=1e-8)
        ms_std, _ = _timed_iterations(c, argparse.Namespace(steps=args.steps, warmup=args.warmup), "standard f64")
    n_kt = args.warmup + args.steps
    u = kt["u:ao_eri_tau"]
    u_flops = 2.0 * nbf ** 4 * o * o
    u_ms = u["ms"] / u["calls"]
    cpu = None
    if not args.no_cpu_baseline:
        import numpy as np
        from oracle.ccsd_direct import compute_u2_u11
        rng = np.random.default_rng(0)
        t1 = rng.normal(0, 0.01, (v, o))
        t2 = rng.normal(0, 0.01, (v, v, o, o))
        tb = time.perf_counter()
        compute_u2_u11(t2, t1, scf.eri, Ca)
        dt = time.perf_counter() - tb
        threads = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))
        cpu = {"value": round(u_flops / dt / 1e12, 3), "unit": "TFLOP/s", "cores": threads, "kind": "port",
               "seconds": round(dt, 3),
               "sample": f"the oracle's compute_u2_u11 (numpy einsum over the AO integrals) at the same size, "
                         f"{u_flops:.3e} FLOPs in its U contraction"}
    line = {
        "metric": "direct-method CCSD iteration time on one GPU",
        "value": round(ms, 3), "unit": "ms per iteration", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(ms, 3), "higher_is_better": False,
        "scaling": "weak", "vs_baseline": None, "dtype": "f64",
        "data": "synthetic molecule (seeded geometry), RHF + AO integrals on the host",
        "config": {"workload": f"method direct for {SYSTEMS['ccsd-h2o8']}", "nbf": nbf, "o": o, "v": v,
                   "parallelism": "single-gpu", "E_corr": E, "E_corr_standard": E_std,
                   "dE_vs_standard": E - E_std, "iterations": n_it,
                   "standard_ms_per_iteration": round(ms_std, 3), "ao_upload_s": round(upload_s, 3),
                   "u_gemm_flops": u_flops, "algorithmic_flops_standard": ccsd_flops(o, v)},
        "roofline": {"bound": "mfma", "achieved": round(u_flops / u_ms / 1e9, 3), "peak": PEAK["f64"],
                     "unit": "TFLOP/s", "frac": round(u_flops / u_ms / 1e9 / PEAK["f64"], 4), "traffic": None,
                     "kernel": f"U GEMM (M = K = nbf^2, N = o^2) avg {u_ms:.3f} ms"},
        "kernels": {k: {"calls": x["calls"], "avg_ms": x["ms"] / max(1, x["calls"])} for k, x in kt.items()
                    if x["ms"] / n_kt > 0.2},
        "cpu_baseline": cpu,
    }
    return line


def main():
    args = _args()
    if args.gpus != 1:
        print(json.dumps({"error": "this library runs on one GPU; sharding across GPUs is "
                                   "designed but not built", "n_gpus": args.gpus}))
        sys.exit(2)
    import torch
    if not torch.cuda.is_available():
        print(json.dumps({"error": "no GPU visible"}))
        sys.exit(1)
    if args.workload == "copy":
        line = bench_copy(args)
    elif args.workload == "pp-ladder":
        line = bench_pp_ladder(args)
    elif args.workload == "batched-hchains":
        line = bench_batched(args)
    elif args.workload == "adjoint-h2o6":
        line = bench_adjoint(args)
    elif args.workload == "df-h2o8":
        line = bench_df(args)
    elif args.workload == "transform-h2o8":
        line = bench_transform(args)
    elif args.workload in ("triples-h2o6", "triples-h2o8"):
        line = bench_triples(args)
    elif args.workload == "eom-h2o6":
        line = bench_eom(args)
    elif args.workload == "direct-h2o8":
        line = bench_direct(args)
    else:
        line = bench_ccsd(args)
    emit(line)


# keys every bench line keeps; anything else moves to stderr when the line would
# pass LINE_LIMIT bytes (the line is parsed from the tail of stdout)
LINE_LIMIT = 4000
CORE_KEYS = ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better",
             "scaling", "vs_baseline", "dtype", "data", "config", "roofline", "cpu_baseline", "forms",
             "small_system")


def emit(line):
    text = json.dumps(line)
    while len(text) > LINE_LIMIT:
        extra = [k for k in line if k not in CORE_KEYS]
        if not extra:
            break
        k = max(extra, key=lambda k: len(json.dumps(line[k])))
        log(f"(moved from the JSON line) {k}: {json.dumps(line.pop(k))}")
        text = json.dumps(line)
    if len(text) > LINE_LIMIT:
        log(f"warning: bench line is {len(text)} bytes")
    print(text, flush=True)


if __name__ == "__main__":
    main()
