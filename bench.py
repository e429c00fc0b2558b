#!/usr/bin/env python3
"""Benchmark: batched stiff-ODE integration on one MI355X.

Workload (one "step"): 2^20 independent hhe6 systems (H/He ionisation +
internal energy, 6 ODEs, rates A T^b exp(-C/T)), semi-implicit Euler with
step doubling, integrated over 1 Myr from seeded synthetic initial
conditions already resident in HBM.  Each step restores the initial state
(a device-to-device copy) and integrates every system to t_end.

The headline runs the persistent lane-per-system kernel in fast arithmetic
with the adaptive (error-norm) step controller at abs = rel = 2e-6, the
loosest setting of a sweep at which every sampled final state meets rel err
<= 1e-3 vs FP64; looser tolerances (faster, with part of the sample outside
the bound) are reported beside it, and so is the same integration with the
previous step's per-system sub-step counts as cost hints (longest systems
first; bit-identical results), the case of a caller that integrates the
same cells again.
Also reported (one JSON line with the main figures, all of them in the --detail
file): the final-state relative error of a
512-system sample against FP64 Radau solutions (tests/golden/truth_hhe6.npz),
per-step latency p50/p99, the integration kernel's roofline position, the
reference algorithm as the reference runs it (exact arithmetic, reference
controller, tol 1e-3) with its own accuracy, the one-workgroup-per-system
kernel with the headline's algorithm on a subset (the 5x target's
denominator), and the oracle (CPU restatement of the reference c_baseline)
timed on this host's cores.  Beside the headline: the mixed-N mass-action
workload (2^18 systems, N in {5, 10, 32, 64, 157}) in one autotuned,
graph-captured batch with its accuracy against FP64 and the plain
one-workgroup-per-system kernel's rate; WIND's own published benchmark (Katz96
tiled to N = 5 .. 250, 80 systems, through the drop-in) beside its published
time-to-solution fits; the N = 157 dense kernel against the
FP32 MFMA peak on a sample and on all 65,536 systems of that workload; and the
request server under Poisson arrivals (p50/p99).

    python bench.py [--steps K] [--warmup W] [--mode fast|exact] [--gpus 1]
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

N_SPECIES = 6
NSYS = 1 << 20
SEED = 1
# Headline tolerance (adaptive controller): the loosest of a sweep at which
# every system of the FP64 sample ends within 1e-3 (at 1e-5, 97% do).
TOL = 2e-6
SWEEP_TOLS = (1e-5, 5e-6)  # looser tolerances reported beside the headline
REF_TOL = 1e-3      # the reference controller's run
# Algorithmic work of hhe6 (counted once, LAPACK-style): network RHS +
# Jacobian 674 flops (+ 8 exp, 1 log, 3 div, counted apart); per solve: form
# I - hJ 2N^2, LU 2/3 N^3, two triangular solves 2N^2, update 2N.  An attempt
# evaluates the network twice (at y for the full step and the first half
# step, and at the half-step state) and solves three systems; per sub-step
# (3 per attempt) that is F_SUBSTEP.  The executed count of the fast kernel
# and its VALU issue share come from the counters in profiles/valu_counts.json.
F_NET = 674
F_SOLVE = 2 * N_SPECIES**2 + (2 * N_SPECIES**3) // 3 + 2 * N_SPECIES**2 + 2 * N_SPECIES
F_SUBSTEP = (2 * F_NET + 3 * F_SOLVE) / 3.0
# Algorithmic HBM bytes per system: state in + out (2N floats) + 1 constant.
BYTES_PER_SYSTEM = 4 * (2 * N_SPECIES + 1)
PEAK_HBM_GBS = 8000.0
PEAK_FP32_TFLOPS = 157.3          # published FP32 vector peak (counts packed dual-issue FP32)
PEAK_FP32_UNPACKED_TFLOPS = 78.6  # one FMA per lane per cycle: the ceiling without packed FP32


def progress(msg):
    """One line per finished leg on stderr (the JSON line stays alone on
    stdout)."""
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def host_cores():
    """Threads for the CPU baseline: the CPUs this process may run on
    (sched_getaffinity), capped by the cgroup CPU quota when one is set.
    Returns (threads, visible CPUs, quota or None)."""
    vis = len(os.sched_getaffinity(0))
    quota = None
    try:
        with open("/sys/fs/cgroup/cpu.max") as f:
            q, per = f.read().split()[:2]
        if q != "max":
            quota = float(q) / float(per)
    except (OSError, ValueError):
        pass
    n = vis if quota is None else max(1, min(vis, int(quota + 0.5)))
    return n, vis, quota


def rel_err(y, truth, floor=1e-3):
    return np.max(np.abs(y - truth) / np.maximum(np.abs(truth), floor), axis=1)


def _acc_stats(e):
    if len(e) == 0:
        return None
    # with infinite errors in the sample, quantiles without interpolation
    # (interpolating between inf values gives nan)
    qm = "linear" if np.isfinite(e).all() else "higher"
    return {"sample": int(len(e)), "frac_rel_err_le_1e-3": float(np.mean(e <= 1e-3)),
            "median_rel_err": float(np.quantile(e, 0.5, method=qm)),
            "p90_rel_err": float(np.quantile(e, 0.9, method=qm)),
            "p99_rel_err": float(np.quantile(e, 0.99, method=qm)), "max_rel_err": float(np.max(e)),
            "nonfinite": int(np.sum(~np.isfinite(e)))}


def accuracy(yf, nsys):
    """Final-state error against FP64 Radau solutions: the 512-system
    uniform sample (every 2048th system, truth_hhe6.npz) and the 8192-system
    tail sample (6144 stratified over log T x log n_H plus the 2048 with the
    most sub-steps, truth_hhe6_tail.npz); the headline figures are over both."""
    parts, out = [], {}
    for name, fn in (("uniform", "truth_hhe6.npz"), ("tail", "truth_hhe6_tail.npz")):
        tp = os.path.join(ROOT, "tests", "golden", fn)
        if not os.path.exists(tp):
            continue
        T = np.load(tp)
        idx = T["idx"]
        keep = idx < nsys
        if not keep.any():
            continue
        e = rel_err(yf[idx[keep]].astype(np.float64), T["y"][keep])
        e = np.where(np.isnan(e), np.inf, e)
        parts.append(e)
        out[name] = _acc_stats(e)
        if name == "tail":
            strat = (np.arange(len(idx)) < int(T["n_stratified"]))[keep]
            out[name]["stratified"] = _acc_stats(e[strat])
            out[name]["most_substeps"] = _acc_stats(e[~strat])
    if not parts:
        return None
    res = _acc_stats(np.concatenate(parts))
    res.update(out)
    return res


def cpu_baseline(params, y0, nH, seconds, tol, controller):
    """The oracle (CPU restatement of c_baseline) on this host's cores over
    bounded samples of the same workload: all cores (one contiguous slice of
    systems per thread, median of 3 runs) and one core."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import oracle_lib as O

    net = O.hhe6(params)
    threads, visible, quota = host_cores()

    def run(n, nthreads):
        y = y0[: n * N_SPECIES].copy()
        t = time.perf_counter()
        O.gold_integrate(O.SIE, net, 0.0, 1.0e6, 1, nH[:n].copy(), y, n, tol, tol, const_stride=1, threads=nthreads,
                         controller=controller)
        return time.perf_counter() - t

    # calibrate on 32 systems, then size each run for a quarter of `seconds`
    per_sys = run(32, 1) / 32
    budget = seconds / 4.0
    n = int(max(threads * 8, min(NSYS, budget * threads / max(per_sys, 1e-9))))
    n = (n // threads) * threads
    dt = float(np.median([run(n, threads) for _ in range(3)]))
    n1 = int(max(8, min(NSYS, budget / max(per_sys, 1e-9))))
    dt1 = run(n1, 1)
    return {"value": n / dt, "unit": "systems/s", "cores": threads, "kind": "port",
            "host_cpus_visible": visible, "cgroup_cpu_quota": quota,
            "sample": f"first {n} of the {NSYS} systems, one contiguous slice per thread; median of 3 runs, "
                      f"{dt:.1f} s each",
            "single_core": {"value": n1 / dt1, "unit": "systems/s", "cores": 1,
                            "sample": f"first {n1} of the {NSYS} systems, {dt1:.1f} s"},
            "algorithm": ("reference controller" if controller == 0 else "adaptive controller") + f", tol {tol:g}"}


# ------------------------------------------------------ NR_test (config 1)
def nr_test_c1(W, reps=5):
    """The reference's stiff linear test system: 1024 systems, N = 2, t in
    [0, 1], dt0 = 1e-3, abs = rel = 1e-3, SIE.  GPU: the drop-in
    cudaIntegrateSystem of wind_amd/lib/nr_test/sie.so (exact mode, host
    arrays, as WIND's harness calls it); CPU: the oracle (c_baseline's
    algorithm) on one core, as the reference's goldIntegrateSystem runs.
    Accuracy against the closed form y1 = 2 e^-at - e^-1000at,
    y2 = -e^-at + e^-1000at."""
    import ctypes as C

    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import oracle_lib as O

    n = 1024
    y0, c, a = W.nr_test_systems(n, seed=0)
    so = C.CDLL(os.path.join(ROOT, "wind_amd", "lib", "nr_test", "sie.so"))
    fn = getattr(so, "_Z19cudaIntegrateSystemffiPfS_iiff")
    fn.argtypes = [C.c_float, C.c_float, C.c_int, C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_float, C.c_float]
    ts, y = [], None
    for _ in range(reps + 1):
        y = y0.copy()
        t = time.perf_counter()
        fn(0.0, 1.0, 1000, c.ctypes.data, y.ctypes.data, n, 2, 1e-3, 1e-3)
        ts.append(time.perf_counter() - t)
    gpu_s = float(np.median(ts[1:]))
    yr = y0.copy()
    t = time.perf_counter()
    O.gold_integrate(O.SIE, O.nr_test(), 0.0, 1.0, 1000, c, yr, n, 1e-3, 1e-3, const_stride=4)
    cpu_s = time.perf_counter() - t
    exact = W.nr_test_exact(a, 1.0).reshape(-1, 2)
    e = np.max(np.abs(y.reshape(-1, 2) - exact) / np.maximum(np.abs(exact), 1e-3), axis=1)
    return {"workload": "NR_test stiff linear system, 1024 systems, N = 2, t in [0, 1], dt0 = 1e-3, "
                        "abs = rel = 1e-3, SIE, reference controller",
            "gpu": {"value": n / gpu_s, "unit": "systems/s", "ms_per_call": gpu_s * 1e3,
                    "path": "drop-in cudaIntegrateSystem (nr_test/sie.so), exact mode, host arrays in and out"},
            "cpu": {"value": n / cpu_s, "unit": "systems/s", "cores": 1, "kind": "port",
                    "sample": "all 1024 systems, one thread (the reference's goldIntegrateSystem is serial)"},
            "bit_identical_to_oracle": bool(np.array_equal(y.view(np.uint32), yr.view(np.uint32))),
            "accuracy_vs_closed_form": {"max_rel_err": float(e.max()), "median_rel_err": float(np.median(e)),
                                        "frac_rel_err_le_1e-3": float(np.mean(e <= 1e-3))}}


# ----------------------------------------- the reference's published benchmark
# Least-squares fits of WIND's Ntile-scaling time to solution (tts = b + a N for
# RK2, b + a N^3 for SIE), python/ntbks/NtileScaling.ipynb:173,185,245-254:
# hardware -> method -> (b seconds, a seconds per N or per N^3).
WIND_PUBLISHED_TTS = {
    "Tesla K20x": {"rk2": (0.208, 117.2e-6), "sie": (0.269, 32.6e-6)},
    "Tesla K40m": {"rk2": (0.153, 393.9e-6), "sie": (0.214, 5.5e-6)},
    "GTX 1050 Ti": {"rk2": (0.061, 114.5e-6), "sie": (0.088, 3.3e-6)},
    "K40m node host CPU": {"rk2": (0.004, 118.2e-6), "sie": (0.004, 3.9e-6)},
    "laptop host CPU": {"rk2": (0.001, 39.1e-6), "sie": (0.003, 2.7e-6)},
}


def wind_published_katz96(W, reps=3, cpu_max_n=100):
    """WIND's own published benchmark, run the way its harness runs it: Katz96
    tiled Ntile times (N = 5 Ntile), the 4 systems of its smoke-test input
    repeated 20 times (80 systems), t in [0, 200] yr, one output step,
    n_integration_steps = 1, abs = rel = 5e-3 (Katz96_neqntile.<T>_
    nsystemtile.20_fixed.1_abs.5e3_rel.5e3).  Time to solution of one call of
    the drop-in cudaIntegrateSystem (sie.so / rk2.so of the generated network:
    exact mode, host arrays in and out), median of `reps` after a warm-up call,
    beside the published fits evaluated at the same N; the oracle on one core
    for N <= cpu_max_n, and the GPU result checked against it bit for bit."""
    import ctypes as C

    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import oracle_lib as O

    rows = []
    for T in W.KATZ96_SCALING_NTILES:
        name = "katz96_gen" if T == 1 else f"katz96_t{T}"
        d = os.path.join(ROOT, "wind_amd", "lib", "gen", name)
        if not os.path.exists(os.path.join(d, "sie.so")):
            continue
        N = 5 * T
        y0, c = W.katz96_scaling_systems(T)
        ns = len(y0) // N
        row = {"ntile": T, "N": N, "systems": ns}
        for meth, lib in (("sie", "sie.so"), ("rk2", "rk2.so")):
            fn = getattr(C.CDLL(os.path.join(d, lib)), "_Z19cudaIntegrateSystemffiPfS_iiff")
            fn.argtypes = [C.c_float, C.c_float, C.c_int, C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_float,
                           C.c_float]
            ts, y = [], None
            for _ in range(reps + 1):
                y = y0.copy()
                t = time.perf_counter()
                fn(0.0, 200.0, 1, c.ctypes.data, y.ctypes.data, ns, N, 5e-3, 5e-3)
                ts.append(time.perf_counter() - t)
            r = {"tts_ms": float(np.median(ts[1:])) * 1e3}
            expo = 3 if meth == "sie" else 1
            pub = {hw: (f[meth][0] + f[meth][1] * N ** expo) * 1e3 for hw, f in WIND_PUBLISHED_TTS.items()}
            r["published_fit_tts_ms"] = pub
            best_gpu = min(v for hw, v in pub.items() if "CPU" not in hw)
            r["speedup_vs_best_published_gpu"] = best_gpu / r["tts_ms"]
            if N <= cpu_max_n:
                yr = y0.copy()
                t = time.perf_counter()
                O.gold_integrate(O.SIE if meth == "sie" else O.RK2, O.generated(name), 0.0, 200.0, 1, c, yr, ns,
                                 5e-3, 5e-3, const_stride=10)
                r["oracle_one_core_ms"] = (time.perf_counter() - t) * 1e3
                r["bit_identical_to_oracle"] = bool(np.array_equal(y.view(np.uint32), yr.view(np.uint32)))
            row[meth] = r
        rows.append(row)
        progress(f"WIND published benchmark: N = {N} done (SIE {row['sie']['tts_ms']:.2f} ms, "
                 f"RK2 {row['rk2']['tts_ms']:.2f} ms)")
    return {"workload": "Katz96 tiled Ntile times (N = 5 Ntile), 80 systems (the 4 smoke-test systems x 20), "
                        "t in [0, 200] yr, n_integration_steps = 1, abs = rel = 5e-3, one cudaIntegrateSystem "
                        "call through the drop-in (exact mode, host arrays)",
            "source": "python/ntbks/NtileScaling.ipynb (published fits tts = b + a N for RK2, b + a N^3 for SIE)",
            "rows": rows}


# ------------------------------------------------------- hhe6 RK2 (config 2)
def rk2_hhe6(torch, api, W, net, y0, cst, nsys, tol, reps=2):
    """The RK2 leg of the hhe6 workload: the same systems, fast lane kernel,
    adaptive controller at the headline tolerance."""
    y = torch.empty_like(y0)
    steps = torch.zeros(nsys, dtype=torch.int32, device=y0.device)
    status = torch.zeros(nsys, dtype=torch.int32, device=y0.device)
    ts, kern = [], []
    tot = 0
    for _ in range(reps):
        y.copy_(y0)
        torch.cuda.synchronize()
        t = time.perf_counter()
        tot, kms = api.integrate(net, 0.0, W.HHE6_TEND_YR, 1, cst, y, nsys, tol, tol, method=api.RK2,
                                 mode=api.MODE_FAST, kernel=api.KERNEL_LANE, device_pointers=True, steps_out=steps,
                                 status_out=status, want_kernel_ms=True, controller=api.CTRL_ADAPTIVE)
        torch.cuda.synchronize()
        ts.append(time.perf_counter() - t)
        kern.append(kms)
    st = status.cpu().numpy()
    sub = steps.cpu().numpy().astype(np.int64)
    acc = accuracy(y.cpu().numpy().reshape(-1, N_SPECIES), nsys)
    return {"workload": f"hhe6, {nsys} systems, 1 Myr, RK2 (explicit), fast lane kernel, adaptive controller, "
                        f"abs = rel = {tol:g}",
            "value": nsys / min(ts), "unit": "systems/s", "kernel_ms": float(min(kern)), "substeps": int(tot),
            "substeps_per_system": {"mean": float(sub.mean()), "max": int(sub.max())},
            "status": {"ok": int(np.sum(st == 0)), "stalled": int(np.sum(st == 1)),
                       "exhausted": int(np.sum(st == 2))},
            "accuracy": acc}


# ----------------------------------------------------------- mixed-N batch
MIXED_NSYS = 1 << 18
# Mass-action controller tolerances: every system of the FP64 sample ends
# within 1e-3 (at rel 1e-4 the worst N = 5 system ends at 1.2e-3).
MA_ABS, MA_REL = 1e-10, 8e-5
# Plain-kernel samples per bucket: at least 8 workgroups per CU (2048
# systems on 256 CUs) so that the rate is the device's, not one system's.
PLAIN_SAMPLE = {5: 8192, 10: 8192, 32: 4096, 64: 2048, 157: 2048}


def dense_flops(N):
    """Algorithmic flops per sub-step of a mass-action system (counted once):
    RHS + Jacobian 64N, form I - hJ 2N^2, LU 2/3 N^3, two triangular solves
    2N^2, update 2N."""
    return 64 * N + 2 * N * N + (2 * N**3) // 3 + 2 * N * N + 2 * N


def ma_rel_err(y, yt, floor=1e-6):
    tot = np.abs(yt).sum(axis=1, keepdims=True)
    e = np.abs(y - yt) / np.maximum(np.abs(yt), floor * tot)
    return np.where(np.isnan(e), np.inf, e).max(axis=1)


def mixed_batch(torch, api, W, nsys, steps, plain, use_generated=True):
    """Mixed-N mass-action workload in one batched, autotuned, graph-captured
    call; its accuracy on the FP64-truth sample; the plain one-workgroup-per-
    system kernel (exact arithmetic, same controller and tolerances) timed
    per bucket on samples."""
    dev = torch.device("cuda:0")
    wl = W.mixed_workload(nsys, seed=4)
    bk = []
    for b in wl:
        n = len(b["scale"])
        y0 = torch.from_numpy(b["y0"]).to(dev)
        table = api.Network.mass_action(b["N"], b["rx"], b["k"])
        net, kind = table, ("table (register-resident dense solver)" if b["N"] in (32, 64, 157)
                            else "table (dense LDS solver)")
        plugin = os.path.join(ROOT, "wind_amd", "lib", "gen", f"mixed{b['N']}", "libwind_net.so")
        if use_generated and b["N"] in W.GENERATED_MIXED and os.path.exists(plugin):
            net, kind = api.Network.plugin(plugin), "generated (lane per system)"
        bk.append(dict(net=net, table=table, kind=kind, N=b["N"], nsys=n, y0=y0,
                       equations=y0.clone(), constants=torch.from_numpy(b["scale"]).to(dev),
                       steps_out=torch.zeros(n, dtype=torch.int32, device=dev),
                       status_out=torch.zeros(n, dtype=torch.int32, device=dev)))
    tend = W.MASS_ACTION_TEND
    t = time.perf_counter()
    api.integrate_batch(bk, 0.0, tend, 1, MA_ABS, MA_REL, graph=True, max_attempts=100000)  # tune + capture
    torch.cuda.synchronize()
    warm_s = time.perf_counter() - t
    progress(f"mixed batch: first call (autotune + capture) {warm_s:.1f} s")
    times = []
    for _ in range(steps):
        for b in bk:
            b["equations"].copy_(b["y0"])
        torch.cuda.synchronize()
        t = time.perf_counter()
        total, _ = api.integrate_batch(bk, 0.0, tend, 1, MA_ABS, MA_REL, graph=True, max_attempts=100000)
        torch.cuda.synchronize()
        times.append(time.perf_counter() - t)
        progress(f"mixed batch: step {len(times)} {times[-1]:.2f} s")
    sec = float(np.median(times))
    # The same integration with each bucket started from cost hints (its
    # sub-step counts from the step before); results are bit-identical.
    ref_y = [b["equations"].clone() for b in bk]
    for b in bk:
        b["cost_hint"] = b["steps_out"].clone()
        b["equations"].copy_(b["y0"])
    torch.cuda.synchronize()
    t = time.perf_counter()
    api.integrate_batch(bk, 0.0, tend, 1, MA_ABS, MA_REL, graph=True, max_attempts=100000)
    torch.cuda.synchronize()
    hinted_s = time.perf_counter() - t
    same = all(bool(torch.equal(b["equations"], r)) for b, r in zip(bk, ref_y))
    for b in bk:
        del b["cost_hint"]
    progress(f"mixed batch: step with cost hints {hinted_s:.2f} s (results identical: {same})")
    out = {"workload": f"mixed-N mass-action, {nsys} systems, N in {list(W.MIXED_SIZES)} with weights "
                       f"{list(W.MIXED_WEIGHTS)}, rate scales logU[0.1, 10], t in [0, {tend:g}], SIE, adaptive "
                       f"controller abs {MA_ABS:g} rel {MA_REL:g}",
           "value": nsys / sec, "unit": "systems/s", "ms_per_step": sec * 1e3, "steps": steps,
           "first_call_s_incl_autotune_and_capture": warm_s, "substeps": int(total), "buckets": {},
           "with_cost_hint": {"value": nsys / hinted_s, "ms_per_step": hinted_s * 1e3,
                              "results_identical": same,
                              "hints": "each bucket's steps_out from the step before (one step, graph "
                                       "captured with the hints in the same call)"}}
    tp = os.path.join(ROOT, "tests", "golden", "truth_mass_action.npz")
    T = np.load(tp) if os.path.exists(tp) else None
    fracs = []
    for b in bk:
        st = b["status_out"].cpu().numpy()
        sp = b["steps_out"].cpu().numpy().astype(np.int64)
        info = {"nsys": b["nsys"], "network": b["kind"], "substeps_mean": float(sp.mean()),
                "substeps_p90": float(np.quantile(sp, 0.9)),
                "status_ok": int(np.sum(st == 0))}
        if T is not None and nsys == int(T["mixed_nsys"]):
            sel = T[f"mixed_{b['N']}_idx"]
            y = b["equations"].cpu().numpy().reshape(-1, b["N"])[sel].astype(np.float64)
            e = ma_rel_err(y, T[f"mixed_{b['N']}_y"])
            info["frac_rel_err_le_1e-3"] = float(np.mean(e <= 1e-3))
            info["median_rel_err"] = float(np.median(e))
            fracs.append(e)
        out["buckets"][str(b["N"])] = info
    if fracs:
        e = np.concatenate(fracs)
        out["accuracy"] = {"sample": int(len(e)), "frac_rel_err_le_1e-3": float(np.mean(e <= 1e-3)),
                           "median_rel_err": float(np.median(e)),
                           "error_definition": "max over species |y - y_fp64| / max(|y_fp64|, 1e-6 sum|y_fp64|)"}
    if plain:
        est = 0.0
        rates = {}
        for b in bk:
            n = min(b["nsys"], PLAIN_SAMPLE.get(b["N"], 1024))
            y = b["y0"][: n * b["N"]].clone()
            torch.cuda.synchronize()
            t = time.perf_counter()
            api.integrate(b["table"], 0.0, tend, 1, b["constants"][:n], y, n, MA_ABS, MA_REL, mode=api.MODE_EXACT,
                          kernel=api.KERNEL_BLOCK, device_pointers=True, controller=api.CTRL_ADAPTIVE,
                          max_attempts=100000)
            torch.cuda.synchronize()
            rates[str(b["N"])] = n / (time.perf_counter() - t)
            est += b["nsys"] / rates[str(b["N"])]
            progress(f"mixed batch: plain kernel, N = {b['N']}: {rates[str(b['N'])]:.1f} systems/s")
        out["plain_gpu"] = {"value": nsys / est, "unit": "systems/s",
                            "kernel": "ma_block_integrate: one workgroup per system, equation per thread, "
                                      "Gauss-Jordan inverse (the reference's algorithm), exact arithmetic, same "
                                      "controller and tolerances",
                            "method": "per-bucket rates on the first systems of each bucket "
                                      f"({PLAIN_SAMPLE}), summed over the bucket sizes",
                            "bucket_rates": rates, "speedup": (nsys / sec) / (nsys / est)}
    return out


def dense_full(torch, api, W):
    """The whole N = 157 dense workload (all its systems) in one call with the
    default solver: systems/s, and the final-state error of the 32 systems
    with FP64 truth (tests/golden/truth_mass_action.npz) taken from this run."""
    dev = torch.device("cuda:0")
    nsys = W.DENSE_NSYS
    rx, k, y0, sc = W.dense_workload(nsys)
    net = api.Network.mass_action(W.DENSE_N, rx, k)
    y = torch.from_numpy(y0).to(dev)
    c = torch.from_numpy(sc).to(dev)
    st = torch.zeros(nsys, dtype=torch.int32, device=dev)
    tot, kms = api.integrate(net, 0.0, W.MASS_ACTION_TEND, 1, c, y, nsys, MA_ABS, MA_REL, mode=api.MODE_FAST,
                             device_pointers=True, controller=api.CTRL_ADAPTIVE, want_kernel_ms=True,
                             max_attempts=100000, status_out=st)
    out = {"workload": f"N = 157 mass-action, all {nsys} systems, t in [0, {W.MASS_ACTION_TEND:g}], SIE, adaptive "
                       f"controller abs {MA_ABS:g} rel {MA_REL:g}",
           "kernel": "ma_dense_reg_integrate<10>", "systems_per_s": nsys / (kms / 1e3), "kernel_ms": kms,
           "substeps": int(tot), "status_ok": int((st == 0).sum())}
    F = dense_flops(W.DENSE_N)
    ach = F * float(tot) / (kms / 1e3) / 1e12
    out.update({"achieved": ach, "peak": PEAK_FP32_TFLOPS, "unit": "TFLOP/s", "frac": ach / PEAK_FP32_TFLOPS})
    tp = os.path.join(ROOT, "tests", "golden", "truth_mass_action.npz")
    if os.path.exists(tp):
        T = np.load(tp)
        if float(T["tend"]) == W.MASS_ACTION_TEND:
            sel = T["dense_157_idx"]
            e = ma_rel_err(y.cpu().numpy().reshape(-1, W.DENSE_N)[sel].astype(np.float64), T["dense_157_y"])
            out["accuracy"] = {"sample": int(len(e)), "frac_rel_err_le_1e-3": float(np.mean(e <= 1e-3)),
                               "median_rel_err": float(np.median(e)), "max_rel_err": float(e.max())}
    return out


def dense_roofline(torch, api, W, nsys):
    """The N = 157 dense workload alone on a sample: algorithmic flops per
    second of the dense kernel against the FP32 MFMA peak."""
    dev = torch.device("cuda:0")
    rx, k, y0, sc = W.dense_workload(nsys)
    net = api.Network.mass_action(W.DENSE_N, rx, k)
    y = torch.from_numpy(y0).to(dev)
    c = torch.from_numpy(sc).to(dev)
    steps = torch.zeros(nsys, dtype=torch.int32, device=dev)
    tot, kms = api.integrate(net, 0.0, W.MASS_ACTION_TEND, 1, c, y, nsys, MA_ABS, MA_REL, mode=api.MODE_FAST,
                             device_pointers=True, controller=api.CTRL_ADAPTIVE, want_kernel_ms=True,
                             max_attempts=100000, steps_out=steps)
    F = dense_flops(W.DENSE_N)
    ach = F * float(tot) / (kms / 1e3) / 1e12
    # the same systems again, started longest first from the sub-step counts above
    yh = torch.from_numpy(y0).to(dev)
    _, kh = api.integrate(net, 0.0, W.MASS_ACTION_TEND, 1, c, yh, nsys, MA_ABS, MA_REL, mode=api.MODE_FAST,
                          device_pointers=True, controller=api.CTRL_ADAPTIVE, want_kernel_ms=True,
                          max_attempts=100000, cost_hint=steps)
    # the LDS-resident solver on the same systems (WIND_FLAG_DENSE_LDS)
    yl = torch.from_numpy(y0).to(dev)
    _, kl = api.integrate(net, 0.0, W.MASS_ACTION_TEND, 1, c, yl, nsys, MA_ABS, MA_REL, mode=api.MODE_FAST,
                          device_pointers=True, controller=api.CTRL_ADAPTIVE, want_kernel_ms=True,
                          max_attempts=100000, flags=api.FLAG_DENSE_LDS)
    return {"workload": f"N = 157 mass-action, first {nsys} of {W.DENSE_NSYS} systems, t in [0, 1e9]",
            "sample": f"first {nsys} of the {W.DENSE_NSYS} systems of the N = 157 workload",
            "kernel": "ma_dense_reg_integrate<10> (register-resident matrix, four systems per CU)",
            "systems_per_s": nsys / (kms / 1e3),
            "kernel_ms": kms, "substeps": int(tot), "flops_per_substep": F,
            "us_per_substep_per_cu": kms * 1e3 / (float(tot) / 256.0),
            "bound": "mfma", "achieved": ach, "peak": PEAK_FP32_TFLOPS, "unit": "TFLOP/s",
            "frac": ach / PEAK_FP32_TFLOPS,
            "with_cost_hint": {"systems_per_s": nsys / (kh / 1e3), "kernel_ms": kh,
                               "identical_results": bool(torch.equal(yh.view(torch.int32), y.view(torch.int32)))},
            "lds_resident_solver": {"kernel": "ma_dense_integrate<SIE, MFMA_F32> (WIND_FLAG_DENSE_LDS)",
                                    "systems_per_s": nsys / (kl / 1e3), "kernel_ms": kl}}


def dense_precision(torch, api, W, nsys):
    """The dense solver's precision forms on the N = 157 workload: FP32 MFMA,
    BF16-input MFMA + 2 refinement sweeps (FP64 residual), split-BF16 (x3) + 1
    sweep.  Throughput on the first `nsys` systems; accuracy on the 32 systems
    with FP64 truth (tests/golden/truth_mass_action.npz)."""
    dev = torch.device("cuda:0")
    rx, k, y0, sc = W.dense_workload(W.DENSE_NSYS)
    net = api.Network.mass_action(W.DENSE_N, rx, k)
    tp = os.path.join(ROOT, "tests", "golden", "truth_mass_action.npz")
    T = np.load(tp) if os.path.exists(tp) else None
    out = {}
    for name, solver, ir in (("fp32_mfma", api.SOLVER_MFMA_F32, 0), ("bf16_mfma_ir2", api.SOLVER_MFMA_BF16, 2),
                             ("bf16x3_mfma_ir1", api.SOLVER_MFMA_BF16X3, 1)):
        y = torch.from_numpy(y0[: nsys * W.DENSE_N]).to(dev)
        c = torch.from_numpy(sc[:nsys]).to(dev)
        tot, kms = api.integrate(net, 0.0, W.MASS_ACTION_TEND, 1, c, y, nsys, MA_ABS, MA_REL, mode=api.MODE_FAST,
                                 device_pointers=True, controller=api.CTRL_ADAPTIVE, solver=solver, ir_sweeps=ir,
                                 want_kernel_ms=True, max_attempts=100000)
        r = {"systems_per_s": nsys / (kms / 1e3), "substeps": int(tot), "ir_sweeps": ir}
        if T is not None:
            sel = T["dense_157_idx"]
            ya = y0.reshape(-1, W.DENSE_N)[sel].reshape(-1).copy()
            api.integrate(net, 0.0, float(T["tend"]), 1, sc[sel].copy(), ya, len(sel), MA_ABS, MA_REL,
                          mode=api.MODE_FAST, controller=api.CTRL_ADAPTIVE, solver=solver, ir_sweeps=ir,
                          max_attempts=100000)
            e = ma_rel_err(ya.reshape(-1, W.DENSE_N).astype(np.float64), T["dense_157_y"])
            r["frac_rel_err_le_1e-3"] = float(np.mean(e <= 1e-3))
            r["median_rel_err"] = float(np.median(e))
            r["max_rel_err"] = float(e.max())
        out[name] = r
    return {"workload": f"N = 157 mass-action, first {nsys} systems (accuracy: the 32 FP64-truth systems)",
            "forms": out}


# ------------------------------------------------------------------ serving
def serving(api, W, seconds, load_frac, seed=5):
    """Continuous-batching request server: resident cell blocks of mixed
    networks; Poisson arrivals at 50%, `load_frac` and 90% of the capacity
    measured with a closed-loop burst, `seconds` each; each request advances
    one block by dt and returns its state to the host.  The headline serving
    figures are those at `load_frac`; each load also reports what its
    slowest 1% of requests carry."""
    rng = np.random.default_rng(seed)
    hp = W.hhe6_params()
    nets = {"hhe6": api.Network.builtin(api.NET_HHE6, hp)}
    for b in W.mixed_workload(1 << 12, seed=4):
        plugin = os.path.join(ROOT, "wind_amd", "lib", "gen", f"mixed{b['N']}", "libwind_net.so")
        if b["N"] in W.GENERATED_MIXED and os.path.exists(plugin):
            nets[b["N"]] = (api.Network.plugin(plugin), b)
        else:
            nets[b["N"]] = (api.Network.mass_action(b["N"], b["rx"], b["k"]), b)
    srv = api.Server(8 << 30, nslots=8)
    blocks = []
    for i in range(24):
        if i % 3 != 2:
            n = int(np.exp(rng.uniform(np.log(1e3), np.log(256e3))))
            y0, c = W.hhe6_systems(n, seed=200 + i)
            blocks.append(dict(kind="hhe6", n=n, N=6, h=srv.block(nets["hhe6"], c, y0, n), out=np.empty_like(y0),
                               dt=lambda: float(np.exp(rng.uniform(np.log(1e3), np.log(1e6)))), tol=(TOL, TOL)))
        else:
            N = int(rng.choice(np.array(W.MIXED_SIZES), p=np.array(W.MIXED_WEIGHTS)))
            net = nets[N][0]
            n = int(np.exp(rng.uniform(np.log(1e3), np.log(256e3))) / max(1.0, (N / 10.0) ** 2))
            n = max(n, 64)
            y0, c = W.mass_action_systems(n, N, seed=300 + i, scale_range=W.MIXED_SCALE_RANGE)
            blocks.append(dict(kind=f"mass_action_{N}", n=n, N=N, h=srv.block(net, c, y0, n), out=np.empty_like(y0),
                               dt=lambda: float(np.exp(rng.uniform(np.log(1e6), np.log(1e9)))), tol=(MA_ABS, MA_REL)))
    clock = {id(b): 0.0 for b in blocks}

    def submit(b):
        t0 = clock[id(b)]
        t1 = t0 + b["dt"]()
        clock[id(b)] = t1
        return srv.submit(t0, t1, b["tol"][0], b["tol"][1], block=b["h"], equations=b["out"])

    # capacity: closed-loop burst, one request per block
    t = time.perf_counter()
    ids = [submit(b) for b in blocks]
    for i in ids:
        srv.wait(i)
    burst_s = time.perf_counter() - t
    sys_per_req = float(np.mean([b["n"] for b in blocks]))
    cap_req_s = len(ids) / burst_s
    def open_loop(frac):
        """Poisson arrivals at `frac` of the measured capacity for `seconds`;
        returns per-request (latency ms, systems, substeps)."""
        rate = frac * cap_req_s
        reqs = []
        t_start = time.perf_counter()
        t_next = t_start
        while True:
            now = time.perf_counter()
            if now - t_start >= seconds:
                break
            if now >= t_next:
                b = blocks[int(rng.integers(len(blocks)))]
                reqs.append((submit(b), b))
                t_next += rng.exponential(1.0 / rate)
            else:
                time.sleep(min(0.0005, t_next - now))
        out = []
        for rid, b in reqs:
            l_us, steps = srv.wait(rid)
            out.append((l_us / 1e3, b["n"], steps, b["kind"]))
        return out, time.perf_counter() - t_start

    loads = {}
    for frac in sorted({0.5, load_frac, 0.9}):
        res, wall = open_loop(frac)
        progress(f"serving: offered load {frac:g} done ({len(res)} requests)")
        lat = np.array([r[0] for r in res])
        nsys = np.array([r[1] for r in res], np.float64)
        work = np.array([r[2] for r in res], np.float64)
        p99 = float(np.quantile(lat, 0.99))
        tail = lat >= p99
        loads[f"{frac:g}"] = {
            "requests": int(len(lat)), "systems_per_s": float(nsys.sum() / wall),
            "latency_ms": {"p50": float(np.quantile(lat, 0.5)), "p90": float(np.quantile(lat, 0.9)), "p99": p99,
                           "max": float(lat.max())},
            # the slowest 1%: how much work they carry against the average request
            "p99_tail": {"requests": int(tail.sum()), "mean_systems": float(nsys[tail].mean()),
                         "mean_substeps": float(work[tail].mean()),
                         "substeps_vs_mean_request": float(work[tail].mean() / max(work.mean(), 1.0)),
                         "kinds": sorted({r[3] for r, t in zip(res, tail) if t})},
            "latency_vs_work_spearman": float(_spearman(lat, work)),
        }
    srv.close()
    main_load = loads[f"{load_frac:g}"]
    return {"workload": "24 resident cell blocks (2/3 hhe6 with logU[1k, 256k] systems and dt logU[1e3, 1e6] yr; "
                        "1/3 mixed-N mass-action with logU[1k, 256k]/max(1, (N/10)^2) systems and dt logU[1e6, 1e9]); "
                        "each request advances one block and copies its state to the host",
            "slots": 8, "capacity_requests_per_s": cap_req_s, "mean_systems_per_request": sys_per_req,
            "offered_load": load_frac, "requests": main_load["requests"],
            "systems_per_s": main_load["systems_per_s"], "latency_ms": main_load["latency_ms"],
            "seconds_per_load": seconds, "by_offered_load": loads}


def _spearman(a, b):
    ra = np.argsort(np.argsort(a)).astype(np.float64)
    rb = np.argsort(np.argsort(b)).astype(np.float64)
    ra -= ra.mean()
    rb -= rb.mean()
    return float((ra * rb).sum() / np.sqrt((ra * ra).sum() * (rb * rb).sum()))


LINE_MAX = 4000  # characters of the printed line: a captured output's tail holds all of it


def compact(line, limit=LINE_MAX):
    """The report as one JSON line of at most `limit` characters: numbers to six digits, and beside the headline's
    own fields the legs as deep as there is room for (the --detail file has all of them)."""
    def prune(v, depth):
        if isinstance(v, float):
            return float(f"{v:.6g}") if np.isfinite(v) else None
        if isinstance(v, dict):
            if depth == 0:
                return None
            kept = {k: prune(x, depth - 1) for k, x in v.items() if not (isinstance(x, str) and len(x) > 40)}
            return {k: x for k, x in kept.items() if x is not None} or None
        return None if isinstance(v, (list, tuple)) else v

    own = ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
           "vs_baseline", "dtype", "data", "config", "latency_ms")
    for depth in range(6, -1, -1):
        text = json.dumps({k: v if k in own else prune(v, depth) for k, v in line.items()
                           if k in own or prune(v, depth) is not None})
        if len(text) <= limit:
            break
    return text


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--mode", choices=["fast", "exact"], default="fast")
    ap.add_argument("--controller", choices=["adaptive", "reference"], default="adaptive")
    ap.add_argument("--tol", type=float, default=None)
    ap.add_argument("--nsys", type=int, default=NSYS)
    ap.add_argument("--cpu-seconds", type=float, default=15.0)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-plain", action="store_true")
    ap.add_argument("--mixed-nsys", type=int, default=MIXED_NSYS)
    ap.add_argument("--mixed-steps", type=int, default=2)
    ap.add_argument("--no-mixed", action="store_true")
    ap.add_argument("--no-rk2", action="store_true", help="skip the RK2 leg of the hhe6 workload")
    ap.add_argument("--no-c1", action="store_true", help="skip the NR_test (1024 systems) GPU and CPU row")
    ap.add_argument("--no-wind-published", action="store_true",
                    help="skip WIND's published Katz96 Ntile-scaling benchmark (N = 5 .. 250)")
    ap.add_argument("--no-generated", action="store_true",
                    help="mixed batch: table-driven networks for every N (no generated plugins)")
    ap.add_argument("--serve-seconds", type=float, default=10.0, help="open-loop seconds per offered load")
    ap.add_argument("--serve-load", type=float, default=0.7)
    ap.add_argument("--no-serve", action="store_true")
    ap.add_argument("--dense-nsys", type=int, default=4096)
    ap.add_argument("--no-dense", action="store_true", help="skip the N = 157 dense roofline and precision forms")
    ap.add_argument("--no-dense-full", action="store_true",
                    help="skip the run of all 65,536 systems of the N = 157 workload (about 35 s)")
    ap.add_argument("--hint-steps", type=int, default=3,
                    help="timed steps of the headline with the previous step's sub-step counts as cost hints")
    ap.add_argument("--copy-probe", type=int, default=0,
                    help="only copy this many bytes device to device three times (HBM counter calibration)")
    ap.add_argument("--detail", default=os.path.join(ROOT, "bench_detail.json"),
                    help="file for the whole report; the printed line holds its main figures")
    a = ap.parse_args()
    if a.gpus != 1:
        print(f"bench.py measures one GPU only (--gpus {a.gpus} requested): systems are independent, so "
              "N GPUs would each run this benchmark on their own shard; no multi-GPU run is made here.",
              file=sys.stderr)
        sys.exit(2)

    import torch

    from wind_amd import api
    from wind_amd import networks as W

    dev = torch.device("cuda:0")
    if a.copy_probe:
        src = torch.ones(a.copy_probe // 4, dtype=torch.float32, device=dev)
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        print(json.dumps({"copy_probe_bytes": a.copy_probe}))
        return
    progress("start")
    params = W.hhe6_params()
    y0_h, nH_h = W.hhe6_systems(NSYS, seed=SEED)
    nsys = a.nsys
    net = api.Network.builtin(api.NET_HHE6, params)
    mode = api.MODE_FAST if a.mode == "fast" else api.MODE_EXACT
    ctrl = api.CTRL_ADAPTIVE if a.controller == "adaptive" else api.CTRL_REFERENCE
    tol = a.tol if a.tol is not None else (TOL if ctrl == api.CTRL_ADAPTIVE else REF_TOL)
    y0 = torch.from_numpy(y0_h[: nsys * N_SPECIES]).to(dev)
    cst = torch.from_numpy(nH_h[:nsys]).to(dev)
    y = torch.empty_like(y0)
    steps_d = torch.zeros(nsys, dtype=torch.int32, device=dev)
    status_d = torch.zeros(nsys, dtype=torch.int32, device=dev)
    stream = torch.cuda.current_stream(dev)

    def one_step():
        y.copy_(y0)
        tot, kms = api.integrate(net, 0.0, W.HHE6_TEND_YR, 1, cst, y, nsys, tol, tol, method=api.SIE,
                                 mode=mode, kernel=api.KERNEL_LANE, device_pointers=True,
                                 steps_out=steps_d, status_out=status_d, stream=stream.cuda_stream,
                                 want_kernel_ms=True, controller=ctrl)
        return tot, kms

    for _ in range(a.warmup):
        one_step()
    torch.cuda.synchronize()
    lat, kms_all, tot = [], [], 0
    t0 = time.perf_counter()
    for _ in range(a.steps):
        s = time.perf_counter()
        tot, kms = one_step()
        lat.append(time.perf_counter() - s)
        kms_all.append(kms)
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    value = nsys * a.steps / elapsed
    progress(f"headline: {a.steps} timed steps, {value:.4g} systems/s")
    kernel_s = float(np.mean(kms_all)) / 1e3

    yf = y.cpu().numpy().reshape(-1, N_SPECIES)
    st = status_d.cpu().numpy()
    sub = steps_d.cpu().numpy().astype(np.int64)

    acc = accuracy(yf, nsys)
    if acc:
        acc["error_definition"] = "max over species |y - y_fp64| / max(|y_fp64|, 1e-3)"

    algo_bytes = BYTES_PER_SYSTEM * nsys
    kname = "lane_fast_kernel<NetHHe6, SIE>" if mode == api.MODE_FAST else "lane_integrate<NetHHe6, SIE, MathExact>"
    # FP32 work per sub-step: the algorithmic count (2 network evaluations
    # and 3 dense solves per attempt) sets `achieved`; the executed count and
    # the VALU issue share of the same launch come from the PMC summary in
    # profiles/valu_counts.json (the fast kernel executes fewer FP32
    # operations than the dense algorithm: a rank-structured Jacobian and a
    # shifted solve), when measured for this kernel and tolerance.
    flops = F_SUBSTEP * float(tot)
    executed = None
    vcp = os.path.join(ROOT, "profiles", "valu_counts.json")
    if os.path.exists(vcp):
        with open(vcp) as f:
            vc = json.load(f).get(f"lane_hhe6_{a.mode}")
        if vc and abs(vc.get("tol", tol) - tol) < 1e-12:
            fx = vc["fp32_flops_per_substep_executed"] * float(tot)
            executed = {"fp32_flops_per_substep": vc["fp32_flops_per_substep_executed"],
                        "tflops": fx / kernel_s / 1e12,
                        "frac_of_unpacked_fp32_peak": fx / kernel_s / 1e12 / PEAK_FP32_UNPACKED_TFLOPS,
                        "valu_issue_frac_pmc": vc["valu_issue_frac"], "valu_busy_frac_pmc": vc["valu_busy_frac"],
                        "source": vcp[len(ROOT) + 1:]}
    roofline = {
        # the roofline that binds this kernel: the FP32 vector ALU (it issues
        # no MFMA work and its HBM traffic is the state in and out)
        "bound": "valu", "achieved": flops / kernel_s / 1e12, "peak": PEAK_FP32_TFLOPS, "unit": "TFLOP/s",
        "frac": flops / kernel_s / 1e12 / PEAK_FP32_TFLOPS, "traffic": None,
        "kernel": kname, "kernel_ms": kernel_s * 1e3,
        "kernel_ms_includes": "the start-order pre-pass (lane_probe: 16 attempts per system, lane_activity_hints, "
                              "hint_* kernels)",
        "flops_per_substep": F_SUBSTEP,
        "flops_source": "algorithmic (2 network evaluations and 3 dense solves per attempt)",
        "frac_of_unpacked_fp32_peak": flops / kernel_s / 1e12 / PEAK_FP32_UNPACKED_TFLOPS,
        "executed": executed,
        "hbm": {"achieved": algo_bytes / kernel_s / 1e9, "peak": PEAK_HBM_GBS, "unit": "GB/s",
                "frac": algo_bytes / kernel_s / 1e9 / PEAK_HBM_GBS,
                "algorithmic_bytes_per_system": BYTES_PER_SYSTEM},
    }
    trp = os.path.join(ROOT, "profiles", "traffic.json")
    if os.path.exists(trp):
        with open(trp) as f:
            tr = json.load(f).get(f"lane_hhe6_{a.mode}")
        if tr:
            roofline["traffic"] = tr["bytes_per_launch"] * nsys / tr["nsys"]

    # Start order from cost hints: each system's sub-step count from the step
    # before (what a caller integrating the same cells again would pass) as
    # wind_options.cost_hint.  Same kernel and arithmetic, longest systems
    # first; the results must be bit-identical to the unhinted step's.
    hinted = None
    if mode == api.MODE_FAST and a.hint_steps > 0:
        hint = steps_d.clone()
        yh = torch.empty_like(y0)
        wall, kern = [], []
        for i in range(1 + a.hint_steps):
            torch.cuda.synchronize()
            s = time.perf_counter()
            yh.copy_(y0)
            _, kms = api.integrate(net, 0.0, W.HHE6_TEND_YR, 1, cst, yh, nsys, tol, tol, method=api.SIE,
                                   mode=mode, kernel=api.KERNEL_LANE, device_pointers=True,
                                   stream=stream.cuda_stream, want_kernel_ms=True, controller=ctrl,
                                   cost_hint=hint)
            torch.cuda.synchronize()
            if i:
                wall.append(time.perf_counter() - s)
                kern.append(kms)
        hinted = {"value": nsys / float(np.mean(wall)), "unit": "systems/s",
                  "ms_per_step": float(np.mean(wall)) * 1e3, "kernel_ms": float(np.mean(kern)),
                  "steps": a.hint_steps,
                  "identical_results": bool(torch.equal(yh.view(torch.int32), y.view(torch.int32))),
                  "hint": "each system's sub-step count from the previous step (steps_out), passed as cost_hint"}

    # The same kernel at looser tolerances: faster, with part of the systems
    # outside the 1e-3 bound.
    sweep = {}
    if mode == api.MODE_FAST and ctrl == api.CTRL_ADAPTIVE and a.tol is None:
        for stol in SWEEP_TOLS:
            ys = torch.empty_like(y0)
            tms = []
            for _ in range(2):
                ys.copy_(y0)
                torch.cuda.synchronize()
                t = time.perf_counter()
                api.integrate(net, 0.0, W.HHE6_TEND_YR, 1, cst, ys, nsys, stol, stol, method=api.SIE, mode=mode,
                              kernel=api.KERNEL_LANE, device_pointers=True, stream=stream.cuda_stream,
                              controller=ctrl)
                torch.cuda.synchronize()
                tms.append(time.perf_counter() - t)
            sweep[f"{stol:g}"] = {"value": nsys / min(tms), "unit": "systems/s",
                                  "accuracy": accuracy(ys.cpu().numpy().reshape(-1, N_SPECIES), nsys)}

    # The reference algorithm as the reference runs it: exact arithmetic,
    # reference controller, tol 1e-3 (one timed pass, same systems).
    y.copy_(y0)
    torch.cuda.synchronize()
    t = time.perf_counter()
    api.integrate(net, 0.0, W.HHE6_TEND_YR, 1, cst, y, nsys, REF_TOL, REF_TOL, method=api.SIE,
                  mode=api.MODE_EXACT, kernel=api.KERNEL_LANE, device_pointers=True, stream=stream.cuda_stream,
                  controller=api.CTRL_REFERENCE)
    torch.cuda.synchronize()
    ref_alg = {"value": nsys / (time.perf_counter() - t), "unit": "systems/s",
               "algorithm": f"exact arithmetic, reference controller, tol {REF_TOL:g} (bit-identical to c_baseline)",
               "accuracy": accuracy(y.cpu().numpy().reshape(-1, N_SPECIES), nsys)}

    # The same integration through host buffers (the legacy ABI's contract):
    # copies in and out over PCIe included.  Reported beside, never as value.
    yh = y0_h[: nsys * N_SPECIES].copy()
    ch = nH_h[:nsys].copy()
    t = time.perf_counter()
    api.integrate(net, 0.0, W.HHE6_TEND_YR, 1, ch, yh, nsys, tol, tol, method=api.SIE, mode=mode,
                  kernel=api.KERNEL_LANE, controller=ctrl)
    host_path = {"value": nsys / (time.perf_counter() - t), "unit": "systems/s",
                 "path": "host float32 arrays in and out (H2D + kernel + D2H per call), same settings"}

    plain = None
    if not a.no_plain:
        npl = min(nsys, 65536)
        yp = y0[: npl * N_SPECIES].clone()
        torch.cuda.synchronize()
        t = time.perf_counter()
        api.integrate(net, 0.0, W.HHE6_TEND_YR, 1, cst[:npl], yp, npl, tol, tol, method=api.SIE,
                      mode=api.MODE_EXACT, kernel=api.KERNEL_BLOCK, device_pointers=True,
                      stream=stream.cuda_stream, controller=ctrl)
        torch.cuda.synchronize()
        pv = npl / (time.perf_counter() - t)
        plain = {"value": pv, "unit": "systems/s", "sample": f"first {npl} systems",
                 "kernel": "block_integrate: one workgroup per system, equation per thread (the reference's "
                           "launch shape), same controller and tolerance as the headline",
                 "speedup": value / pv}

    progress(f"headline and its variants done: {value:.4g} systems/s")
    rk2 = None if a.no_rk2 else rk2_hhe6(torch, api, W, net, y0, cst, nsys, tol)
    progress("rk2 leg done")
    c1 = None if a.no_c1 else nr_test_c1(W)
    progress("NR_test row done")
    wind_pub = None if a.no_wind_published else wind_published_katz96(W)
    progress("WIND published benchmark done")
    mixed = None if a.no_mixed else mixed_batch(torch, api, W, a.mixed_nsys, a.mixed_steps, not a.no_plain,
                                                not a.no_generated)
    progress("mixed batch done")
    dense = None if a.no_dense else dense_roofline(torch, api, W, a.dense_nsys)
    progress("dense N = 157 done")
    if dense is not None and not a.no_dense_full:
        dense["full_workload"] = dense_full(torch, api, W)
        progress("dense N = 157, all systems, done")
    precision = None if a.no_dense else dense_precision(torch, api, W, 1024)
    progress("precision forms done")
    serve = None if a.no_serve else serving(api, W, a.serve_seconds, a.serve_load)
    progress("serving done")
    cpu = None if a.no_cpu else cpu_baseline(params, y0_h, nH_h, a.cpu_seconds, REF_TOL, 0)
    progress("CPU baseline (reference algorithm) done")
    cpu_same = None if a.no_cpu else cpu_baseline(params, y0_h, nH_h, a.cpu_seconds, tol, ctrl)
    progress("CPU baseline (headline algorithm) done")

    line = {
        "metric": "ODE systems/sec @ rel err<=1e-3 vs FP64; p50/p99 request latency",
        "value": value, "unit": "systems/s", "n_gpus": 1, "steps": a.steps, "warmup": a.warmup,
        "ms_per_step": elapsed / a.steps * 1e3, "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "f32" if mode == api.MODE_FAST else "f32 (error test f64)",
        "dtype_note": ("fast lane kernel: state, arithmetic and the adaptive error norm in float"
                       if mode == api.MODE_FAST else "exact mode: float state, relative error test in double"),
        "data": "synthetic (seeded)",
        "config": {"workload": "hhe6 H/He ionisation + energy, 6 ODEs, 2^20 systems, 1 Myr, SIE, "
                               f"abs=rel={tol:g}", "nsys": nsys, "method": "SIE", "mode": a.mode,
                   "controller": a.controller, "parallelism": "one GPU"},
        "latency_ms": {"p50": float(np.quantile(lat, 0.5) * 1e3), "p99": float(np.quantile(lat, 0.99) * 1e3),
                       "request": "one step (all systems)"},
        "substeps_per_system": {"mean": float(sub.mean()), "max": int(sub.max())},
        "status": {"ok": int(np.sum(st == 0)), "stalled": int(np.sum(st == 1)), "exhausted": int(np.sum(st == 2))},
        "accuracy": acc, "with_cost_hint": hinted, "looser_tolerances": sweep, "roofline": roofline, "host_buffers_pcie_inclusive": host_path,
        "reference_algorithm": ref_alg, "plain_gpu": plain, "rk2": rk2, "nr_test_1024": c1,
        "cpu_baseline": cpu, "cpu_same_algorithm": cpu_same,
        "wind_published_katz96": wind_pub, "mixed_batch": mixed, "dense_157": dense, "dense_157_precision": precision, "serving": serve,
    }
    with open(a.detail, "w") as f:
        json.dump(line, f, indent=1)
    print(compact(line))


if __name__ == "__main__":
    main()
