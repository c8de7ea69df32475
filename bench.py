"""Throughput benchmark of the adaptive MWDG2 step on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--L 12] [--no-cpu]

Workload: the urban-plain headline case (4096 x 4096 finest cells, max_ref_lvl
12, MWDG2, FP32, epsilon 1e-3, Manning 0.02, 30% seeded building blocks, a 2 m
deep strip on the northern 256 rows, 16 point sources of 5 m^3/s, closed
walls), written as .par/raster/.bci files and loaded through the drop-in
input path. A "step" is one full adaptive time step (grid rebuild, both RK
stages, CFL reduction). Metric: finest-equivalent cell updates per second,
4^L * steps / wall time of the timed steps (inputs resident in HBM).

Besides the metric (the plain step, bit-exact with the reference method),
the line carries the device, the dominant kernel's roofline, the whole
step's roofline (`step_roofline`), the Z-order sort's rate
(`zorder_sort`), the CPU baseline in FP32 and FP64 with the host's lscpu
description, the learned step (`learned`: the network trained on the GPU
from plain-step traces of two other layouts, held-out precision/recall, the
plain step, the step with the network and with the guard alone, each timed
over the same whole 32-step cycles, and again in a window later in the run),
both steps' accuracy against the FP64 product, and the other workloads
(`other_workloads`: the dam break over its whole run, the max_ref_lvl-10
hydrograph in both solvers and precisions, and the 64-scenario ensemble).
`--ensemble N` instead times only N scenarios advanced together (one JSON
line).

Prints one JSON line (see the field list at the end of main()).
"""
from __future__ import annotations

import argparse
import json
import os
import platform
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "gpu-mwdg2_amd"))

METRIC = "finest-equiv cell-updates/s on 1 MI355X; learned vs plain at matched h error"
_T0 = time.time()


def progress(msg: str) -> None:
    """One line on stderr per finished part (the JSON line is stdout's only line)."""
    print(f"bench [{time.time() - _T0:6.1f} s] {msg}", file=sys.stderr, flush=True)
HBM_PEAK_GBS = 8000.0


def cpu_model() -> str:
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return platform.processor() or "unknown"


def cpu_description() -> dict:
    """The host CPU as lscpu reports it (model, sockets, cores, threads) and
    the threads this process may run on."""
    out = {"model": cpu_model(), "usable_threads": len(os.sched_getaffinity(0))}
    try:
        import subprocess
        txt = subprocess.run(["lscpu"], capture_output=True, text=True, timeout=10).stdout
        kv = {}
        for line in txt.splitlines():
            if ":" in line:
                k, v = line.split(":", 1)
                kv[k.strip()] = v.strip()
        out["model"] = kv.get("Model name", out["model"])
        for key, name in (("Socket(s)", "sockets"), ("Core(s) per socket", "cores_per_socket"),
                          ("Thread(s) per core", "threads_per_core"), ("CPU(s)", "logical_cpus")):
            if key in kv:
                out[name] = int(kv[key]) if kv[key].isdigit() else kv[key]
    except (OSError, ValueError):
        pass
    return out


def make_case(L: int) -> str:
    import cases
    d = os.path.join(os.environ.get("TMPDIR", "/tmp"), f"mwdg2_bench_urban_L{L}")
    par = os.path.join(d, "case.par")
    if not os.path.exists(par):
        cases.urban(d, L=L, t_end=1800.0)
    return par


def kernel_bytes(s: int, L: int, leaves: int, wet1: int, wet2: int, p_enc: int = 0, p_dec: int = 0,
                 p_res: int = 0, steps: int = 0) -> dict:
    """Algorithmic HBM bytes of the leaf and MRA band kernels over the timed
    steps.

    Every logical element a kernel must touch is counted once (neighbour
    re-reads are not). A leaf holds 12 coefficients (eta, qx, qy, z x
    {0, 1x, 1y}); 9 of them (not z) are written. Stage 1: the sweep reads all
    leaves and writes the dry ones (and a 4-byte list entry per wet leaf); the
    wet kernel reads and writes the wet leaves. Stage 2 likewise, where a leaf
    also reads its 9 stage-start coefficients from A. The tree passes (flat
    and band kernels together, `steps` passes each): an encoded parent reads its 4
    children's 9 coefficients and writes its own 9; a decoded parent reads
    and writes its children's 36; a re-encoded (stage-1) parent reads 36 and
    writes 9; plus one byte per node from level 6 down for each mask read or written
    (encode: previous tree and preflags in, new tree and extra-significance
    flags out; decode: three in, tree and leaf labels out; re-encode: the
    tree in).
    """
    i = 4
    D = ((1 << (2 * L)) - 1) // 3 + 3
    band = max(0, D - (((1 << 12) - 1) // 3 + 3)) if L > 6 else 0
    return {
        "encode": p_enc * (36 * s + 9 * s) + 4 * band * steps,
        "decode": p_dec * (36 * s + 36 * s) + 5 * band * steps,
        "encode_scale": p_res * (36 * s + 9 * s) + band * steps,
        # leaf emission (labels of the level L-1 nodes read, leaf indices
        # written; the 4 neighbour indices only for the wet leaves, which the
        # wet kernel reads) fused with the stage-1 sweep
        "emit_sweep1": (D >> 2) + leaves * i + leaves * 12 * s + (leaves - wet1) * 9 * s + wet1 * 5 * i,
        "sweep1": leaves * 12 * s + (leaves - wet1) * 9 * s + wet1 * 5 * i,
        "wet1": wet1 * (12 * s + 9 * s),
        "sweep2": leaves * 12 * s + (leaves - wet2) * (9 * s + 9 * s) + wet2 * 5 * i,
        "wet2": wet2 * (12 * s + 9 * s + 9 * s),
        # one-pass kernels (HWFV1 and the limiter path)
        "stage1": leaves * (12 * s + 9 * s),
        "stage2": leaves * (12 * s + 9 * s + 9 * s + s),
    }


def step_bytes_method(s: int, L: int, leaves: float, p_enc: float, p_dec: float, friction: bool) -> dict:
    """Algorithmic HBM bytes of one adaptive MWDG2 step by pass of the method
    (every logical element the step must read or write counted once, b = 1,
    i = 4), whatever the kernels that implement the passes: leaves written
    back into the hierarchy, encode + threshold, regularisation + extra
    significance, decode, leaf list + neighbours, friction, the two RK stages
    with dt, the stage-1 write-back and re-encode for neighbour reads."""
    i, b = 4, 1
    D = ((1 << (2 * L)) - 1) // 3 + 3
    na, pe, pd = leaves, p_enc, p_dec
    passes = {
        "reinsert": na * (12 * s + i) + na * 9 * s,
        "encode": pe * (36 * s + 36 * s + s + 3 * b),
        "regularise_extra": D * 3 * b + pd * s,
        "decode": pd * (36 * s + 36 * s),
        "leaf_list_neighbours": D * b + na * 10 * i,
        "friction": na * (9 * s + 6 * s) if friction else 0,
        "stages": na * (12 * s + 9 * s + s) + na * (12 * s + 9 * s + 9 * s + s),
        "reencode_for_neighbours": na * 9 * s + pe * (36 * s + 9 * s),
    }
    passes["total"] = sum(passes.values())
    return passes


def measured_traffic(kernel: str):
    """HBM bytes per dispatch of `kernel` (read + write) from the committed
    rocprofv3 FETCH_SIZE / WRITE_SIZE summary of this workload, each counter
    scaled by its reading for a 1 GiB copy kernel; None if not recorded."""
    # the tree passes at max_ref_lvl 12: a band kernel and the flat kernel of
    # levels 10 and 11, two launches a step
    names = {"encode": {"k_encode_band<float,true>": 1, "k_encode_level<float,true>": 2},
             "decode": {"k_topdown_band<float,true>": 1, "k_topdown_level<float,true>": 2},
             "encode_scale": {"k_scale_band<float>": 1, "k_scale_level<float>": 2},
             "emit_sweep1": {"k_emit_sweep1<float,1024>": 1}}.get(kernel, {f"k_{kernel}<float>": 1})
    path = os.path.join(ROOT, "profiles", "hbm_traffic_urban_L12.txt")
    total, found = 0, False
    try:
        with open(path) as f:
            for line in f:
                parts = line.split()
                if len(parts) == 4 and parts[0] == "traffic" and parts[1] in names:
                    total += names[parts[1]] * int(float(parts[2]) + float(parts[3]))
                    found = True
    except OSError:
        pass
    return total if found else None


def finest_fields(sim, L: int):
    """Leaf cell means (h, qx, qy) repeated over the finest cells each leaf
    covers, in Morton order, and the water volume sum(h0 * area)."""
    import numpy as np
    leaves = sim.get("leaves").astype(np.int64)
    lev = (np.floor(np.log2(3 * (leaves - 3) + 1) / 2)).astype(np.int64)
    reps = 4 ** (L - lev)
    eta0 = sim.get("A.eta0")[leaves].astype(np.float64)
    z0 = sim.get("z0")[leaves].astype(np.float64)
    h0 = eta0 - z0
    qx = sim.get("A.qx0")[leaves].astype(np.float64)
    qy = sim.get("A.qy0")[leaves].astype(np.float64)
    vol = float(np.sum(h0 * reps))          # dx = 1 m: a level-l cell has area 4^(L-l)
    return np.repeat(h0, reps), np.repeat(qx, reps), np.repeat(qy, reps), vol


def accuracy_vs_fp64(par: str, L: int, runs: dict) -> dict:
    """FP32 runs (plain, learned) against the plain FP64 product (bit-identical
    to the FP64 oracle) after the same number of steps of the same case as
    each run took: max, mean and 99.9th percentile of |dh| over the finest
    cells, max |dq|, and the volume difference. runs: name -> (h, qx, qy,
    volume, time, steps)."""
    import numpy as np
    import mwdg2
    s64 = mwdg2.Simulation(par, "f64")
    fl = ((1 << (2 * L)) - 1) // 3 + 3           # first finest node: the initial state lives there
    v0 = float(np.sum(s64.get("A.eta0")[fl:].astype(np.float64) - s64.get("z0")[fl:]))
    out = {}
    done = 0
    for name, (h, qx, qy, v, t, steps) in sorted(runs.items(), key=lambda kv: kv[1][5]):
        s64.step(steps - done)
        done = steps
        s64.sync()
        h64, qx64, qy64, v64 = finest_fields(s64, L)
        t64 = s64.counters()["time"]
        d = np.abs(h - h64)
        out[name] = {"steps": steps, "time": t, "time_fp64": t64, "max_abs_dh": float(d.max()),
                     "mean_abs_dh": float(d.mean()), "p999_abs_dh": float(np.quantile(d, 0.999)),
                     "max_abs_dqx": float(np.max(np.abs(qx - qx64))), "max_abs_dqy": float(np.max(np.abs(qy - qy64))),
                     "volume_fp64": v64, "volume_change_fp64": v64 - v0, "volume_rel_diff": (v - v64) / v64}
    s64.close()
    return out


def learned_fp64(par: str, L: int, m, warmup: int, n_timed: int) -> dict:
    """The plain and the learned step in FP64 on the benchmark case, timed
    over the same n_timed steps after the same warm-up, and the learned
    step's finest-cell depths against the plain FP64 step's (the FP64 oracle
    bit for bit) at the end of the window."""
    import numpy as np
    import mwdg2
    out = {}
    fields = {}
    for mode, thr in (("plain", None), ("learned", 0.5), ("guard_only", 2.0)):
        with mwdg2.Simulation(par, "f64") as sim:
            if thr is not None:
                sim.set_learned(m, decide_every=8, full_every=32, threshold=thr)
            sim.step(warmup)
            sim.sync()
            t0 = time.perf_counter()
            sim.step(n_timed)
            sim.sync()
            wall = time.perf_counter() - t0
            out[mode] = {"ms_per_step": round(1000.0 * wall / n_timed, 4)}
            h, qx, qy, v = finest_fields(sim, L)
            fields[mode] = (h, v, sim.counters()["time"])
    h0, v0, t0 = fields["plain"]
    for mode in ("learned", "guard_only"):
        h, v, t = fields[mode]
        out[mode]["speedup_vs_plain"] = round(out["plain"]["ms_per_step"] / out[mode]["ms_per_step"], 4)
        out[mode]["max_abs_dh_vs_plain_fp64"] = float(np.max(np.abs(h - h0)))
        out[mode]["volume_rel_diff_vs_plain_fp64"] = (v - v0) / v0
        out[mode]["time_diff_vs_plain_fp64"] = t - t0
    return out


def late_window(par: str, L: int, m, t_late: float, n_timed: int) -> dict:
    """A window later in the run: the plain step advanced to t_late, timed
    over n_timed steps there, then the learned step (network, then every
    unit frozen) switched on in the same run and timed over n_timed steps
    after one 32-step cycle of settling."""
    import mwdg2
    out = {"t_start": t_late, "steps_each": n_timed}
    with mwdg2.Simulation(par, "f32") as sim:
        ta = time.perf_counter()
        c = sim.counters()
        while c["time"] < t_late and not c["done"]:
            sim.step(512)
            c = sim.counters()
        out["advance_steps"] = c["steps"]
        out["advance_s"] = round(time.perf_counter() - ta, 2)
        progress(f"late window: advanced to t = {c['time']:.2f} s in {c['steps']} steps")

        def window(label):
            sim.sync()
            c0 = sim.counters()
            t0 = time.perf_counter()
            sim.step(n_timed)
            sim.sync()
            t1 = time.perf_counter()
            c1 = sim.counters()
            k = c1["steps"] - c0["steps"]
            out[label] = {"ms_per_step": round(1000.0 * (t1 - t0) / max(1, k), 4), "window": [c0["time"], c1["time"]],
                          "mean_leaves": (c1["leaf_updates"] - c0["leaf_updates"]) / max(1, k),
                          "mean_wet_leaves": (c1["wet_updates"][1] - c0["wet_updates"][1]) / max(1, k)}

        window("plain")
        for label, thr in (("learned", 0.5), ("guard_only", 2.0)):
            sim.set_learned(m, decide_every=8, full_every=32, threshold=thr)
            sim.step(32)
            window(label)
            out[label]["speedup_vs_plain"] = round(out["plain"]["ms_per_step"] / out[label]["ms_per_step"], 4)
    return out


def learned_leg(par: str, L: int, warmup: int, steps: int, trace_steps: int, late_t: float) -> tuple:
    """Trains the refinement network on the GPU from plain-step traces of two
    other seeded urban layouts of the same size, checks it on a third, then
    times the plain step, the learned step and the step with every unit
    frozen (the exact guard alone) on the benchmark case over the same whole
    32-step cycles, and again later in the run (late_window)."""
    import mwdg2
    import cases
    base = os.environ.get("TMPDIR", "/tmp")
    t0 = time.time()
    m = mwdg2.Mlp(seed=7)
    for seed in (4, 5):
        d = os.path.join(base, f"mwdg2_bench_urban_L{L}_s{seed}")
        tp = os.path.join(d, "case.par")
        if not os.path.exists(tp):
            cases.urban(d, L=L, seed=seed, src_seed=30 + seed, t_end=1800.0)
        with mwdg2.Simulation(tp, "f32") as s:
            m.record(s, trace_steps)
    n = m.build_labels(8)
    t_rec = time.time() - t0
    progress(f"learned leg: {n} samples recorded")
    t1 = time.time()
    losses = m.fit(10, batch=4096, lr=2e-3, pos_weight=2.0)
    t_fit = time.time() - t1
    held = mwdg2.Mlp(seed=7)
    d = os.path.join(base, f"mwdg2_bench_urban_L{L}_s6")
    hp = os.path.join(d, "case.par")
    if not os.path.exists(hp):
        cases.urban(d, L=L, seed=6, src_seed=36, t_end=1800.0)
    with mwdg2.Simulation(hp, "f32") as s:
        held.record(s, trace_steps // 2)
    held.build_labels(8)
    untrained = held.params
    held.params = m.params
    ct = held.eval(0.5)
    held.params = untrained
    cu = held.eval(0.5)
    held.close()

    def f1(c):
        p = c["tp"] / max(1, c["tp"] + c["fp"])
        r = c["tp"] / max(1, c["tp"] + c["fn"])
        return {"precision": round(p, 4), "recall": round(r, 4), "f1": round(2 * p * r / max(1e-12, p + r), 4)}

    res = {"training": {"samples": n, "trace_steps": 2 * trace_steps, "record_s": round(t_rec, 2),
                        "fit_s": round(t_fit, 3), "epochs": len(losses), "loss_first": float(losses[0]),
                        "loss_last": float(losses[-1]), "held_out_trained": f1(ct), "held_out_untrained": f1(cu)}}
    fields = None
    # every mode is timed over whole 32-step cycles (one plain step in each)
    # after the same warm-up, on a fresh simulation of the benchmark case
    cycles = max(2, -(-steps // 32))
    n_timed = 32 * cycles
    for mode, thr in (("plain_same_window", None), ("learned", 0.5), ("guard_only", 2.0)):
        sim = mwdg2.Simulation(par, "f32")
        if thr is not None:
            sim.set_learned(m, decide_every=8, full_every=32, threshold=thr)
        sim.step(warmup)
        sim.sync()
        c0 = sim.counters()
        ta = time.perf_counter()
        sim.step(n_timed)
        sim.sync()
        tb = time.perf_counter()
        c1 = sim.counters()
        k = c1["steps"] - c0["steps"]
        r = {"ms_per_step": 1000.0 * (tb - ta) / max(1, k), "value": (4 ** L) * k / (tb - ta), "steps": k,
             "window": [c0["time"], c1["time"]]}
        if mode == "learned":
            sim.profile(2)
            sim.step(n_timed)
            sim.sync()
            sim.profile(0)
            lc = sim.learn_counters()
            r["frozen_unit_fraction"] = round(lc["frozen_unit_steps"] / max(1, lc["steps"] * 4096), 4)
            r["quiet_unit_fraction"] = round(lc["quiet_unit_steps"] / max(1, lc["steps"] * 4096), 4)
            r["parents_kept_per_step"] = lc["parents_kept"] / max(1, lc["steps"])
            h, qx, qy, v = finest_fields(sim, L)
            cc = sim.counters()
            fields = (h, qx, qy, v, cc["time"], cc["steps"])
        res[mode] = r
        sim.close()
    base = res["plain_same_window"]["ms_per_step"]
    for mode in ("learned", "guard_only"):
        res[mode]["speedup_vs_plain_same_window"] = round(base / res[mode]["ms_per_step"], 4)
    res["fp64"] = learned_fp64(par, L, m, warmup, n_timed)
    progress("learned leg: same-window timings done")
    res["late_window"] = late_window(par, L, m, late_t, n_timed)
    m.close()
    return res, fields


def run_cpu_baseline(par: str, L: int, budget_s: float, prec: str = "f32") -> dict:
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle
    oracle.build()
    t0 = time.time()
    o = oracle.Oracle(par, prec)
    t_init = time.time() - t0
    n = 0
    t1 = time.time()
    while time.time() - t1 < budget_s and o.step():
        n += 1
    el = time.time() - t1
    threads = int(oracle.lib().mwo_omp_threads())
    o.close()
    return {"value": (4 ** L) * n / el if el > 0 else 0.0, "unit": "finest-equiv cell-updates/s",
            "cores": threads, "kind": "port",
            "precision": prec,
            "sample": f"first {n} steps of the same case from its initial state ({el:.1f} s of stepping, "
                      f"{t_init:.1f} s set-up not timed), C++ oracle ({prec}) with OpenMP on {threads} threads "
                      f"of {cpu_model()}"}


def config_legs(steps: int) -> dict:
    """The other single-scenario workloads, timed on the GPU: the circular
    dam break (max_ref_lvl 8, MWDG2 FP64) over its whole run to t = 3.5 s,
    and the wet/dry hydrograph (max_ref_lvl 10) for HWFV1 and MWDG2 in FP32
    and FP64, advanced to t = 300 s (the hydrograph rise) and timed over
    `steps` steps there. Rates are finest-equivalent cell updates per
    second."""
    import mwdg2
    import cases
    base = os.environ.get("TMPDIR", "/tmp")
    out = {}
    par = cases.circular_dam_break(os.path.join(base, "mwdg2_bench_cdb8"), L=8, eps=1e-3, t_end=3.5, cfl=0.33)
    with mwdg2.Simulation(par, "f64") as s:
        t0 = time.perf_counter()
        c = s.run(max_steps=100000, batch=64)
        wall = time.perf_counter() - t0
        out["dam_break_L8_mwdg2_fp64"] = {"steps": c["steps"], "sim_time": c["time"], "wall_s": round(wall, 4),
                                          "ms_per_step": round(1000.0 * wall / max(1, c["steps"]), 4),
                                          "value": (4 ** 8) * c["steps"] / wall}
    for solver in ("mwdg2", "hwfv1"):
        d = os.path.join(base, f"mwdg2_bench_hydro10_{solver}")
        par = os.path.join(d, "case.par")
        if not os.path.exists(par):
            cases.wetdry_hydrograph(d, L=10, solver=solver, t_end=3600.0)
        for prec in ("f32", "f64"):
            with mwdg2.Simulation(par, prec) as s:
                c = s.counters()
                while c["time"] < 300.0:
                    s.step(1024)
                    c = s.counters()
                s.sync()
                c0 = s.counters()
                t0 = time.perf_counter()
                s.step(steps)
                s.sync()
                wall = time.perf_counter() - t0
                c1 = s.counters()
                k = c1["steps"] - c0["steps"]
                out[f"hydrograph_L10_{solver}_{prec}"] = {
                    "window": [c0["time"], c1["time"]], "steps": k, "ms_per_step": round(1000.0 * wall / max(1, k), 4),
                    "value": (4 ** 10) * k / wall, "mean_leaves": (c1["leaf_updates"] - c0["leaf_updates"]) / max(1, k)}
    return out


def ensemble_bench(n: int, steps: int, warmup: int, autotune: int, ms_single: float | None = None) -> dict:
    """n wet/dry hydrograph scenarios (seeds 4000 + i; max_ref_lvl uniform in
    8..11, bed std 1-10 m, Manning 0.01-0.06, inflow peak 5-100 m^3/s, MWDG2
    FP32) stepped eagerly scenario by scenario (warm-up), then as one
    ensemble in its default launch shape (every pass of all scenarios batched
    into one launch, the step one graph) or the one its autotuner chose,
    timed in two halves of `steps` steps with the other shapes timed in
    between (the same simulated period up to the drift the halves bracket).
    value: sum over scenarios of 4^L * steps / mean wall of the halves;
    vs_single_L12_plain: that rate over the single 4096^2 plain step's."""
    import numpy as np
    import mwdg2
    import cases
    base = os.environ.get("TMPDIR", "/tmp")
    pars, Ls = [], []
    t0 = time.time()
    for i in range(n):
        seed = 4000 + i
        u = cases.uniform(seed, 4)
        L = 8 + min(3, int(u[0] * 4))
        d = os.path.join(base, f"mwdg2_ens_{seed}")
        par = os.path.join(d, "case.par")
        if not os.path.exists(par):
            cases.wetdry_hydrograph(d, L=L, seed=seed, std=1.0 + 9.0 * float(u[1]), manning=0.01 + 0.05 * float(u[2]),
                                    peak=5.0 + 95.0 * float(u[3]), t_end=3600.0)
        pars.append(par)
        Ls.append(L)
    t_cases = time.time() - t0
    progress(f"ensemble: {n} scenario inputs written")
    sims = [mwdg2.Simulation(p, "f32") for p in pars]
    cells = sum(4 ** L for L in Ls)
    for s in sims:
        s.step(warmup)
    for s in sims:
        s.sync()
    ta = time.perf_counter()
    for _ in range(steps):
        for s in sims:
            s.step(1)
    for s in sims:
        s.sync()
    tb = time.perf_counter()
    t1 = time.time()
    ens = mwdg2.Ensemble(sims, autotune_steps=autotune)
    t_create = time.time() - t1
    groups, _ = ens.groups()
    mode, mode_ms = ens.launch_mode()
    ens.step(warmup)
    ens.sync()
    names = ["parent graph", "graph per scenario stream", "direct launches per scenario stream",
             "batched passes, one graph"]

    def timed(m: int) -> float:
        ens.set_launch_mode(m)
        tc = time.perf_counter()
        ens.step(steps)
        ens.sync()
        return time.perf_counter() - tc

    # the chosen shape in two halves around the other shapes: the scenarios'
    # work grows as they wet, and the halves bracket the others' period
    n_modes = 4 if mode_ms[3] > 0 or mode == 3 else 3

    def leaf_total() -> int:
        ens.sync()
        return sum(s.counters()["leaf_updates"] for s in sims)

    la = leaf_total()
    t_a = timed(mode)
    lb = leaf_total()
    others = {names[m]: 1000.0 * timed(m) / steps for m in range(n_modes) if m != mode}
    lc = leaf_total()
    t_b = timed(mode)
    ld = leaf_total()
    leaf_rate = ((lb - la) + (ld - lc)) / (t_a + t_b)
    wall = 0.5 * (t_a + t_b)
    value = cells * steps / wall
    ens.close()
    for s in sims:
        s.close()
    single = 4 ** 12 / (ms_single * 1e-3) if ms_single else None
    return {"metric": "ensemble finest-equiv cell-updates/s on 1 MI355X", "value": value,
            "vs_single_L12_plain": round(value / single, 4) if single else None,
            "leaf_updates_per_s": leaf_rate,
            "unit": "finest-equiv cell-updates/s", "n_gpus": 1, "steps": steps, "warmup": warmup,
            "ms_per_step": 1000.0 * wall / steps, "higher_is_better": True, "scaling": "weak",
            "vs_baseline": None, "dtype": "f32", "data": "synthetic (seeded GRF beds, hydrograph inflow)",
            "config": {"workload": f"ensemble of {n} wet/dry hydrograph scenarios, max_ref_lvl 8-11, MWDG2 FP32",
                       "scenarios": n, "levels": {str(L): Ls.count(L) for L in sorted(set(Ls))},
                       "finest_cells": cells,
                       "eager_before_ensemble_ms_per_step": 1000.0 * (tb - ta) / steps,
                       "autotune_steps": autotune, "sweep_groups": groups,
                       "launch_mode": names[mode], "launch_mode_ms_autotuner": [round(x, 4) for x in mode_ms],
                       "chosen_halves_ms_per_step": [round(1000.0 * t_a / steps, 4), round(1000.0 * t_b / steps, 4)],
                       "other_modes_ms_per_step_between_halves": {k: round(v, 4) for k, v in others.items()},
                       "graph_create_s": round(t_create, 2), "case_files_s": round(t_cases, 1)}}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--L", type=int, default=12)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--cpu-budget", type=float, default=20.0)
    ap.add_argument("--profile-all", action="store_true", help="time every kernel (adds event overhead)")
    ap.add_argument("--no-accuracy", action="store_true",
                    help="skip comparing the FP32 state after the run with an FP64 run of the same steps")
    ap.add_argument("--no-learned", action="store_true", help="skip training and timing the learned step")
    ap.add_argument("--trace-steps", type=int, default=200, help="plain steps recorded per training layout")
    ap.add_argument("--late-time", type=float, default=30.0,
                    help="simulated time at which the late window of the learned leg starts")
    ap.add_argument("--ensemble", type=int, default=0,
                    help="instead of the headline case, time an ensemble of this many scenarios")
    ap.add_argument("--autotune", type=int, default=2, help="autotuner steps per candidate (ensemble)")
    ap.add_argument("--no-configs", action="store_true",
                    help="skip the dam-break, hydrograph and 64-scenario ensemble legs of the default line")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU only (asked for --gpus {args.gpus}); "
              "the multi-GPU decomposition is a design note, not an implementation.", file=sys.stderr)
        sys.exit(2)
    if args.ensemble > 0:
        print(json.dumps(ensemble_bench(args.ensemble, args.steps, args.warmup, args.autotune)))
        return

    import mwdg2
    par = make_case(args.L)
    t0 = time.time()
    sim = mwdg2.Simulation(par, "f32")
    t_setup = time.time() - t0
    sweep_groups = sim.sweep_groups()
    sim.step(args.warmup)
    sim.sync()
    # the timed steps run without events; the kernel durations come from a
    # second pass of as many steps with HIP events on the context stream
    c0 = sim.counters()
    t1 = time.perf_counter()
    sim.step(args.steps)
    sim.sync()
    t2 = time.perf_counter()
    c1 = sim.counters()
    steps = c1["steps"] - c0["steps"]
    wall = t2 - t1
    ms_per_step = 1000.0 * wall / max(1, steps)
    value = (4 ** args.L) * steps / wall
    progress(f"plain step timed: {ms_per_step:.4f} ms")

    sim.profile(1 if args.profile_all else 2)     # events recorded by the update kernels' dispatches
    sim.sync()
    tp1 = time.perf_counter()
    sim.step(args.steps)
    sim.sync()
    tp2 = time.perf_counter()
    prof = sim.profile_read()
    sim.profile(0)
    c2 = sim.counters()
    # the tree passes are a band kernel and flat kernels of the levels below
    # it: timed together, one pass per step
    passes = dict(prof)
    for band, flat in (("encode", "encode_level"), ("decode", "decode_level"),
                       ("encode_scale", "encode_scale_level")):
        if flat in passes:
            n, ms = passes.pop(flat)
            passes[band] = (passes[band][0], passes[band][1] + ms) if band in passes else (n, ms)
    ms_profiled = 1000.0 * (tp2 - tp1) / max(1, c2["steps"] - c1["steps"])

    leaves = c2["leaf_updates"] - c1["leaf_updates"]
    wet = [c2["wet_updates"][q] - c1["wet_updates"][q] for q in range(2)]
    pd = lambda k: c2[k] - c1[k]
    alg = kernel_bytes(4, args.L, leaves, wet[0], wet[1], pd("parents_encoded"), pd("parents_decoded"),
                       pd("parents_rescaled"), c2["steps"] - c1["steps"])
    kern = {}
    for k in alg:
        if k in passes:
            n, ms = passes[k]
            kern[k] = {"launches": n, "avg_ms": ms / n, "alg_bytes_per_launch": alg[k] / n,
                       "gbs": (alg[k] / n) / (ms / n * 1e-3) / 1e9}
    dom = max(kern, key=lambda k: kern[k]["avg_ms"]) if kern else None
    roof = None
    if dom:
        a = kern[dom]["gbs"]
        roof = {"bound": "hbm", "kernel": dom, "achieved": round(a, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": round(a / HBM_PEAK_GBS, 4),
                "traffic": measured_traffic(dom) if args.L == 12 else None,
                "alg_bytes_per_launch": int(kern[dom]["alg_bytes_per_launch"]),
                "avg_launch_ms": round(kern[dom]["avg_ms"], 4)}

    plain_fields = finest_fields(sim, args.L) + (c2["time"], c2["steps"]) if not args.no_accuracy else None

    copy_gbs = mwdg2.stream_copy_gbs(1 << 30, 20)
    if roof:
        roof["measured_copy_gbs"] = round(copy_gbs, 1)
        roof["frac_of_measured_copy"] = round(roof["achieved"] / copy_gbs, 4)
    if args.profile_all:
        out_k = {}
        for name, (n, ms) in sorted(prof.items()):
            out_k[name] = {"launches": n, "avg_us": round(1000.0 * ms / n, 2), "ms_per_step": round(ms / max(1, steps), 4)}
        print(json.dumps({"per_kernel": out_k}), file=sys.stderr)

    # the whole step against the roofline: the method's bytes per step over
    # the step time (the kernels run back to back, so their times sum to it)
    per = lambda k: (c1[k] - c0[k]) / max(1, steps)
    sb = step_bytes_method(4, args.L, leaves / max(1, steps), per("parents_encoded"), per("parents_decoded"), True)
    own = sum(v["alg_bytes_per_launch"] * v["launches"] for k, v in kern.items()
              if k not in ("encode", "decode", "encode_scale")) / max(1, steps)
    step_gbs = sb["total"] / (ms_per_step * 1e-3) / 1e9
    step_roof = {"alg_bytes_per_step": int(sb["total"]), "by_pass": {k: int(v) for k, v in sb.items() if k != "total"},
                 "achieved": round(step_gbs, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                 "frac": round(step_gbs / HBM_PEAK_GBS, 4), "measured_copy_gbs": round(copy_gbs, 1),
                 "frac_of_measured_copy": round(step_gbs / copy_gbs, 4),
                 "update_kernels_alg_bytes_per_step": int(own)}

    # the Z-order build (two pair sorts of the 4^L finest cells, ceil(2L/8)
    # digit passes each, built on first use) timed with HIP events: a pass
    # reads the keys (histogram) and the pairs (scatter) and writes the pairs,
    # 20 bytes per pair
    sim.profile(1)
    sim.get("rev_z_order")
    zs = sim.profile_read().get("zorder_sort")
    sim.profile(0)
    zsort = None
    if zs:
        n_cells = 4 ** args.L
        passes = (2 * args.L + 7) // 8
        zb = 2 * passes * 20 * n_cells
        zsort = {"sorts": zs[0], "pairs": n_cells, "passes_per_sort": passes, "ms_total": round(zs[1], 4),
                 "alg_bytes": zb, "achieved_gbs": round(zb / (zs[1] * 1e-3) / 1e9, 1),
                 "frac_of_peak": round(zb / (zs[1] * 1e-3) / 1e9 / HBM_PEAK_GBS, 4)}

    sim.close()
    progress("kernel events, copy rate and Z-order sort timed")
    learned, lf = (None, None)
    if not args.no_learned and 7 <= args.L <= 12:
        learned, lf = learned_leg(par, args.L, args.warmup, args.steps, args.trace_steps, args.late_time)
        progress("learned leg done")
        learned["speedup_vs_plain"] = learned["learned"]["speedup_vs_plain_same_window"]
        learned["guard_only"]["speedup_vs_plain"] = learned["guard_only"]["speedup_vs_plain_same_window"]
    acc = None
    if not args.no_accuracy:
        runs = {"plain": plain_fields}
        if lf is not None:
            runs["learned"] = lf
        acc = accuracy_vs_fp64(par, args.L, runs)
        progress("accuracy against FP64 done")

    legs = None
    if not args.no_configs:
        legs = config_legs(max(200, args.steps))
        progress("dam break and hydrograph legs done")
        legs["ensemble_64"] = ensemble_bench(64, args.steps, args.warmup, 0, ms_single=ms_per_step)
        progress("ensemble leg done")

    cpu = None
    if not args.no_cpu:
        cpu = run_cpu_baseline(par, args.L, args.cpu_budget, "f32")
        progress("CPU baseline FP32 done")
        cpu["fp64"] = run_cpu_baseline(par, args.L, args.cpu_budget, "f64")
        progress("CPU baseline FP64 done")
        cpu["host"] = cpu_description()

    out = {
        "metric": METRIC, "value": value, "unit": "finest-equiv cell-updates/s", "n_gpus": 1,
        "steps": steps, "warmup": args.warmup, "ms_per_step": ms_per_step, "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f32",
        "data": "synthetic (seeded urban blocks written as .par/ESRI rasters/.bci)",
        "config": {"workload": f"urban plain {1 << args.L}x{1 << args.L} (max_ref_lvl {args.L}), MWDG2 FP32, "
                               "eps 1e-3, n 0.02, 30% blocks, 16 point sources, closed walls",
                   "max_ref_lvl": args.L, "epsilon": 1e-3, "solver": "mwdg2", "precision": "fp32",
                   "mean_leaves": leaves / max(1, steps),
                   "leaf_updates_per_s": (c1["leaf_updates"] - c0["leaf_updates"]) / wall,
                   "mean_parents_encoded": (c1["parents_encoded"] - c0["parents_encoded"]) / max(1, steps),
                   "mean_parents_decoded": (c1["parents_decoded"] - c0["parents_decoded"]) / max(1, steps),
                   "mean_wet_leaves": [w / max(1, steps) for w in wet],
                   "sim_time_reached": c2["time"], "setup_s": round(t_setup, 2), "sweep_groups": sweep_groups,
                   "ms_per_step_with_kernel_events": round(ms_profiled, 4),
                   "kernels": {k: {kk: (round(vv, 4) if isinstance(vv, float) else vv) for kk, vv in v.items()}
                               for k, v in kern.items()}},
        "device": mwdg2.device_name(),
        "roofline": roof,
        "step_roofline": step_roof,
        "zorder_sort": zsort,
        "cpu_baseline": cpu,
    }
    if legs is not None:
        out["other_workloads"] = legs
    if learned is not None:
        out["learned"] = learned
    if acc is not None:
        out["accuracy_fp32_vs_fp64"] = acc
    print(json.dumps(out))


if __name__ == "__main__":
    main()
