"""Benchmark of the MI355X dycore large step (plain FP64).

Workload: stratified flow over a bell-shaped hill, 433 x 433 x 50 mass points,
dx = 3 km, stretched eta, dt = 18 s, 6 acoustic substeps (the configuration
the headline cell-substeps/s metric is quoted on).  Synthetic seeded initial
condition (wrf_gpu_amd.ic.stratified_terrain_3d); inputs are resident in HBM
before the timed region.

A "step" is one RK3 large step (3 stages, 1 + 3 + 6 acoustic substeps).
Throughput counts namelist substeps: cell-substeps/s = N * ns * steps / wall.

Prints ONE JSON line with the metric, the dominant kernel's roofline (its
algorithmic bytes per launch divided by its average launch duration, timed
with HIP events on the launch stream over the timed region), its measured HBM
traffic per launch (from the committed rocprofv3 counter summary, when
present) and a CPU baseline (the oracle on a bounded sample of the same
workload, this host's cores).  The headline value is the plain FP64 form;
"forms" adds the mixed-precision form on the same workload (throughput and
per-field error against FP64 after --form-steps large steps, 200 = one
forecast hour), the launch-bound 64x64x40 warm bubble stepped eagerly and by
graph replay, the 32-member uneven ensemble (members stepped one after
another, and the batched graph in FP64 and in the mixed form), and the same
workload with the 6th-order numerical filter on (diff_6th_opt = 2), with
the 2-D Smagorinsky horizontal diffusion on (diff_opt = 1, km_opt = 4) and
with the monotonic limiter on theta's final-stage advection
(scalar_adv_opt = 2), and carrying the six moisture species, coupled and
transported (moist = 1, moist_adv_opt = 2).

  python bench.py [--gpus 1] [--steps K] [--warmup W]
  python bench.py --pmc-summary FETCH_DIR WRITE_DIR --calibration-copy-mib 1024 > summary.json
      (summarise two rocprofv3 --pmc runs, FETCH_SIZE then WRITE_SIZE, of
       `bench.py --steps 1 --warmup 0 --cpu-baseline-steps 0 --calibration-copy-mib 1024`)
"""

from __future__ import annotations

import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

METRIC = "cell-substeps/s, chosen form vs plain FP64 at stated err; % HBM roofline"
HBM_PEAK_GBS = 8000.0
TRAFFIC_FILE = os.path.join(ROOT, "profiles", "hbm_traffic_terrain_433x433x50.json")

# Algorithmic HBM bytes per mass cell for one launch of each kernel: every 3-D
# array the kernel must read or write, counted once at 8 B per mass cell
# (staggering extras, 2-D fields, neighbour re-reads and kernel-internal
# scratch excluded).
ALG_ARRAYS_PER_CELL = {
    # column march, advance_mu_t kernel: reads u_work, v_work, u, v, theta,
    # th_work, t_tend, t_2ave, rom (9); writes th_work, t_2ave, ww (3)
    "k_column_mu": 12,
    # column march, advance_w + calc_p_rho kernel: reads ph_1 total, ph_tend,
    # w_work, ph_work, rw_tend, a, alpha, gamma, ww, c2a, alt, t_2ave, theta,
    # th_work, pm1, w_save (16); writes ph_work, w_work, p, pm1 (4)
    "k_column_w": 20,
    # advance_uv for u and v: reads u_work, v_work, u_tend, v_tend, p, ph_work,
    # pb, alt, php; writes u_work, v_work
    "k_uv": 11,
    # column block, advance_mu_t + advance_w + calc_p_rho: reads u_work, v_work,
    # u, v, theta, rom, th_work, t_tend, t_2ave, ph_1 total, ph_work, w_work,
    # ph_tend, rw_tend, c2a, alt, gamma, pm1 (18); writes th_work, t_2ave,
    # ph_work, w_work, p, pm1 (6)
    "k_column_block": 24,
    # LDS-tiled column kernel (WRFDYN_COLUMN_TILE=TXxKT): the work of both march
    # kernels in one launch, 23 reads and 7 writes
    "k_column": 30,
}
# Per-large-step compulsory traffic model (cells x 8 B x passes):
# 3 stages x 55 stage passes + S(ns) x 35 substep passes, S(ns) = 1 + ns//2 + ns.


def step_bytes_per_cell(ns: int) -> int:
    s = 1 + max(1, ns // 2) + ns
    return 8 * (3 * 55 + s * 35)


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--nx", type=int, default=433)
    ap.add_argument("--ny", type=int, default=433)
    ap.add_argument("--nz", type=int, default=50)
    ap.add_argument("--cpu-baseline-steps", type=int, default=8,
                    help="large steps of the oracle timed on the host (0 skips)")
    ap.add_argument("--cpu-threads", type=int, default=0, help="0 = all cores in this process's affinity")
    ap.add_argument("--cpu-small-steps", type=int, default=100,
                    help="large steps of the oracle on the 64x64x40 warm bubble, timed beside the main sample "
                         "(0 skips)")
    ap.add_argument("--form-steps", type=int, default=200,
                    help="large steps of the mixed-precision form leg (error measured after them); 0 skips it")
    ap.add_argument("--filter-steps", type=int, default=20,
                    help="large steps of the 6th-order-filter leg on the same workload (0 skips it)")
    ap.add_argument("--smagorinsky-steps", type=int, default=20,
                    help="large steps of the 2-D Smagorinsky diffusion leg on the same workload (0 skips it)")
    ap.add_argument("--limiter-steps", type=int, default=20,
                    help="large steps of the monotonic theta-limiter leg on the same workload (0 skips it)")
    ap.add_argument("--constk-steps", type=int, default=20,
                    help="large steps of the constant-K diffusion leg on the same workload (0 skips it)")
    ap.add_argument("--graph-steps", type=int, default=20,
                    help="large steps of the same workload replayed from a captured graph (0 skips it)")
    ap.add_argument("--moist-steps", type=int, default=20,
                    help="large steps of the moist leg (six species, coupled and transported) on the same workload "
                         "(0 skips it)")
    ap.add_argument("--small-steps", type=int, default=100,
                    help="large steps of the 64x64x40 warm-bubble leg (eager and graph-replayed); 0 skips it")
    ap.add_argument("--ensemble-steps", type=int, default=3,
                    help="timed large steps per form of the 32-member ensemble leg; 0 skips it")
    ap.add_argument("--breakdown-steps", type=int, default=3,
                    help="untimed steps after the timed region with every kernel timed (0 skips)")
    ap.add_argument("--calibration-copy-mib", type=int, default=0,
                    help="also run one device-to-device copy of this many MiB (counter calibration)")
    ap.add_argument("--pmc-summary", nargs=2, metavar=("FETCH_DIR", "WRITE_DIR"),
                    help="summarise rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE output directories and exit")
    return ap.parse_args()


def pmc_summary(fetch_dir: str, write_dir: str, copy_mib: int) -> dict:
    """Per-kernel average FETCH_SIZE / WRITE_SIZE (KiB per dispatch) from two
    rocprofv3 --pmc runs, plus the same counters on the calibration copy (the
    largest copy dispatch, `copy_mib` MiB read and written)."""

    import glob
    import re
    import sqlite3

    def read(d, counter):
        db = glob.glob(os.path.join(d, "**", "*.db"), recursive=True)
        if not db:
            raise SystemExit(f"no rocprofv3 database under {d}")
        con = sqlite3.connect(db[0])
        per, copies = {}, []
        for name, cname, val in con.execute("select name, counter_name, counter_value from pmc_events"):
            if cname != counter:
                continue
            m = re.search(r"::(k_\w+)", name)
            if "copyBuffer" in name:
                copies.append(val)
            if m:
                per.setdefault(m.group(1), []).append(val)
        return {k: sum(v) / len(v) for k, v in per.items()}, (max(copies) if copies else None)

    fetch, fetch_copy = read(fetch_dir, "FETCH_SIZE")
    write, write_copy = read(write_dir, "WRITE_SIZE")
    return {
        "unit": "KiB per dispatch (rocprofv3 FETCH_SIZE / WRITE_SIZE)",
        "calibration": {"copy_bytes": copy_mib << 20, "fetch_kib": fetch_copy, "write_kib": write_copy},
        "kernels": {k: {"fetch_kib": fetch[k], "write_kib": write.get(k)} for k in sorted(fetch)},
    }


def traffic_for(kernel: str):
    """HBM bytes per launch of `kernel` from the committed counter summary:
    each counter scaled by what it reads for the plain calibration copy."""

    if not os.path.exists(TRAFFIC_FILE):
        return None, None
    with open(TRAFFIC_FILE) as f:
        summ = json.load(f)
    cal = summ["calibration"]
    k = summ["kernels"].get(kernel)
    if not k or not cal.get("fetch_kib") or not cal.get("write_kib") or k.get("write_kib") is None:
        return None, None
    f_scale = cal["copy_bytes"] / (cal["fetch_kib"] * 1024.0)
    w_scale = cal["copy_bytes"] / (cal["write_kib"] * 1024.0)
    bytes_ = k["fetch_kib"] * 1024.0 * f_scale + k["write_kib"] * 1024.0 * w_scale
    return bytes_, {"fetch_scale": round(f_scale, 3), "write_scale": round(w_scale, 3),
                    "source": os.path.relpath(TRAFFIC_FILE, ROOT)}


def field_errors(got: dict, ref: dict) -> dict:
    """Per field: [max|got-ref| / max|ref|, rms(got-ref) / rms(ref)]."""

    import torch

    out = {}
    for k in ref:
        d = (got[k] - ref[k]).abs()
        mx = float(ref[k].abs().max())
        rms = float(ref[k].pow(2).mean().sqrt())
        out[k] = [float(d.max()) / mx if mx > 0 else float(d.max()),
                  float(d.pow(2).mean().sqrt()) / rms if rms > 0 else float(d.pow(2).mean().sqrt())]
    return out


def timed_steps(step, n: int, stream) -> float:
    """Wall milliseconds of `step(n)` between HIP events on `stream`."""

    import torch

    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    a.record(stream)
    step(n)
    b.record(stream)
    torch.cuda.synchronize()
    return a.elapsed_time(b)


def mixed_form_leg(case, steps: int, fp64_ms_per_step: float, dev) -> dict:
    """The mixed-precision form on the same workload: throughput over `steps`
    large steps from the initial state, and the per-field error against the
    plain FP64 form after the same steps from the same state."""

    import torch

    from wrf_gpu_amd.dycore import Dycore, state_to_device

    m, nl = case.metrics, case.namelist
    stream = torch.cuda.current_stream(dev)
    runs = {}
    for prec in ("mixed", "fp64"):
        dyn = Dycore(m, nl, precision=prec)
        st = state_to_device(case.state, dev)
        ms = timed_steps(lambda n: dyn.step(st, n), steps, stream)
        runs[prec] = (st, ms / steps)
        dyn.close()
    ms_mixed = runs["mixed"][1]
    value = m.n_cells * nl.acoustic_substeps / (ms_mixed * 1e-3)
    errs = field_errors(runs["mixed"][0], runs["fp64"][0])
    return {"form": "mixed", "value": value, "unit": "cell-substeps/s", "ms_per_step": ms_mixed, "steps": steps,
            "speedup_vs_fp64": fp64_ms_per_step / ms_mixed,
            "fp64_ms_per_step_same_run": runs["fp64"][1],
            "error_vs_fp64_after_steps": {k: [float(f"{a:.3e}"), float(f"{b:.3e}")] for k, (a, b) in errs.items()},
            "error_columns": ["max|mixed-fp64|/max|fp64|", "rms(mixed-fp64)/rms(fp64)"],
            "max_rel_err": max(a for a, _ in errs.values()),
            "note": "the plain FP64 form is bit-identical to the CPU oracle (GPU parity tests), so this is the "
                    "error against the oracle"}


def diffusion_leg(case, steps: int, fp64_ms_per_step: float, dev, kind: str) -> dict:
    """The same workload with explicit diffusion on: throughput, and its
    kernels' rate over their algorithmic bytes per RK stage (each array
    they must read or write counted once; the tendency kernels then read the
    diffusion tendencies back, a cost included in the step time).

    kind "filter": the 6th-order filter (diff_6th_opt = 2), k_diff6, which
    reads u, v, w, theta and writes one coupled tendency for each.
    kind "smagorinsky": the 2-D Smagorinsky diffusion (diff_opt 1,
    km_opt 4), k_smag: the viscosity from u and v (read 2 fields, write K),
    then the four flux divergences (read each field and K, write its
    tendency).
    kind "limiter": the monotonic limiter on theta's advection in the final
    RK stage (scalar_adv_opt 2), k_limiter (three kernels), once per large
    step in place of that stage's plain theta advection, against the bytes
    of the two-pass scheme: the scales (read theta, the origin theta, ru,
    rv, rom; write the inflow and outflow scales), then the limited
    divergence (read the same five and the two scales; write the
    tendency).
    kind "constk": the constant-K diffusion (const_nu_m2_s = 75), k_constk:
    the grid-mean layer thickness (read ph_total, write and read one sum per
    column), then the four flux divergences (read each field, write its
    tendency)."""

    import torch

    from wrf_gpu_amd.dycore import Dycore, state_to_device

    m = case.metrics
    nx, ny, nz = m.nx, m.ny, m.nz
    eu, ev, ew, em = nz * ny * (nx + 1), nz * (ny + 1) * nx, (nz + 1) * ny * nx, nz * ny * nx
    if kind == "filter":
        nl, kernel, form = case.namelist.replace(diff_6th_opt=2), "k_diff6", "diff_6th_opt=2"
        alg_bytes = 2 * 8 * (eu + ev + ew + em)
    elif kind == "smagorinsky":
        nl, kernel, form = case.namelist.replace(diff_opt=1, km_opt=4), "k_smag", "diff_opt=1,km_opt=4"
        alg_bytes = 8 * ((eu + ev + em) + 2 * (eu + ev + ew + em) + 4 * em)
    elif kind == "constk":
        nl, kernel, form = case.namelist.replace(const_nu_m2_s=75.0), "k_constk", "const_nu_m2_s=75"
        alg_bytes = 8 * (ew + 2 * ny * nx + 2 * (eu + ev + ew + em))
    else:
        nl, kernel, form = case.namelist.replace(scalar_adv_opt=2), "k_limiter", "scalar_adv_opt=2"
        alg_bytes = 8 * ((4 * em + ew + 2 * em) + (4 * em + ew + 2 * em + em))
    stream = torch.cuda.current_stream(dev)
    dyn = Dycore(m, nl)
    st = state_to_device(case.state, dev)
    ms = timed_steps(lambda n: dyn.step(st, n), steps, stream) / steps
    dyn.profile([kernel])
    dyn.step(st, 2)
    torch.cuda.synchronize(dev)
    tot_ms, launches = dyn.profile_read()[kernel]
    dyn.close()
    avg = tot_ms / launches
    return {"form": form, "value": m.n_cells * nl.acoustic_substeps / (ms * 1e-3),
            "unit": "cell-substeps/s", "ms_per_step": ms, "steps": steps,
            "overhead_vs_fp64": ms / fp64_ms_per_step,
            kernel: {"avg_ms_per_stage": avg, "alg_bytes_per_stage": alg_bytes,
                     "achieved_GBs": alg_bytes / (avg * 1e-3) / 1e9, "peak_GBs": 8000.0,
                     "frac": alg_bytes / (avg * 1e-3) / 8e12}}


def moist_leg(case, steps: int, fp64_ms_per_step: float, dev) -> dict:
    """The same workload carrying the six moisture species (ic.with_moisture:
    qv decaying with height, cloud and precipitation blobs), coupled into the
    dynamics and transported with the monotonic limiter on the final stage
    (moist = 1, moist_adv_opt = 2): throughput, and per large step the
    moisture kernels against their algorithmic bytes.

    k_moist per step: three times the factors (read six species, write cqu,
    cqv and the raw cqw), two stages of plain flux advection of each species
    (read it, ru, rv, rom; write its tendency) and one stage of the two-pass
    limiter per species (the theta limiter's bytes).  k_moist_update per
    step: three updates (read six origin species and six tendencies, write
    six species; the 2-D masses are negligible)."""

    import torch

    from wrf_gpu_amd import ic
    from wrf_gpu_amd.dycore import Dycore, state_to_device

    mcase = ic.with_moisture(case, moist_adv_opt=2)
    m, nl = mcase.metrics, mcase.namelist
    nx, ny, nz = m.nx, m.ny, m.nz
    eu, ev, ew, em = nz * ny * (nx + 1), nz * (ny + 1) * nx, (nz + 1) * ny * nx, nz * ny * nx
    factors = 8 * (6 * em + eu + ev + ew)
    plain = 8 * (4 * em + ew)
    limited = 8 * ((4 * em + ew + 2 * em) + (4 * em + ew + 2 * em + em))
    alg = {"k_moist": 3 * factors + 6 * (2 * plain + limited), "k_moist_update": 3 * 8 * 18 * em}
    stream = torch.cuda.current_stream(dev)
    dyn = Dycore(m, nl)
    st = state_to_device(mcase.state, dev)
    ms = timed_steps(lambda n: dyn.step(st, n), steps, stream) / steps
    finite = all(bool(torch.isfinite(t).all()) for t in st.values())
    dyn.profile(list(alg))
    dyn.step(st, 2)
    torch.cuda.synchronize(dev)
    prof = dyn.profile_read()
    dyn.close()
    out = {"form": "moist=1,moist_adv_opt=2", "value": m.n_cells * nl.acoustic_substeps / (ms * 1e-3),
           "unit": "cell-substeps/s", "ms_per_step": ms, "steps": steps,
           "overhead_vs_fp64": ms / fp64_ms_per_step, "finite": finite}
    for k, b in alg.items():
        tot_ms, _ = prof[k]
        per_step = tot_ms / 2
        out[k] = {"ms_per_step": per_step, "alg_bytes_per_step": b, "achieved_GBs": b / (per_step * 1e-3) / 1e9,
                  "peak_GBs": 8000.0, "frac": b / (per_step * 1e-3) / 8e12}
    del st
    torch.cuda.empty_cache()
    return out


def small_workload_leg(steps: int, dev) -> dict:
    """The 64x64x40 warm bubble (dt 6 s, ns 6): a launch-bound size, stepped
    eagerly, by replaying the graph-captured large step, and as a one-member
    persistent step, then by the autotuned graph and the autotuned persistent
    step."""

    import torch

    from wrf_gpu_amd import ic
    from wrf_gpu_amd.dycore import Dycore, Ensemble, state_to_device

    case = ic.bubble_3d()
    m, nl = case.metrics, case.namelist
    stream = torch.cuda.current_stream(dev)
    out = {"workload": "plain FP64 dry 3-D warm bubble 64x64x40, dx=1 km, dt=6 s, ns=6", "n_cells": m.n_cells,
           "steps": steps}
    eager, graphed = Dycore(m, nl), Dycore(m, nl)
    se, sg = state_to_device(case.state, dev), state_to_device(case.state, dev)
    eager.step(se, 1)
    graphed.capture_graph(sg)
    graphed.graph_step(1)
    for name, fn in (("eager", lambda n: eager.step(se, n)), ("graph", lambda n: graphed.graph_step(n))):
        ms = timed_steps(fn, steps, stream) / steps
        out[name] = {"ms_per_step": ms, "value": m.n_cells * nl.acoustic_substeps / (ms * 1e-3)}
    out["graph_speedup"] = out["eager"]["ms_per_step"] / out["graph"]["ms_per_step"]
    out["graph_equals_eager"] = all(bool(torch.equal(se[k], sg[k])) for k in se)
    # the persistent step with this one member: one launch per large step instead of ~85
    pers = Dycore(m, nl)
    sp = state_to_device(case.state, dev)
    ens = Ensemble([(pers, sp)], persistent=True)
    ens.step(1)
    ens.status()
    ms = timed_steps(ens.step, steps, stream) / steps
    ens.status()
    out["persistent"] = {"ms_per_step": ms, "value": m.n_cells * nl.acoustic_substeps / (ms * 1e-3),
                         "workgroups": ens.workgroups}
    out["persistent_equals_eager"] = all(bool(torch.equal(se[k], sp[k])) for k in se)
    ens.close()
    pers.close()
    # the autotuner's pick for this size (k-marching kernels have one wave per 64 columns here)
    out["autotuned_config"] = graphed.autotune(sg, trial_steps=2)
    graphed.capture_graph(sg)
    graphed.graph_step(1)
    ms = timed_steps(lambda n: graphed.graph_step(n), steps, stream) / steps
    out["autotuned_graph"] = {"ms_per_step": ms, "value": m.n_cells * nl.acoustic_substeps / (ms * 1e-3)}
    # the persistent step with the autotuned handle: its column tile runs inside the launch
    ens = Ensemble([(graphed, sg)], persistent=True)
    ens.step(1)
    ens.status()
    ms = timed_steps(ens.step, steps, stream) / steps
    ens.status()
    out["persistent_autotuned"] = {"ms_per_step": ms, "value": m.n_cells * nl.acoustic_substeps / (ms * 1e-3),
                                   "workgroups": ens.workgroups, "column_kernel": ens.column_kernel(0)}
    ens.close()
    eager.close()
    graphed.close()
    return out


def ensemble_leg(steps: int, dev) -> dict:
    """32 members (8 each of 129^2, 201^2, 257^2, 321^2 columns, 50 levels):
    members stepped one after another with the plain step, then the batched
    graph (4 branches) and the persistent step (one launch per large step),
    each in FP64 and in the mixed form, and the batched graph and the
    persistent step in FP64 with each member's autotuned column kernel and
    workgroup order."""

    import torch

    from wrf_gpu_amd import ic
    from wrf_gpu_amd.dycore import Dycore, Ensemble, state_to_device

    t0 = time.time()
    cases = ic.ensemble_32()
    members = [(Dycore(c.metrics, c.namelist), state_to_device(c.state, dev)) for c in cases]
    del cases
    cells = sum(d.metrics.n_cells for d, _ in members)
    ns = members[0][0].namelist.acoustic_substeps
    print(f"[bench] ensemble of {len(members)} members built in {time.time() - t0:.1f}s", file=sys.stderr, flush=True)
    stream = torch.cuda.current_stream(dev)

    def seq(n):
        for _ in range(n):
            for d, s in members:
                d.step(s, 1)

    out = {"workload": "32 members, 8 each of 129x129, 201x201, 257x257, 321x321, 50 levels, flat neutral base of "
                       "the 64x64x40 warm-bubble workload, correlated theta' (0.5 K) and u' (1 m/s), seeds 100+m",
           "n_cells": cells, "members": len(members), "steps": steps}
    seq(1)
    ms = timed_steps(seq, steps, stream) / steps
    out["sequential_fp64"] = {"ms_per_step": ms, "value": cells * ns / (ms * 1e-3)}
    for prec in ("fp64", "mixed"):
        for d, _ in members:
            d.set_precision(prec)
        ens = Ensemble(members, branches=4)
        ens.step(1)
        ms = timed_steps(ens.step, steps, stream) / steps
        out[f"batched_graph_{prec}"] = {"ms_per_step": ms, "value": cells * ns / (ms * 1e-3),
                                        "branches": ens.branches}
        ens.close()
        # one persistent launch per large step (the barrier's report is checked after the timing)
        ens = Ensemble(members, persistent=True)
        ens.step(1)
        ens.status()
        ms = timed_steps(ens.step, steps, stream) / steps
        ens.status()
        out[f"persistent_{prec}"] = {"ms_per_step": ms, "value": cells * ns / (ms * 1e-3),
                                     "workgroups": ens.workgroups}
        ens.close()
    # the batched FP64 graph with every member's autotuned column kernel and workgroup order
    for d, _ in members:
        d.set_precision("fp64")
    t1 = time.time()
    ens = Ensemble(members, branches=4, autotune=True, trial_steps=1)
    tune_s = time.time() - t1
    ens.step(1)
    ms = timed_steps(ens.step, steps, stream) / steps
    picks = {}
    tuned = list(ens.tuned)
    for cfg in ens.tuned:
        key = f"column_tile={cfg['column_tile']},xcd_remap={cfg['xcd_remap']}"
        picks[key] = picks.get(key, 0) + 1
    out["batched_graph_fp64_autotuned"] = {"ms_per_step": ms, "value": cells * ns / (ms * 1e-3),
                                           "branches": ens.branches, "member_picks": picks,
                                           "trial": ens.batch_trial, "autotune_s": tune_s}
    ens.close()
    # the persistent step with the members' picks made alone: tuned 16x16 column tiles run inside the launch
    for (d, _), cfg in zip(members, tuned):
        d.set_tuned_config(cfg["column_tile"], cfg["xcd_remap"])
    ens = Ensemble(members, persistent=True)
    ens.step(1)
    ens.status()
    ms = timed_steps(ens.step, steps, stream) / steps
    ens.status()
    kernels = [ens.column_kernel(q) for q in range(len(members))]
    out["persistent_fp64_member_tuned"] = {"ms_per_step": ms, "value": cells * ns / (ms * 1e-3),
                                           "workgroups": ens.workgroups,
                                           "members_on_column_tile": sum(k >= 0 for k in kernels)}
    ens.close()
    # the autotuned persistent step: members tuned alone, then the step timed with their tiles and with
    # every member off its tile, the faster kept
    ens = Ensemble(members, persistent=True, autotune=True, trial_steps=1)
    ens.step(1)
    ens.status()
    ms = timed_steps(ens.step, steps, stream) / steps
    ens.status()
    kernels = [ens.column_kernel(q) for q in range(len(members))]
    out["persistent_fp64_autotuned"] = {"ms_per_step": ms, "value": cells * ns / (ms * 1e-3),
                                        "workgroups": ens.workgroups, "trial": ens.persistent_trial,
                                        "members_on_column_tile": sum(k >= 0 for k in kernels)}
    ens.close()
    base = out["sequential_fp64"]["ms_per_step"]
    out["speedup_vs_sequential_fp64"] = {k: base / out[k]["ms_per_step"]
                                         for k in ("batched_graph_fp64", "batched_graph_mixed",
                                                   "persistent_fp64", "persistent_mixed",
                                                   "batched_graph_fp64_autotuned", "persistent_fp64_member_tuned",
                                                   "persistent_fp64_autotuned")}
    for d, _ in members:
        d.close()
    return out


def main():
    args = parse()
    if args.pmc_summary:
        print(json.dumps(pmc_summary(*args.pmc_summary, args.calibration_copy_mib or 1024), indent=1))
        return
    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print(json.dumps({"error": "this build runs on one GPU: sharding across GPUs is designed but not "
                                   "built, so only --gpus 1 is measured", "n_gpus": args.gpus}))
        sys.exit(2)

    import torch

    from wrf_gpu_amd import _lib, ic
    from wrf_gpu_amd.dycore import Dycore, state_to_device

    if not torch.cuda.is_available():
        print(json.dumps({"error": "no GPU visible"}))
        sys.exit(1)

    t0 = time.time()
    case = ic.stratified_terrain_3d(nx=args.nx, ny=args.ny, nz=args.nz)
    m, nl = case.metrics, case.namelist
    n_cells = m.n_cells
    print(f"[bench] IC {m.nx}x{m.ny}x{m.nz} built in {time.time() - t0:.1f}s", file=sys.stderr, flush=True)

    dev = torch.device("cuda:0")
    state = state_to_device(case.state, dev)
    dyn = Dycore(m, nl)
    stream = torch.cuda.current_stream(dev)

    if args.calibration_copy_mib > 0:
        # a plain copy of known size: HBM byte counters read on it calibrate
        # the counters read on the dycore kernels
        n = args.calibration_copy_mib * (1 << 20) // 8
        src = torch.ones(n, dtype=torch.float64, device=dev)
        dst = torch.empty_like(src)
        dst.copy_(src)
        torch.cuda.synchronize()
        del src, dst

    # warmup
    dyn.step(state, args.warmup)
    torch.cuda.synchronize()
    print(f"[bench] warmup {args.warmup} steps done", file=sys.stderr, flush=True)

    # timed region; the candidate dominant kernels carry HIP events on the launch stream
    names = _lib.kernel_names()
    profiled = [k for k in ("k_column", "k_column_block", "k_column_mu", "k_column_w", "k_uv") if k in names]
    dyn.profile(profiled)
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    start.record(stream)
    dyn.step(state, args.steps)
    end.record(stream)
    torch.cuda.synchronize()
    wall_ms = start.elapsed_time(end)
    kern = dyn.profile_read()
    dyn.profile(())
    print(f"[bench] timed {args.steps} steps: {wall_ms:.1f} ms", file=sys.stderr, flush=True)

    finite = all(bool(torch.isfinite(t).all()) for t in state.values())
    ms_per_step = wall_ms / max(args.steps, 1)
    ns = nl.acoustic_substeps
    value = n_cells * ns * args.steps / (wall_ms / 1e3)
    executed = n_cells * (1 + max(1, ns // 2) + ns) * args.steps / (wall_ms / 1e3)

    # roofline of the dominant profiled kernel
    per_kernel = {}
    for name, (ms, cnt) in kern.items():
        avg_ms = ms / cnt
        alg = ALG_ARRAYS_PER_CELL[name] * 8 * n_cells
        per_kernel[name] = {"avg_ms": avg_ms, "launches": cnt, "share_of_wall": ms / wall_ms,
                            "alg_bytes": alg, "achieved_GBs": alg / (avg_ms * 1e-3) / 1e9}
    dom = max(per_kernel, key=lambda k: per_kernel[k]["avg_ms"] * per_kernel[k]["launches"])
    d = per_kernel[dom]
    traffic, traffic_info = traffic_for(dom)
    roofline = {"bound": "hbm", "kernel": dom, "achieved": round(d["achieved_GBs"], 1), "peak": HBM_PEAK_GBS,
                "unit": "GB/s", "frac": round(d["achieved_GBs"] / HBM_PEAK_GBS, 4),
                "traffic": None if traffic is None else round(traffic),
                "alg_bytes_per_launch": d["alg_bytes"], "avg_launch_ms": round(d["avg_ms"], 4)}
    if traffic_info:
        roofline["traffic_calibration"] = traffic_info
        roofline["traffic_GBs"] = round(traffic / (d["avg_ms"] * 1e-3) / 1e9, 1)
    step_bytes = step_bytes_per_cell(ns) * n_cells
    step_roofline = {"model_bytes_per_step": step_bytes,
                     "achieved": round(step_bytes / (ms_per_step * 1e-3) / 1e9, 1), "unit": "GB/s",
                     "frac": round(step_bytes / (ms_per_step * 1e-3) / 1e9 / HBM_PEAK_GBS, 4)}

    # untimed per-kernel breakdown: every kernel bracketed by events
    breakdown = None
    if args.breakdown_steps > 0:
        dyn.profile(names)
        dyn.step(state, args.breakdown_steps)
        torch.cuda.synchronize()
        br = dyn.profile_read()
        dyn.profile(())
        breakdown = {k: {"avg_ms": round(v[0] / v[1], 4), "ms_per_step": round(v[0] / args.breakdown_steps, 4)}
                     for k, v in sorted(br.items(), key=lambda kv: -kv[1][0])}

    # CPU baseline: the oracle (a C restatement of the reference path) on a
    # bounded sample of the same workload
    cpu = None
    if args.cpu_baseline_steps > 0:
        from oracle import oracle

        threads = args.cpu_threads or len(os.sched_getaffinity(0))
        oracle.build()
        t1 = time.time()
        oracle.run(m, nl, case.state, args.cpu_baseline_steps, threads=threads)
        cpu_s = time.time() - t1
        cpu = {"value": n_cells * ns * args.cpu_baseline_steps / cpu_s, "unit": "cell-substeps/s",
               "cores": threads, "kind": "port",
               "sample": f"{args.cpu_baseline_steps} large step(s) of the same {m.nx}x{m.ny}x{m.nz} workload "
                         f"from the initial state, CPU oracle (C, OpenMP), {cpu_s:.1f} s"}
        print(f"[bench] cpu baseline {cpu_s:.1f}s on {threads} threads", file=sys.stderr, flush=True)
        if args.cpu_small_steps > 0:
            # the CPU-runnable 64x64x40 warm bubble, over the oracle as well
            small = ic.bubble_3d()
            t1 = time.time()
            oracle.run(small.metrics, small.namelist, small.state, args.cpu_small_steps, threads=threads)
            small_s = time.time() - t1
            cpu["small_workload"] = {
                "value": small.metrics.n_cells * small.namelist.acoustic_substeps * args.cpu_small_steps / small_s,
                "unit": "cell-substeps/s", "cores": threads,
                "sample": f"{args.cpu_small_steps} large steps of the 64x64x40 warm bubble (dt=6 s, ns=6), "
                          f"CPU oracle (C, OpenMP), {small_s:.1f} s"}
            print(f"[bench] cpu baseline, 64x64x40: {small_s:.1f}s", file=sys.stderr, flush=True)

    # the layered forms: mixed precision on this workload, and the batched ensemble
    forms = {}
    if args.graph_steps > 0:
        # the same step captured once into a HIP graph and replayed (wd_capture_graph / wd_graph_step)
        gdyn = Dycore(m, nl)
        gst = state_to_device(case.state, dev)
        gdyn.capture_graph(gst)
        gdyn.graph_step(1)
        gms = timed_steps(lambda n: gdyn.graph_step(n), args.graph_steps, torch.cuda.current_stream(dev))
        gms /= args.graph_steps
        forms["graph_replay"] = {"ms_per_step": gms, "value": n_cells * ns / (gms * 1e-3), "steps": args.graph_steps,
                                 "vs_eager": ms_per_step / gms}
        gdyn.close()
        del gst
        print(f"[bench] graph replay leg done", file=sys.stderr, flush=True)
    if args.form_steps > 0:
        forms["mixed"] = mixed_form_leg(case, args.form_steps, ms_per_step, dev)
        print(f"[bench] mixed form leg done", file=sys.stderr, flush=True)
    if args.filter_steps > 0:
        forms["filter"] = diffusion_leg(case, args.filter_steps, ms_per_step, dev, "filter")
        print(f"[bench] filter leg done", file=sys.stderr, flush=True)
    if args.smagorinsky_steps > 0:
        forms["smagorinsky"] = diffusion_leg(case, args.smagorinsky_steps, ms_per_step, dev, "smagorinsky")
        print(f"[bench] smagorinsky leg done", file=sys.stderr, flush=True)
    if args.limiter_steps > 0:
        forms["limiter"] = diffusion_leg(case, args.limiter_steps, ms_per_step, dev, "limiter")
        print(f"[bench] limiter leg done", file=sys.stderr, flush=True)
    if args.constk_steps > 0:
        forms["constk"] = diffusion_leg(case, args.constk_steps, ms_per_step, dev, "constk")
        print(f"[bench] constant-K leg done", file=sys.stderr, flush=True)
    if args.moist_steps > 0:
        forms["moist"] = moist_leg(case, args.moist_steps, ms_per_step, dev)
        print(f"[bench] moist leg done", file=sys.stderr, flush=True)
    if args.small_steps > 0:
        forms["small_workload"] = small_workload_leg(args.small_steps, dev)
        print(f"[bench] small workload leg done", file=sys.stderr, flush=True)
    if args.ensemble_steps > 0:
        dyn.close()
        del state
        torch.cuda.empty_cache()
        forms["batched_ensemble"] = ensemble_leg(args.ensemble_steps, dev)
        print(f"[bench] ensemble leg done", file=sys.stderr, flush=True)

    out = {
        "metric": METRIC,
        "value": value,
        "unit": "cell-substeps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_per_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": {"workload": f"plain FP64 stratified flow over terrain {m.nx}x{m.ny}x{m.nz}, dx=3 km, "
                               f"stretched eta, dt={nl.dt_s:g} s, ns={ns}",
                   "n_cells": n_cells, "form": "plain_fp64", "parallelism": "single GPU"},
        "executed_cell_substeps_per_s": executed,
        "roofline": roofline,
        "step_roofline": step_roofline,
        "kernels": {k: {kk: (round(vv, 5) if isinstance(vv, float) else vv) for kk, vv in v.items()}
                    for k, v in per_kernel.items()},
        "kernel_breakdown": breakdown,
        "cpu_baseline": cpu,
        "forms": forms or None,
        "finite": finite,
    }
    print(json.dumps(out))
    dyn.close()


if __name__ == "__main__":
    main()
