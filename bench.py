#!/usr/bin/env python3
"""Benchmark: LJ energy grids + Widom insertion over the batching mix.

Workload (default): 256 synthetic frameworks, atoms log-uniform in [50,5000],
cell lengths U[8,40] A, angles U[60,120] deg, grid spacing in {0.1,0.2,0.5} A
(FP32 grids), 1e6 Widom insertions each at 298 K, guests CH4/Xe/Kr, r_c 12.5 A.

A step is one pass of the hot path over the whole batch: every grid and every
Widom run, launched as one batch (binning kernels, a persistent tiled-kernel launch
for each of its variants, reductions).  Inputs are resident in HBM before the timed region.
After the timed steps, the default run also measures:
- the plain path (one framework per launch, synchronous, grids left
  resident as the batch leaves them) on the same work: batched/plain, against
  the workload's 5x target;
- the tiled kernels on the step's grids alone (the roofline launches: 16 FLOP
  for every in-cutoff grid pair, VALU-bound; the far pairs of fine grids are
  evaluated at an eighth of the points and interpolated) and on its Widom
  runs alone (an insertion rate: saturated insertions stop early);
- the same step with FP64 grids (the drop-in writegrid's default precision)
  and the FP64 grids alone against the FP64 vector peak;
- the reference's direct method on the same GPU (FP64, every (point, image,
  atom) triple, one framework per launch) on a sample of the mix, scaled to
  the whole mix by pair-evals, with the batch's errors against it;
- the FP64 oracle on the host (all the cores this job may use, and one) on
  a bounded sample of the mix, and the plain-method config in full;
- a serving leg: Poisson arrivals at 500 requests/s for 2 s into the
  continuous-batching server (p50/p99 latency, sustained requests/s,
  rejections, framework uploads avoided by residency).

value = pair-evals/s in the reference's enumeration (P*N*I for grids plus
n_ins*N*I for Widom, the same count for every path), so a rate of the
reference's work, not of pairs evaluated here: interpolated far fields and
saturated insertions count in full.  roofline.achieved likewise is the direct
method's work per second; roofline.valu_issue is the share of the device's
VALU issue slots that the launches use (instructions from the committed
counters).
"""
import argparse
import json
import math
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

PEAK_FP32_TFLOPS = 157.3  # MI355X FP32 vector peak (packed FP32)
PEAK_FP32_UNPACKED_TFLOPS = 78.6  # without packed FP32, as this build compiles
PEAK_FP64_TFLOPS = 78.6  # MI355X FP64 vector peak
VALU_ISSUE_PER_S = 256 * 2.4e9  # wave instructions: one a clock and CU (four SIMDs, four clocks)
TARGET_BATCHED_OVER_PLAIN = 5.0
DEFAULT_TUNING_FILE = os.path.join(ROOT, "emptyroom_amd", "tuning", "mi355x_config3.json")
WORKLOAD_TEXT = {
    "config3": "config3: {n} frameworks, grids FP32 at 0.1/0.2/0.5 A + 1e6 Widom insertions "
               "each, one batched launch",
    "config2": "config2: one 3000-atom triclinic framework, FP32 grid at 0.1 A + 1e7 Widom "
               "insertions, one batched launch",
    "config1": "config1: one 400-atom cubic framework, grid at 0.5 A (FP32 here) + 1e5 Widom "
               "insertions, one batched launch",
}
FLOP_PER_PAIR = 16


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def make_workload(name, count):
    from emptyroom_amd import synth
    if name == "config3":
        return synth.config3(count)
    if name == "config2":
        return [synth.config2()]
    if name == "config1":
        return [synth.config1()]
    raise SystemExit(f"unknown workload {name}")


def pair_evals(f):
    n = f.grid_n()
    img = (2 * f.rep[0] + 1) * (2 * f.rep[1] + 1) * (2 * f.rep[2] + 1)
    grid = n[0] * n[1] * n[2] * f.n_atoms * img
    widom = f.n_insertions * f.n_atoms * img
    return grid, widom


def host_cpu():
    """Host CPU facts for the baseline: logical CPUs, the ones this process may
    use, the thread budget of the job (OMP_NUM_THREADS) and the model name."""
    model = None
    try:
        with open("/proc/cpuinfo") as fh:
            for line in fh:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    try:
        usable = len(os.sched_getaffinity(0))
    except (AttributeError, OSError):
        usable = os.cpu_count() or 1
    omp = os.environ.get("OMP_NUM_THREADS", "")
    budget = int(omp) if omp.isdigit() and int(omp) > 0 else usable
    return dict(nproc=os.cpu_count(), usable=usable, omp_num_threads=omp or None,
                threads=max(1, min(usable, budget)), model=model)


def cpu_baseline(fws, uploaded, ctx, batch, budget_s, threads, every=16):
    """Time the oracle on a bounded sample; also report GPU errors on it."""
    from emptyroom_amd import api
    from oracle import oracle
    # sample: every `every`-th framework of the mix, a few x-sheets and the
    # first insertions of each, sized by a quick calibration of the oracle's rate
    idx = list(range(0, len(fws), max(1, every)))
    f0 = fws[idx[0]]
    a0 = f0.particles()
    t0 = time.perf_counter()
    oracle.lj_grid(f0.t, a0, f0.rep, f0.rc2, f0.grid_n(), sheets=(0, 1, 1), nthreads=threads)
    dt = time.perf_counter() - t0
    n0 = f0.grid_n()
    rate0 = n0[1] * n0[2] * f0.n_atoms * (2 * f0.rep[0] + 1) * (2 * f0.rep[1] + 1) * \
        (2 * f0.rep[2] + 1) / max(dt, 1e-6)
    per_fw = budget_s * rate0 / len(idx)
    evals = 0
    secs = 0.0
    grid_err = 0.0
    kh_err = 0.0
    e_err = 0.0
    n_grid_cmp = n_kh_cmp = 0  # points with E < 1e4 K / runs with a nonzero sum compared
    for i in idx:
        f = fws[i]
        a = f.particles()
        n = f.grid_n()
        img = (2 * f.rep[0] + 1) * (2 * f.rep[1] + 1) * (2 * f.rep[2] + 1)
        per_sheet = n[1] * n[2] * f.n_atoms * img
        nsheets = max(1, min(n[0], int(0.5 * per_fw / per_sheet)))
        step = max(1, n[0] // nsheets)
        sheets = (0, n[0], step)
        nins = int(max(64, min(f.n_insertions, 0.5 * per_fw / (f.n_atoms * img))))
        t0 = time.perf_counter()
        ref = oracle.lj_grid(f.t, a, f.rep, f.rc2, n, sheets=sheets, nthreads=threads)
        rb, reb = oracle.widom(f.t, a, f.rep, f.rc2, f.temperature, f.seed, 0, nins,
                               nthreads=threads)
        secs += time.perf_counter() - t0
        evals += len(range(*sheets)) * per_sheet + nins * f.n_atoms * img
        g = batch.grid(i)[sheets[0]:sheets[1]:sheets[2]].astype(np.float64)
        m = ref < 1e4
        if m.any():
            grid_err = max(grid_err, float(np.max(np.abs(g[m] - ref[m]))))
            n_grid_cmp += int(m.sum())
        sb, seb, _ = api.widom(ctx, uploaded[i], nins, f.temperature, f.seed)
        if rb > 0:
            kh_err = max(kh_err, abs(sb - rb) / rb)
            e_err = max(e_err, abs(seb / sb - reb / rb))
            n_kh_cmp += 1
        elif sb != 0:
            kh_err = float("inf")
            n_kh_cmp += 1
    # nothing comparable (every sampled point blocked): no error figure
    if n_grid_cmp == 0:
        grid_err = None
    if n_kh_cmp == 0:
        kh_err = e_err = None
    sample = (f"{len(idx)} of {len(fws)} frameworks (every {every}-th), every k-th x-sheet of "
              f"each grid and the first insertions of each Widom run ({evals:.3g} pair-evals, "
              f"FP64 oracle, {threads} threads; rate extrapolated to the mix by pair-evals; "
              f"errors over {n_grid_cmp} grid points with E < 1e4 K and {n_kh_cmp} Widom runs "
              f"with a nonzero sum)")
    return dict(value=evals / secs, unit="pair-evals/s", cores=threads, kind="port",
                sample=sample, seconds=round(secs, 2)), grid_err, kh_err, e_err


def config1_full(api, synth, ctx, threads):
    """The plain-method config (400-atom cubic cell, 50^3 grid, 1e5 insertions)
    in full: the FP64 oracle on `threads` host threads and on one, and the
    GPU's plain path on the same work, with the GPU's errors against it."""
    from oracle import oracle
    f = synth.config1()
    a = f.particles()
    n = f.grid_n()
    img = (2 * f.rep[0] + 1) * (2 * f.rep[1] + 1) * (2 * f.rep[2] + 1)
    pe = (int(np.prod(n)) + f.n_insertions) * f.n_atoms * img
    out = {"workload": "config1: 400 atoms, 25 A cubic, 50^3 grid + 1e5 insertions at 298 K, "
                       "FP64 oracle in full", "pair_evals": pe}
    for th in sorted({threads, 1}, reverse=True):
        t0 = time.perf_counter()
        ref = oracle.lj_grid(f.t, a, f.rep, f.rc2, n, nthreads=th)
        rb, reb = oracle.widom(f.t, a, f.rep, f.rc2, f.temperature, f.seed, 0, f.n_insertions,
                               nthreads=th)
        dt = time.perf_counter() - t0
        out[f"cpu_seconds_{th}_threads"] = dt
        out[f"cpu_pair_evals_per_s_{th}_threads"] = pe / dt
    fw = api.Framework(ctx, a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2)
    api.compute_grid(ctx, fw, n, api.ER_FP32)  # untimed first call
    t0 = time.perf_counter()
    g = api.Grid.compute(ctx, fw, n, api.ER_FP32)
    sb, seb, _ = api.widom(ctx, fw, f.n_insertions, f.temperature, f.seed)
    gpu_s = time.perf_counter() - t0
    g32 = g.download().astype(np.float64)
    g.close()
    fw.close()
    m = ref < 1e4
    out.update(gpu_plain_seconds=gpu_s, gpu_pair_evals_per_s=pe / gpu_s,
               gpu_over_cpu=out[f"cpu_seconds_{threads}_threads"] / gpu_s,
               grid_max_abs_err_K=float(np.max(np.abs(g32[m] - ref[m]))) if m.any() else None,
               kh_rel_err=abs(sb - rb) / rb if rb > 0 else None)
    return out


def percentile(v, q):
    return float(np.percentile(np.asarray(v), q)) if len(v) else None


def serve_rate(api, synth, ctx, parts, rate, seconds, streams, items_per_launch, cycle=False,
               cache_bytes=-1):
    """One Poisson stream at `rate` requests/s for about `seconds` into a fresh
    server on ctx: grid / Henry requests on frameworks drawn (seeded) from the
    pool, or taken in turn with cycle; latency = completion - submission on the
    server's clock; grids stay resident in HBM and are released unread."""
    import threading
    n_req = max(50, int(rate * seconds))
    arrivals, kinds, temps = synth.config4_stream(rate, n_req)
    if cycle:
        pick = np.arange(n_req) % len(parts)
    else:
        pick = (synth.Rng(synth.framework_seed(4, 1)).u64(n_req) %
                np.uint64(len(parts))).astype(np.int64)
    srv = api.Server(ctx, streams=streams, items_per_launch=items_per_launch,
                     cache_bytes=cache_bytes)
    tickets, codes = [], []

    def submit_all():
        t0 = time.perf_counter()
        for i in range(n_req):
            dt = t0 + arrivals[i] - time.perf_counter()
            if dt > 0:
                time.sleep(dt)
            f, a = parts[pick[i]]
            if kinds[i] == 0:
                code, tk = srv.submit(a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2,
                                      grid_n=f.grid_n(), precision=api.ER_FP32)
            else:
                code, tk = srv.submit(a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2,
                                      n_insertions=f.n_insertions,
                                      temperature=float(temps[i]), seed=f.seed + i)
            codes.append(code)
            tickets.append(tk)

    th = threading.Thread(target=submit_all)
    th.start()
    th.join()
    lat, wait, run, t_first, t_last, done = [], [], [], None, None, 0
    for code, tk in zip(codes, tickets):
        if code != 0:
            continue
        st = srv.poll(tk, wait_ms=-1)
        if st.state == api.RQ_DONE:
            done += 1
            lat.append((st.t_done - st.t_submit) * 1e3)
            wait.append((st.t_admit - st.t_submit) * 1e3)
            run.append((st.t_done - st.t_admit) * 1e3)
            t_first = st.t_submit if t_first is None else min(t_first, st.t_submit)
            t_last = st.t_done if t_last is None else max(t_last, st.t_done)
        srv.release(tk)
    stats = srv.stats()
    cache = srv.cache_stats()
    srv.close()
    span = (t_last - t_first) if done else float("nan")
    return dict(rate=rate, requests=n_req, completed=done,
                rejected=stats["rejected"], rejection_rate=stats["rejected"] / n_req,
                p50_ms=percentile(lat, 50), p99_ms=percentile(lat, 99),
                admit_wait_p50_ms=percentile(wait, 50), admit_wait_p99_ms=percentile(wait, 99),
                run_p50_ms=percentile(run, 50), run_p99_ms=percentile(run, 99),
                sustained_req_per_s=done / span if done else 0.0,
                sustained_fws_per_s=done / span if done else 0.0,
                launches=stats["launches"], framework_uploads=cache["misses"],
                framework_cache_hits=cache["hits"],
                resident_frameworks=cache["resident_frameworks"])


def bench_serving(args, api, synth):
    """Poisson arrivals of grid / Henry requests into the continuous-batching
    server (HBM cap 200 GB)."""
    pool = [synth.config3_framework(i, config=4) for i in range(args.frameworks)]
    parts = [(f, f.particles()) for f in pool]
    ctx = api.Context(0, hbm_cap=200 << 30)
    rates = [float(r) for r in args.rates.split(",")]
    rows = []
    for rate in rates:
        row = serve_rate(api, synth, ctx, parts, rate, args.serve_seconds, args.streams,
                         args.items_per_launch, cycle=args.pick == "cycle",
                         cache_bytes=args.cache_bytes)
        log(f"serving rate {rate:g}/s: {json.dumps(row)}")
        rows.append(row)
    ctx.close()
    top = rows[-1]
    return {
        "metric": "serving: sustained frameworks/s under Poisson arrivals (grid + Henry mix)",
        "value": top["sustained_fws_per_s"], "unit": "frameworks/s", "n_gpus": 1,
        "steps": len(rates), "warmup": 0, "ms_per_step": None, "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None,
        "dtype": "fp32 pair LJ beyond 1.5 sigma, fp64 r^2 / close pairs / accumulation",
        "data": "synthetic (seeded SplitMix64 frameworks, Poisson arrivals)",
        "config": {"workload": "config4: Poisson arrivals of grid / Henry requests, frameworks "
                               "drawn from a pool of the batching mix, T ~ U[250,350] K, "
                               "HBM cap 200 GB",
                   "frameworks_in_pool": len(pool), "streams": args.streams,
                   "items_per_launch": args.items_per_launch, "pick": args.pick,
                   "cache_bytes": args.cache_bytes,
                   "seconds_per_rate": args.serve_seconds, "parallelism": "single GPU"},
        "rates": rows,
    }


def bench_pockets(args, api, synth):
    """Config 5: FP32 grids at 0.2 A, pocket blocking at 15 T, then 1e7
    grid-interpolated insertions per framework (blocked voxels are 1e13 K)."""
    from oracle import oracle
    T = 298.0
    fws = synth.config5(args.frameworks)
    ctx = api.Context(0)
    grids, fwh = [], []
    t0 = time.perf_counter()
    for f in fws:
        a = f.particles()
        fw = api.Framework(ctx, a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2)
        grids.append(api.Grid.compute(ctx, fw, f.grid_n(), api.ER_FP32))
        fwh.append(fw)
    t_grid = time.perf_counter() - t0
    # unblocked copies of every 8th grid for the physics check below
    check = list(range(0, len(fws), 8))
    unblocked = {i: api.Grid.upload(ctx, grids[i].download()) for i in check}
    voxels = sum(int(np.prod(f.grid_n())) for f in fws)
    log(f"{len(fws)} grids, {voxels:.3g} voxels in {t_grid:.2f} s")
    t0 = time.perf_counter()
    pockets = api.pockets_label_batch(ctx, grids, T, block=True)
    t_lab = time.perf_counter() - t0
    ins = 0
    kh = []
    t0 = time.perf_counter()
    for i, (f, g) in enumerate(zip(fws, grids)):
        sb, seb, n = api.widom_grid(ctx, g, f.n_insertions, T, f.seed)
        ins += n
        kh.append(sb / n)
    t_tri = time.perf_counter() - t0
    # batched GCMC-style energy calls: 1e7 positions on one grid, host buffers
    # in and out (PCIe included), after one untimed call
    rng = np.random.default_rng(2)
    pos = rng.uniform(-1.0, 2.0, (10_000_000, 3))
    api.grid_energies(ctx, grids[0], pos[:1000])
    t0 = time.perf_counter()
    api.grid_energies(ctx, grids[0], pos)
    t_en = time.perf_counter() - t0
    # Physics check of the workload: grid-interpolated K_H against the direct
    # FP64 sum (the reference's method on the GPU) at the direct method's
    # first 1e6 insertion points, on every 8th framework; and the trilinear
    # K_H of the blocked grid against the oracle at the same 1e7 points.
    phys = []
    m = 1_000_000
    for i in check:
        f = fws[i]
        a = f.particles()
        pts = oracle.widom_points(f.seed, 0, 0, m)
        e_un = api.grid_energies(ctx, unblocked[i], pts)
        e_bl = api.grid_energies(ctx, grids[i], pts)
        _, _, _, de = api.direct_widom(ctx, a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2, m, T,
                                       f.seed, energies=True)
        k_dir = float(np.exp(-de / T).sum())
        k_un = float(np.exp(-e_un / T).sum())
        open_ = e_bl == e_un
        k_dir_open = float(np.exp(-de[open_] / T).sum())
        k_bl = float(np.exp(-e_bl / T).sum())
        rb, _ = oracle.widom_grid(grids[i].download().astype(np.float64), T, f.seed, 0,
                                  f.n_insertions)
        kh_err = abs(kh[i] * f.n_insertions - rb) / rb if rb > 0 else \
            (0.0 if kh[i] == 0 else float("inf"))
        acc = k_dir > 1e-10 * m  # accessible space (mean Boltzmann factor above 1e-10)
        phys.append(dict(framework=f.name, pockets=int(pockets[i]), accessible=bool(acc),
                         mean_b_direct=k_dir / m, mean_b_trilinear=k_un / m,
                         trilinear_vs_direct_rel=abs(k_un - k_dir) / k_dir if acc else None,
                         blocked_vs_direct_outside_pockets_rel=(abs(k_bl - k_dir_open) / k_dir
                                                                if acc else None),
                         kh_rel_err_vs_oracle=kh_err))
        unblocked[i].close()
    devs = [p["trilinear_vs_direct_rel"] for p in phys if p["trilinear_vs_direct_rel"] is not None]
    log(f"physics check on {len(phys)} frameworks: trilinear vs direct K_H median "
        f"{np.median(devs):.3g}, max {max(devs):.3g}")
    for g in grids:
        g.close()
    for fw in fwh:
        fw.close()
    ctx.close()
    lab_gbs = 8.0 * voxels / t_lab / 1e9
    tri_gbs = 32.0 * ins / t_tri / 1e9
    log(f"labelling {t_lab * 1e3:.1f} ms ({lab_gbs:.1f} GB/s at 8 B/voxel), "
        f"trilinear {ins / t_tri:.3g} inserts/s, energy calls {len(pos) / t_en:.3g}/s "
        f"(host buffers)")
    return {
        "metric": "config5: pocket labelling voxels/s + grid-interpolated Widom inserts/s",
        "value": ins / t_tri, "unit": "inserts/s", "n_gpus": 1, "steps": 1, "warmup": 0,
        "ms_per_step": (t_lab + t_tri) * 1e3, "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "fp32 grid, fp64 interpolation and Boltzmann sums",
        "data": "synthetic (seeded SplitMix64 frameworks)",
        "config": {"workload": f"config5: {len(fws)} frameworks, FP32 grids at 0.2 A, "
                               "threshold 15 T at 298 K, 1e7 trilinear insertions each",
                   "voxels": voxels, "insertions": ins, "parallelism": "single GPU"},
        "labelling_voxels_per_s": voxels / t_lab, "labelling_ms": t_lab * 1e3,
        "pockets_total": int(sum(pockets)), "grid_build_s": t_grid,
        "roofline": {"bound": "hbm", "achieved": lab_gbs, "peak": 8000.0, "unit": "GB/s",
                     "frac": lab_gbs / 8000.0, "traffic": None,
                     "kernel": "pocket labelling of all grids (one er_pockets_label_batch "
                               "call, 8 B/voxel)"},
        "trilinear_GBps_at_32B": tri_gbs,
        "physics_check": {
            "what": "K_H sums by trilinear interpolation of the 0.2 A FP32 grid vs the direct "
                    "FP64 sum (reference method on the GPU), same 1e6 insertion points, every "
                    "8th framework; blocked grid vs the direct sum outside blocked pockets",
            "trilinear_vs_direct_rel_median": float(np.median(devs)),
            "trilinear_vs_direct_rel_max": float(max(devs)),
            "kh_rel_err_vs_oracle_max": max(p["kh_rel_err_vs_oracle"] for p in phys),
            "frameworks": phys},
        "grid_energy_calls_per_s_host_buffers": len(pos) / t_en,
    }


def bench_copy():
    """Plain 1 GiB device-to-device copy (3 times): the known-size reference
    that scales the FETCH_SIZE / WRITE_SIZE counters of the other kernels."""
    import torch
    n = 256 << 20
    x = torch.ones(n, dtype=torch.float32, device="cuda")
    y = torch.empty_like(x)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(3):
        y.copy_(x)
    torch.cuda.synchronize()
    dt = (time.perf_counter() - t0) / 3
    return {"metric": "device copy bandwidth (counter calibration)", "value": 2 * 4 * n / dt / 1e9,
            "unit": "GB/s", "n_gpus": 1, "steps": 3, "warmup": 0, "ms_per_step": dt * 1e3,
            "higher_is_better": True, "config": {"workload": "copy: 1 GiB fp32, 3 times"}}


TRAFFIC_FILE = os.path.join(ROOT, "profiles", "k_tiles_traffic_config3_256fw.txt")


def measured_counters(tuning, n_frameworks):
    """(HBM bytes, VALU wave instructions) of the grid-only launches from the
    committed rocprofv3 runs (bytes scaled by the copy calibration), if they
    were taken on this workload and tuning; else (None, None)."""
    try:
        kv = {}
        with open(TRAFFIC_FILE) as fh:
            for line in fh:
                if ":" in line and not line.startswith("#"):
                    k, v = line.split(":", 1)
                    kv[k.strip()] = v.strip()
        knobs = {k: v for k, v in tuning.items() if k != "source"}
        filed = {k: v for k, v in json.loads(kv["tuning"]).items() if k != "source"}
        if int(kv["frameworks"]) != n_frameworks or filed != knobs:
            return None, None
        return ((float(kv["fetch_kib"]) * float(kv["fetch_scale"]) +
                 float(kv["write_kib"]) * float(kv["write_scale"])) * 1024.0,
                float(kv["valu_insts"]))
    except (OSError, KeyError, ValueError):
        return None, None


def batch_kernel_ms(api, ctx, tasks, runs):
    """Mean HIP-event time of the tiled-kernel launches of a batch of tasks
    (one untimed run first)."""
    b = api.Batch(ctx, tasks, use_graph=False)
    b.set_timing(True)
    b.run()
    b.wait()
    ms = []
    for _ in range(runs):
        b.run()
        b.wait()
        ms.append(b.kernel_ms()[0])
    b.close()
    return float(np.mean(ms))


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--workload", default="config3")
    ap.add_argument("--frameworks", type=int, default=256)
    ap.add_argument("--no-plain", action="store_true")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-fp64", action="store_true", help="skip the FP64-grid leg")
    ap.add_argument("--no-serve", action="store_true", help="skip the serving leg")
    ap.add_argument("--grid-precision", default="fp32", choices=["fp32", "fp64"],
                    help="grids of the batch: fp32 (mixed precision) or fp64 (every pair "
                         "FP64, the drop-in writegrid's default)")
    ap.add_argument("--direct-every", type=int, default=16,
                    help="time the reference's direct method (FP64, every triple, one "
                         "framework per launch) on every k-th framework (0: skip)")
    ap.add_argument("--cpu-seconds", type=float, default=15.0)
    ap.add_argument("--graph", type=int, default=1, help="also time hipGraph replays")
    ap.add_argument("--ppl", type=int, default=0, help="points per lane (0: library default)")
    ap.add_argument("--tile", default="", help="grid tile in points, e.g. 8,8,8")
    ap.add_argument("--lds-records", type=int, default=0)
    ap.add_argument("--region-len", type=float, default=-1.0, help="region edge in A (-1: default)")
    ap.add_argument("--s2-switch", type=float, default=0.0)
    ap.add_argument("--widom-per-bin", type=int, default=0)
    ap.add_argument("--rates", default="50,100,200,500", help="config4 arrival rates (req/s)")
    ap.add_argument("--serve-seconds", type=float, default=4.0)
    ap.add_argument("--serve-rate", type=float, default=500.0,
                    help="arrival rate of the serving leg of the default run (req/s)")
    ap.add_argument("--serve-leg-seconds", type=float, default=2.0)
    ap.add_argument("--pick", default="random", choices=["random", "cycle"],
                    help="config4: frameworks drawn from the pool at random or in turn")
    ap.add_argument("--cache-bytes", type=int, default=-1,
                    help="config4: idle frameworks kept resident (-1 up to the budget, 0 none)")
    ap.add_argument("--streams", type=int, default=3)
    ap.add_argument("--items-per-launch", type=int, default=32768)
    ap.add_argument("--tuning-file", default=DEFAULT_TUNING_FILE,
                    help="knobs from an autotuner file ('' = library defaults)")
    ap.add_argument("--autotune", type=int, default=0,
                    help="autotune on every k-th framework of the workload first (0: off)")
    ap.add_argument("--save-tuning", default="", help="write the autotuner result here")
    args = ap.parse_args()
    if args.gpus != 1:
        print(json.dumps({"error": "this build runs on one GPU only; --gpus must be 1"}))
        sys.exit(2)

    if args.workload == "copy":
        print(json.dumps(bench_copy()))
        return
    from emptyroom_amd import api, synth
    if args.workload == "config4":
        if args.frameworks == 256:
            args.frameworks = 64
        print(json.dumps(bench_serving(args, api, synth)))
        return
    if args.workload == "config5":
        if args.frameworks == 256:
            args.frameworks = 64
        print(json.dumps(bench_pockets(args, api, synth)))
        return
    fws = make_workload(args.workload, args.frameworks)
    log(f"workload {args.workload}: {len(fws)} frameworks")
    ctx = api.Context(0)
    tuning_source = "library defaults"
    if args.tuning_file and os.path.exists(args.tuning_file):
        from emptyroom_amd import autotune
        ctx.tuning = autotune.load(args.tuning_file)
        tuning_source = os.path.relpath(args.tuning_file, ROOT)
    tu = ctx.tuning
    if args.ppl:
        tu.points_per_lane = args.ppl
    if args.tile:
        for d, v in enumerate(args.tile.split(",")):
            tu.tile[d] = int(v)
    if args.lds_records:
        tu.lds_records = args.lds_records
    if args.region_len >= 0:
        tu.region_len = args.region_len
    if args.s2_switch:
        tu.s2_switch = args.s2_switch
    if args.widom_per_bin:
        tu.widom_per_bin = args.widom_per_bin
    ctx.tuning = tu
    uploaded = []
    for f in fws:
        a = f.particles()
        uploaded.append(api.Framework(ctx, a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2))
    gprec = api.ER_FP64 if args.grid_precision == "fp64" else api.ER_FP32
    tasks = [dict(fw=u, grid_n=f.grid_n(), precision=gprec, n_insertions=f.n_insertions,
                  temperature=f.temperature, seed=f.seed) for f, u in zip(fws, uploaded)]
    if args.autotune:
        from emptyroom_amd import autotune
        k = args.autotune
        log(f"autotuning on every {k}-th framework ({len(fws[::k])} of {len(fws)})")
        tuned = autotune.autotune(ctx, tasks[::k], [f.t for f in fws[::k]], log=log)
        log(f"autotuned: step {tuned['start_step_seconds'] * 1e3:.1f} -> "
            f"{tuned['step_seconds'] * 1e3:.1f} ms on the sample, "
            f"{tuned['measurements']} configurations in {tuned['search_seconds']:.0f} s")
        if args.save_tuning:
            autotune.save(args.save_tuning, tuned,
                          meta={"workload": args.workload, "sample_every": k,
                                "frameworks": len(fws), "device": "MI355X (gfx950)"})
        tuning_source = f"autotuned in this run (every {k}-th framework)"
    tu = ctx.tuning
    tuning = dict(ppl=tu.points_per_lane, tile=list(tu.tile), lds_records=tu.lds_records,
                  region_len=tu.region_len, s2_switch=tu.s2_switch,
                  widom_per_bin=tu.widom_per_bin,
                  class_tile=[list(r) for r in tu.class_tile], source=tuning_source)
    log(f"tuning {tuning}")
    grid_pe = sum(pair_evals(f)[0] for f in fws)
    widom_pe = sum(pair_evals(f)[1] for f in fws)
    n_ins = sum(f.n_insertions for f in fws)
    points = sum(int(np.prod(f.grid_n())) for f in fws)
    log(f"{points:.3g} grid points, {n_ins:.3g} insertions, "
        f"{grid_pe + widom_pe:.3g} pair-evals per step")

    batch = api.Batch(ctx, tasks, use_graph=False)
    batch.set_timing(True)
    for _ in range(args.warmup):
        batch.run()
        batch.wait()
    log("warmup done")
    kernel_ms = []
    t0 = time.perf_counter()
    for _ in range(args.steps):
        batch.run()
        batch.wait()
        ms, nl = batch.kernel_ms()  # every tile-kernel launch of the step
        kernel_ms.append(ms)
    t_batched = (time.perf_counter() - t0) / args.steps
    log(f"batched step {t_batched * 1e3:.1f} ms, tiled kernel {np.mean(kernel_ms):.1f} ms")

    graph_ms = None
    if args.graph:
        gb = api.Batch(ctx, tasks, use_graph=True)
        gb.run()
        gb.wait()
        t0 = time.perf_counter()
        for _ in range(args.steps):
            gb.run()
            gb.wait()
        graph_ms = (time.perf_counter() - t0) / args.steps * 1e3
        for i in range(len(fws)):
            assert gb.widom(i) == batch.widom(i), "graph replay differs from eager run"
        gb.close()
        log(f"graph step {graph_ms:.1f} ms")

    # The roofline launches: the same tiled kernels on the step's grids alone.
    # Every in-cutoff pair of a grid counts in it (no early stop): 16 FLOP each is
    # the direct method's work, of which fine grids do less (their far pairs come
    # from nodes, an eighth of the points).  The Widom share of the
    # step is timed on its own too (its insertions may stop once their energy
    # is certain to reach 800 T, so it gets an insertion rate, not FLOP/s).
    grid_tasks = [dict(t, n_insertions=0) for t in tasks]
    widom_tasks = [dict(t, grid_n=(0, 0, 0)) for t in tasks]
    grid_ms = batch_kernel_ms(api, ctx, grid_tasks, max(1, args.steps))
    widom_ms = batch_kernel_ms(api, ctx, widom_tasks, max(1, args.steps))
    log(f"grids alone {grid_ms:.1f} ms, Widom alone {widom_ms:.1f} ms (kernel)")

    fp64 = None
    if not args.no_fp64 and gprec == api.ER_FP32:
        # the drop-in writegrid's default: FP64 grids (every pair FP64) with the
        # same Widom runs, one batch per step; and the FP64 grids alone
        t64 = [dict(t, precision=api.ER_FP64) for t in tasks]
        b64 = api.Batch(ctx, t64, use_graph=False)
        b64.run()
        b64.wait()
        t0 = time.perf_counter()
        for _ in range(args.steps):
            b64.run()
            b64.wait()
        t_fp64 = (time.perf_counter() - t0) / args.steps
        # FP64 grids against the direct method are in the direct-method block
        b64.close()
        g64_ms = batch_kernel_ms(api, ctx, [dict(t, n_insertions=0) for t in t64],
                                 max(1, args.steps))
        fp64 = {"ms_per_step": t_fp64 * 1e3, "frameworks_per_s": len(fws) / t_fp64,
                "grid_kernel_ms": g64_ms}
        log(f"FP64-grid step {t_fp64 * 1e3:.1f} ms, FP64 grids alone {g64_ms:.1f} ms (kernel)")

    plain_s = None
    if not args.no_plain:
        # the same work as a batch step: grids stay resident in HBM (no
        # device-to-host copy), Widom sums come back; one framework per
        # launch, synchronous
        t0 = time.perf_counter()
        for f, u in zip(fws, uploaded):
            api.Grid.compute(ctx, u, f.grid_n(), gprec).close()
            api.widom(ctx, u, f.n_insertions, f.temperature, f.seed)
        plain_s = time.perf_counter() - t0
        log(f"plain step {plain_s * 1e3:.1f} ms")

    direct = None
    if args.direct_every > 0:
        # the reference's method on the same GPU: FP64 arithmetic over every
        # (point, image, atom) triple, one framework per launch, grids kept
        # resident, Widom sums back; timed on a sample of the mix and scaled
        # to the whole mix by pair-evals (its time is linear in them)
        k = args.direct_every
        sample = list(range(0, len(fws), k))
        sample_pe = sum(sum(pair_evals(fws[i])) for i in sample)
        d_grids, d_sums = [], []
        t0 = time.perf_counter()
        for i in sample:
            f = fws[i]
            a = f.particles()
            args_d = (a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2)
            d_grids.append(api.direct_grid(ctx, *args_d, f.grid_n(), download=False))
            d_sums.append(api.direct_widom(ctx, *args_d, f.n_insertions, f.temperature, f.seed))
        t_direct = time.perf_counter() - t0
        est_s = t_direct * (grid_pe + widom_pe) / sample_pe
        # the batch's own results against the direct method's FP64 ones, at
        # every grid point and over every insertion of the sampled frameworks
        gerr, grel, g64err, kerr, eerr = 0.0, 0.0, 0.0, 0.0, 0.0
        n_pts = n_hi = n_kh = n_kh0 = 0
        for i, gd, (db, deb, _) in zip(sample, d_grids, d_sums):
            ref = gd.download()
            gd.close()
            g = batch.grid(i).astype(np.float64)
            m = ref < 1e4
            if m.any():
                gerr = max(gerr, float(np.max(np.abs(g[m] - ref[m]))))
                n_pts += int(m.sum())
            hi = ~m & (ref < 3.0e38)
            if hi.any():
                grel = max(grel, float(np.max(np.abs(g[hi] - ref[hi]) / ref[hi])))
                n_hi += int(hi.sum())
            if fp64 is not None:
                g64 = api.compute_grid(ctx, uploaded[i], fws[i].grid_n(), api.ER_FP64)
                g64err = max(g64err, float(np.max(np.abs(g64 - ref) /
                                                  np.maximum(1.0, np.abs(ref)))))
            bb, beb, _ = batch.widom(i)
            if db > 0:
                kerr = max(kerr, abs(bb - db) / db)
                eerr = max(eerr, abs(beb / bb - deb / db))
                n_kh += 1
            elif bb == 0.0:
                n_kh0 += 1
            else:
                kerr = float("inf")
                n_kh += 1
        direct = {"sample": f"every {k}-th framework ({len(sample)} of {len(fws)}), grid + "
                            "Widom each, scaled to the mix by pair-evals",
                  "seconds": t_direct, "pair_evals_per_s": sample_pe / t_direct,
                  "est_seconds_per_step": est_s,
                  "est_frameworks_per_s": len(fws) / est_s,
                  "batched_over_direct": est_s / t_batched,
                  "batched_errors": {
                      "grid_max_abs_err_K": gerr if n_pts else None,
                      "grid_points_compared": n_pts,
                      "grid_max_rel_err_above_1e4K": grel if n_hi else None,
                      "grid_points_above_1e4K_compared": n_hi,
                      "fp64_grid_max_rel_err": g64err if fp64 is not None else None,
                      "kh_rel_err_max": kerr if n_kh else None,
                      "e_avg_max_abs_err_K": eerr if n_kh else None,
                      "widom_runs_compared": n_kh,
                      "widom_runs_both_exactly_zero": n_kh0,
                      "against": "FP64 direct method (bit-identical to the oracle), every grid "
                                 "point and every insertion of the sample"}}
        log(f"direct method {sample_pe / t_direct:.3g} pair-evals/s on the sample "
            f"({t_direct:.1f} s); whole mix ~{est_s:.1f} s; batched vs direct: grid "
            f"{gerr:.3g} K over {n_pts} points (rel {grel:.3g} over {n_hi} above 1e4 K), "
            f"K_H {kerr:.3g} over {n_kh} runs ({n_kh0} both 0)")

    # in-cutoff pairs of one step (exact GPU counting pass, outside the timed
    # region), grids and Widom runs separately
    incut_grid = incut_widom = 0
    for f, u in zip(fws, uploaded):
        incut_grid += api.count_incut_grid(ctx, u, f.grid_n())
        incut_widom += api.count_incut_widom(ctx, u, f.n_insertions, f.seed)
    incut = incut_grid + incut_widom
    achieved = FLOP_PER_PAIR * incut_grid / (grid_ms / 1e3) / 1e12
    log(f"in-cutoff pairs {incut:.4g} (grids {incut_grid:.4g}, Widom {incut_widom:.4g}); "
        f"grid kernel {achieved:.2f} TFLOP/s")
    if fp64 is not None:
        a64 = FLOP_PER_PAIR * incut_grid / (fp64["grid_kernel_ms"] / 1e3) / 1e12
        fp64["roofline"] = {"bound": "valu", "achieved": a64, "peak": PEAK_FP64_TFLOPS,
                            "unit": "TFLOP/s", "frac": a64 / PEAK_FP64_TFLOPS,
                            "kernel": f"k_tiles<{tuning['ppl']},FP64> on the FP32 step's grids "
                                      "in FP64, alone",
                            "kernel_ms": fp64["grid_kernel_ms"]}

    cpu = cpu1 = cfg1 = None
    grid_err = kh_err = e_err = None
    host = host_cpu()
    if not args.no_cpu:
        threads = host["threads"]
        cpu, grid_err, kh_err, e_err = cpu_baseline(fws, uploaded, ctx, batch, args.cpu_seconds,
                                                    threads)
        cpu.update(nproc=host["nproc"], usable_cpus=host["usable"],
                   omp_num_threads=host["omp_num_threads"], cpu_model=host["model"])
        log(f"cpu baseline {cpu['value']:.3g} pair-evals/s on {threads} threads "
            f"({host['model']}, nproc {host['nproc']}, usable {host['usable']})")
        # the same kind of sample on one core (a third of the time budget)
        cpu1, _, _, _ = cpu_baseline(fws, uploaded, ctx, batch, args.cpu_seconds / 3.0, 1)
        log(f"cpu baseline {cpu1['value']:.3g} pair-evals/s on 1 thread")
        cfg1 = config1_full(api, synth, ctx, threads)
        log(f"config1 in full: {json.dumps(cfg1)}")

    serve = None
    if not args.no_serve and args.workload == "config3":
        pool = [synth.config3_framework(i, config=4) for i in range(64)]
        parts = [(f, f.particles()) for f in pool]
        sctx = api.Context(0, hbm_cap=200 << 30)
        serve = serve_rate(api, synth, sctx, parts, args.serve_rate, args.serve_leg_seconds,
                           args.streams, args.items_per_launch)
        sctx.close()
        serve["workload"] = ("config4: Poisson arrivals, frameworks drawn from a pool of 64 of "
                             "the batching distribution, T ~ U[250,350] K, HBM cap 200 GB")
        log(f"serving {json.dumps(serve)}")

    value = (grid_pe + widom_pe) / t_batched
    ratio = (plain_s / t_batched) if plain_s else None
    traffic = valu_insts = None
    if args.workload == "config3" and gprec == api.ER_FP32:
        traffic, valu_insts = measured_counters(tuning, len(fws))
    out = {
        "metric": "LJ pair-evals/s + Widom inserts/s, batched vs plain, at K_H rel err <=1e-4",
        "value": value,
        "unit": "pair-evals/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": t_batched * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": ratio / TARGET_BATCHED_OVER_PLAIN if ratio else None,
        "vs_baseline_basis": f"batched/plain frameworks/s over the target "
                             f"{TARGET_BATCHED_OVER_PLAIN:g}x (no published number exists)",
        "dtype": ("fp32 pair LJ beyond 1.5 sigma, fp64 r^2 / close pairs / accumulation"
                  if gprec == api.ER_FP32 else
                  "fp64 grids (every pair), Widom fp32 pair LJ beyond 1.5 sigma"),
        "data": "synthetic (seeded SplitMix64 frameworks)",
        "config": {"workload": WORKLOAD_TEXT.get(args.workload, args.workload).format(
                       n=len(fws)).replace("FP32", args.grid_precision.upper()),
                   "frameworks": len(fws), "grid_points": points, "insertions": n_ins,
                   "grid_precision": args.grid_precision, "parallelism": "single GPU"},
        "inserts_per_s": n_ins / t_batched,
        "grid_pair_evals_per_s": grid_pe / t_batched,
        "frameworks_per_s_batched": len(fws) / t_batched,
        "frameworks_per_s_plain": (len(fws) / plain_s) if plain_s else None,
        "batched_over_plain": ratio,
        "batched_over_plain_target": TARGET_BATCHED_OVER_PLAIN,
        "batched_over_plain_target_met": (ratio >= TARGET_BATCHED_OVER_PLAIN) if ratio else None,
        "direct_method": direct,
        "graph_ms_per_step": graph_ms,
        "kernel_ms_per_step": float(np.mean(kernel_ms)),
        "incut_pairs_per_step": incut,
        "incut_pairs_grid": incut_grid,
        "incut_pairs_widom": incut_widom,
        "kh_rel_err_max": kh_err,
        "grid_max_abs_err_K": grid_err,
        "roofline": {"bound": "valu", "engine": "VALU (no MFMA: pairwise LJ)",
                     "achieved": achieved, "peak": PEAK_FP32_TFLOPS, "unit": "TFLOP/s",
                     "frac": achieved / PEAK_FP32_TFLOPS,
                     "attainable_peak": PEAK_FP32_UNPACKED_TFLOPS,
                     "frac_attainable": achieved / PEAK_FP32_UNPACKED_TFLOPS,
                     "valu_issue": valu_insts / (VALU_ISSUE_PER_S * grid_ms / 1e3)
                     if valu_insts else None,
                     "traffic": traffic,
                     "kernel": f"k_tiles<{tuning['ppl']},MIXED> and its variants with nodes and "
                               f"for small grids, on the step's {len(fws)} grids alone (a launch "
                               "each)"
                               if gprec == api.ER_FP32 else
                               f"k_tiles<{tuning['ppl']},FP64> and its variant for small grids, "
                               "on the step's grids alone",
                     "kernel_ms": grid_ms,
                     "flop_per_pair": FLOP_PER_PAIR,
                     "incut_pairs": incut_grid,
                     "note": "achieved and frac: 16 FLOP x every in-cutoff pair of the step's grids "
                             "/ the grid-only launches, the direct method's work per second, not "
                             "issued FLOPs (the far pairs of fine grids are evaluated at an "
                             "eighth of the points and interpolated); valu_issue: VALU wave "
                             "instructions of the committed counter run / issue slots (256 CUs x "
                             "2.4 GHz) of this run; peak 157.3 is the packed-FP32 rate, which "
                             "this build does not use (attainable_peak 78.6)"},
        "widom_alone": {"kernel_ms": widom_ms, "insertions_per_s": n_ins / (widom_ms / 1e3),
                        "incut_pairs": incut_widom,
                        "note": "insertions stop once their energy is certain to reach 800 T "
                                "(exp(-E/T) exactly 0), so no FLOP rate is claimed"},
        "fp64_grid_ms_per_step": fp64["ms_per_step"] if fp64 else None,
        "fp64_grids": fp64,
        "serving": serve,
        "tuning": tuning,
        "cpu_baseline": cpu,
        "cpu_baseline_1core": cpu1,
        "config1_full": cfg1,
    }
    print(json.dumps(out))
    batch.close()
    for u in uploaded:
        u.close()
    ctx.close()


if __name__ == "__main__":
    main()
