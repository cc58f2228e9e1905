"""Benchmark of the Openpipeflow time step on one MI355X.

Headline workload: one state at (N, K, M) = (64, 64, 48), Mp = 1,
alpha = 0.5, Re = 5300, dt = 0.005, implicitness 0.51, constant flux,
seeded perturbation of energy 1e-2, with the corrector iterated to
convergence as main.f90:35-41 does.  The timed region is `--steps`
consecutive steps of the device-resident loop after `--warmup` steps; the
state is in HBM before timing starts.

Printed: one JSON line with the metric (state-steps/s), the parity check of
the energy / friction-velocity series against the reference's own run
(tests/golden/golden_c1.npz, |dE|/E <= 1e-10), the HBM roofline of the
dominant kernel (HIP events on the library's stream), the reference CPU
code timed on this host's cores on a bounded sample of the same workload,
and two more legs: batched mode (512 mixed states at (32,24,12)) and the
request server (Poisson arrivals of three sizes, p50/p99 latency).
"""
from __future__ import annotations

import argparse
import json
import os
import subprocess
import sys
import tempfile
import time

import numpy as np

REPO = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(REPO, "softx-d-17-00015_amd"))

HBM_PEAK_GBS = 8000.0          # MI355X HBM3E peak

WORKLOADS = {
    # name: N, K, M, Re, alpha, dt, E0, seed, golden fixture
    "c1": (64, 64, 48, 5300.0, 0.5, 0.005, 1e-2, 1, "golden_c1.npz"),
    "c0": (32, 24, 12, 2400.0, 1.25, 0.01, 1e-3, 1, "golden_c0.npz"),
    # the large size: the reference's own 20-step run (records of the
    # warm-up steps 0 and 10 are compared)
    "c2": (96, 256, 128, 5300.0, 0.4, 0.0025, 1e-2, 1, "golden_c2.npz"),
}


def factor_bytes(N, K, M):
    """What a step launch reads of the solves: the 4 x 4 block inverses of four
    matrices and the six influence vectors per (|k|, m) pair, and a 4 x 4 inverse
    per harmonic."""
    H = (2 * K - 1) * M - (K - 1)
    return K * M * (4 * 128 * ((N + 3) // 4) + 48 * N) + 128 * H


def alg_bytes(N, K, M):
    """Algorithmic (compulsory) bytes per launch of each kernel: every array
    the kernel must read or write once.  C = one complex coll field."""
    H = (2 * K - 1) * M - (K - 1)
    Z = 3 * K
    C = 16 * N * H
    Y = 16 * N * Z * M                       # one field of the z-transformed intermediates
    F = factor_bytes(N, K, M)
    return dict(C=C, F=F,
                zfwd=6 * C + 6 * Y, theta=9 * Y, zbwd=3 * Y + 3 * C,
                # the whole-plane evaluation of small grids: u, curl u in, N out
                plane=9 * C,
                # predictor: read N and u_, write u and curl u; each corrector
                # also reads N_ and the previous iterate
                step_pred=12 * C + F, step_corr=18 * C + F, curl=6 * C)


def alg_bytes_per_step(N, K, M, ncorr):
    """B_alg = (21 + 27 n_corr) C + (1 + n_corr) F, the two-phase compulsory
    traffic model (factors and influence vectors once per +-k pair)."""
    H = (2 * K - 1) * M - (K - 1)
    C = 16 * N * H
    F = factor_bytes(N, K, M)
    return (21 + 27 * ncorr) * C + (1 + ncorr) * F


def make_ic(ctx, wl):
    from opf import ic
    N, K, M, Re, alpha, dt, E0, seed, _ = wl
    me = ctx.mesh()
    return ic.seeded_perturbation(me["r"], me["intrdr"], K, M, alpha, seed, E0)


def host_cores():
    """Host cores this process may use (the GPU box gives one GPU a share of
    16), for the CPU baselines."""
    try:
        n = len(os.sched_getaffinity(0))
    except AttributeError:
        n = os.cpu_count() or 1
    return max(1, min(16, n))


def _ref_env():
    return dict(os.environ, MKL_NUM_THREADS="1", MKL_THREADING_LAYER="SEQUENTIAL", OMP_NUM_THREADS="1")


def _unlimited_stack():
    import resource
    # the reference keeps large automatic coll temporaries on the stack
    resource.setrlimit(resource.RLIMIT_STACK, (resource.RLIM_INFINITY, resource.RLIM_INFINITY))


def _ref_start(exe, icf, prefix, Re, alpha, dt, nsteps, ranks=1):
    """Start one reference run (oracle/_ref: ref_driver.f90, or
    ref_mpi_driver.f90 under mpiexec with `ranks` ranks); returns the process."""
    cmd = [exe, icf, prefix, repr(Re), repr(alpha), repr(dt), str(nsteps)]
    if ranks > 1:
        cmd = ["/opt/conda/bin/mpiexec", "-n", str(ranks)] + cmd
    return subprocess.Popen(cmd, cwd=os.path.dirname(prefix), env=_ref_env(), preexec_fn=_unlimited_stack,
                            stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)


def _ref_seconds(proc, prefix, timeout=300):
    """Wait for a reference run; the wall seconds of its time loop."""
    if proc.wait(timeout=timeout) != 0:
        raise RuntimeError(f"reference run failed with status {proc.returncode}")
    with open(prefix + "_timing.txt") as f:
        return float(f.read().split()[0])


def _mpi_build(name, cores):
    """The MPI build of the reference for this workload with the most ranks
    that fit the host's cores: (executable, ranks) or None."""
    best = None
    for r in (4, 8, 16):
        exe = os.path.join(REPO, "oracle", "_ref", f"opf_ref_mpi_{name}_{r}")
        if r <= cores and os.path.exists(exe) and os.path.exists("/opt/conda/bin/mpiexec"):
            best = (exe, r)
    return best


def cpu_baseline(name, wl, ic_fields, target_s):
    """The reference's own CPU path on this host's cores, on a bounded
    sample of the same workload: the reference Fortran (oracle/_ref,
    compiled from the reference sources with MKL's LAPACK/FFTW3) as MPI ranks
    (its radial/harmonic decomposition, parallel.h:5-6) when an MPI build and
    mpiexec are present, else one process on one core; median of 3 runs.
    Falls back to the numpy oracle on one core."""
    N, K, M, Re, alpha, dt, E0, seed, _ = wl
    sys.path.insert(0, os.path.join(REPO, "oracle"))
    import opf_oracle as O
    cores = host_cores()
    mpi = _mpi_build(name, cores)
    serial = os.path.join(REPO, "oracle", "_ref", f"opf_ref_{name}")
    runs = [mpi] if mpi else []
    if os.path.exists(serial):
        runs.append((serial, 1))
    for exe, ranks in runs:
        try:
            with tempfile.TemporaryDirectory() as td:
                icf = os.path.join(td, "ic.bin")
                O.write_coll3(icf, *ic_fields)
                pre = os.path.join(td, "b")
                # a 2-step calibration run sizes the sample (about target_s / 3 per run)
                cal = _ref_seconds(_ref_start(exe, icf, pre, Re, alpha, dt, 2, ranks), pre) / 2.0
                nsteps = max(3, int(target_s / 3.0 / max(cal, 1e-6)))
                secs = [_ref_seconds(_ref_start(exe, icf, pre, Re, alpha, dt, nsteps, ranks), pre)
                        for _ in range(3)]
            med = float(np.median(secs))
            how = f"{ranks} MPI ranks (mpiexec, _Nr = {ranks})" if ranks > 1 else "1 process"
            return dict(value=nsteps / med, unit="state-steps/s", cores=ranks, kind="reference",
                        sample=f"{nsteps} steps of the same workload, reference Fortran (amdflang -O2 + "
                               f"MKL sequential), {how}, median of 3 runs "
                               f"({', '.join(f'{x:.2f}' for x in secs)} s); host cores available: {cores}",
                        runs_s=secs)
        except Exception as e:                       # noqa: BLE001
            print(f"cpu_baseline: reference run with {ranks} rank(s) failed ({e})", file=sys.stderr)
    oc = O.Ctx(N, K, M, Re=Re, alpha=alpha, dt=dt)
    oc.set_state(*ic_fields)
    n = 3
    t0 = time.perf_counter()
    oc.run(n)
    secs = time.perf_counter() - t0
    return dict(value=n / secs, unit="state-steps/s", cores=1, kind="port",
                sample=f"{n} steps of the same workload, numpy oracle, 1 process, {secs:.1f} s")


def cpu_concurrent(jobs, target_s):
    """One serial reference process per core, all at once: jobs = list of
    (executable, initial fields, Re, alpha, dt).  Each runs about target_s
    seconds of steps (sized by a 2-step calibration run per executable).
    Returns (summed state-steps/s, per-job (steps, seconds))."""
    sys.path.insert(0, os.path.join(REPO, "oracle"))
    import opf_oracle as O
    with tempfile.TemporaryDirectory() as td:
        per_step = {}
        for exe, f, Re, alpha, dt in jobs:
            if exe not in per_step:
                icf = os.path.join(td, "cal.bin")
                O.write_coll3(icf, *f)
                pre = os.path.join(td, "cal")
                per_step[exe] = _ref_seconds(_ref_start(exe, icf, pre, Re, alpha, dt, 2), pre) / 2.0
        procs = []
        for i, (exe, f, Re, alpha, dt) in enumerate(jobs):
            icf = os.path.join(td, f"ic{i}.bin")
            O.write_coll3(icf, *f)
            n = max(3, int(target_s / max(per_step[exe], 1e-6)))
            pre = os.path.join(td, f"j{i}")
            procs.append((n, pre, _ref_start(exe, icf, pre, Re, alpha, dt, n)))
        res = [(n, _ref_seconds(p, pre)) for n, pre, p in procs]
    return sum(n / s for n, s in res), res


# batched mode: many (32,24,12) states with their own Re, alpha and initial
# energy, advanced together (every launch covers all slots)
BATCH = dict(N=32, K=24, M=12, dt=0.01, seed=2024)


def batched_step_roofline(N, K, M, nstates, s_per_step, ncorr):
    """The batched step against the HBM peak: every state's B_alg per step
    (at the ensemble's mean corrector count) over the time of one step of
    the whole ensemble."""
    b = nstates * alg_bytes_per_step(N, K, M, ncorr)
    gbs = b / s_per_step / 1e9
    return {"B_alg_bytes": b, "ncorr": ncorr, "achieved_GBs": gbs, "frac": gbs / HBM_PEAK_GBS}


def batched_leg(nstates, steps, cpu_s=0.0):
    """Batched throughput, the same states advanced one at a time (plain
    per-state loop), and the parity of slot 0, which holds the reference's
    (32,24,12) case, against the reference's own energy series.  With
    cpu_s > 0, the CPU baseline of the ensemble: the reference on one state
    per host core, all cores at once, summed."""
    import opf
    from opf import ic
    N, K, M, dt = BATCH["N"], BATCH["K"], BATCH["M"], BATCH["dt"]
    rng = np.random.default_rng(BATCH["seed"])
    params = []
    for i in range(nstates):
        Re = float(rng.uniform(1800.0, 3000.0))
        alpha = float(rng.choice([1.0, 1.25, 1.7]))
        E0 = float(10.0 ** rng.uniform(-5.0, -2.0))
        params.append((Re, alpha, E0, i + 1))
    params[0] = (2400.0, 1.25, 1e-3, 1)           # the reference's (32,24,12) case
    ctx = opf.Context(N, K, M, capacity=nstates)
    gpath = os.path.join(REPO, "tests", "golden", "golden_c0.npz")
    golden = None
    if os.path.exists(gpath):
        with np.load(gpath) as g:
            golden = dict(ic=g["ic"], series=g["series"])
    t0 = time.perf_counter()
    me = None
    first = []                                      # the first states, for the CPU baseline
    for s, (Re, alpha, E0, seed) in enumerate(params):
        ctx.setup(s, Re, alpha, dt)
        if me is None:
            me = ctx.mesh()
        if s == 0 and golden is not None:
            f = golden["ic"]
        else:
            f = ic.seeded_perturbation(me["r"], me["intrdr"], K, M, alpha, seed, E0)
        ctx.put_state(s, f[0], f[1], f[2])
        if s < 16:
            first.append((tuple(f[:3]), Re, alpha))
    setup_s = time.perf_counter() - t0
    ctx.run(2, diag_every=10)                       # warm-up (untimed)
    t0 = time.perf_counter()
    ctx.run(steps, diag_every=10)
    secs = time.perf_counter() - t0
    value = nstates * steps / secs
    parity = {"reference": "golden_c0.npz (slot 0)", "checked_records": 0}
    if golden is not None:
        d = ctx.diag(0)
        rows = [r for r in d if int(r[0]) < golden["series"].shape[0]]
        if rows:
            d = np.array(rows)
            ref = golden["series"][d[:, 0].astype(int)]
            dE = np.abs(d[:, 2] - ref[:, 2]) / ref[:, 2]
            parity.update(checked_records=len(rows), max_rel_dE=float(dE.max()),
                          ok=bool(dE.max() <= 1e-10))
    ncorr = [ctx.status(s)["last_ncorr"] for s in range(nstates)]
    ctx.close()
    # plain per-state loop: the same kind of state advanced alone
    one = opf.Context(N, K, M)
    Re, alpha, E0, seed = params[1]
    one.setup(0, Re, alpha, dt)
    f = ic.seeded_perturbation(me["r"], me["intrdr"], K, M, alpha, seed, E0)
    one.put_state(0, *f)
    one.run(5)
    n1 = max(50, steps)
    t0 = time.perf_counter()
    one.run(n1, diag_every=10)
    alone = n1 / (time.perf_counter() - t0)
    one.close()
    cpu = None
    exe = os.path.join(REPO, "oracle", "_ref", "opf_ref_c0")
    if cpu_s > 0 and os.path.exists(exe):
        cores = min(host_cores(), len(first))
        try:
            tot, res = cpu_concurrent([(exe, f, Re, alpha, dt) for f, Re, alpha in first[:cores]], cpu_s)
            cpu = dict(value=tot, unit="state-steps/s", cores=cores, kind="reference",
                       sample=f"reference Fortran (serial build, MKL sequential), {cores} processes at once, "
                              f"one ensemble state each (states 0..{cores - 1}), "
                              f"{res[0][0]} steps each in about {cpu_s:.0f} s; summed state-steps/s")
        except Exception as e:                       # noqa: BLE001
            print(f"batched cpu baseline failed ({e})", file=sys.stderr)
    return {"metric": "batched state-steps/s", "value": value, "unit": "state-steps/s",
            "config": {"workload": f"{nstates} states at (N,K,M)=({N},{K},{M}), Re~U[1800,3000], "
                                   f"alpha in {{1.0,1.25,1.7}}, E0 log-uniform [1e-5,1e-2], dt={dt}, "
                                   f"{steps} steps, corrector to convergence",
                       "states": nstates, "steps": steps},
            "ms_per_step": 1000.0 * secs / steps, "setup_s": setup_s,
            "step_roofline": batched_step_roofline(N, K, M, nstates, secs / steps, float(np.mean(ncorr))),
            "plain_per_state_loop": alone, "speedup_vs_plain_loop": value / alone,
            "mean_last_ncorr": float(np.mean(ncorr)), "parity": parity, "cpu_baseline": cpu,
            "speedup_vs_cpu": value / cpu["value"] if cpu else None}


# serving: Poisson arrivals of integration requests of three sizes (5:3:2),
# one corrector per step (steporbit), T ~ U[5, 50] at dt = 0.01
SERVE = dict(classes=[(32, 24, 12), (48, 48, 24), (64, 64, 48)], ratio=(5, 3, 2), dt=0.01, seed=77,
             block_slots=(32, 8, 4))
SERVE_EXES = ("opf_ref_c0", "opf_ref_s48", "opf_ref_c1")   # reference builds of the three classes


def _serve_requests(nreq, rate, seed, meshes):
    """The configs' request stream: class by the 5:3:2 ratio, Re ~ U[2000,
    5300], alpha in {0.5, 1.25}, T ~ U[5, 50] time units at dt = 0.01,
    seeded initial states, Poisson arrivals at `rate` per second (all at
    once for rate = inf)."""
    from opf import ic
    classes, ratio, dt = SERVE["classes"], np.array(SERVE["ratio"], float), SERVE["dt"]
    rng = np.random.default_rng(seed)
    reqs, t = [], 0.0
    for i in range(nreq):
        cls = int(rng.choice(len(classes), p=ratio / ratio.sum()))
        Re = float(rng.uniform(2000.0, 5300.0))
        alpha = float(rng.choice([0.5, 1.25]))
        nsteps = int(round(float(rng.uniform(5.0, 50.0)) / dt))
        E0 = float(10.0 ** rng.uniform(-5.0, -3.0))
        t += 0.0 if not np.isfinite(rate) else float(rng.exponential(1.0 / rate))
        N, K, M = classes[cls]
        st = ic.seeded_perturbation(meshes[cls]["r"], meshes[cls]["intrdr"], K, M, alpha, 1000 * seed + i, E0)
        reqs.append(dict(cls=cls, Re=Re, alpha=alpha, nsteps=nsteps, state=st, arrival=t))
    return reqs


def _serve_once(reqs, pool_bytes, depth):
    """Submit the stream at its arrival times; latencies and span."""
    import opf
    srv = opf.Server(SERVE["classes"], SERVE["block_slots"], pool_bytes, depth=depth)
    t0 = time.perf_counter()
    ids = []
    peak = 0
    for r in reqs:
        wait = r["arrival"] - (time.perf_counter() - t0)
        if wait > 0:
            time.sleep(wait)
        ids.append(srv.submit(r["cls"], r["Re"], r["alpha"], SERVE["dt"], r["nsteps"], r["state"], corr_fixed=1))
    while not all(srv.poll(i)["done"] for i in ids):
        peak = max(peak, srv.pool()["used"])
        time.sleep(0.005)
    polls = [srv.poll(i) for i in ids]
    return srv, ids, polls, peak


def _plain_step_seconds(reps=60):
    """Seconds per step of each serving class run alone (plain context, one
    corrector per step), the per-request loop the server is compared with."""
    import opf
    from opf import ic
    out = []
    for (N, K, M) in SERVE["classes"]:
        me = opf.host_mesh(N)
        one = opf.Context(N, K, M)
        one.setup(0, 3500.0, 1.25, SERVE["dt"])
        one.put_state(0, *ic.seeded_perturbation(me["r"], me["intrdr"], K, M, 1.25, 7, 1e-4))
        one.run(5, corr_fixed=1)
        t0 = time.perf_counter()
        one.run(reps, corr_fixed=1)
        out.append((time.perf_counter() - t0) / reps)
        one.close()
    return out


def serving_leg(nreq, rates, pool_gb, depth, cpu_s=0.0):
    """The request server on the configs' stream: for each arrival rate, p50/
    p99 latency, served state-steps/s and each request's slowdown against
    the same request run alone; the served throughput at saturation against
    the plain per-request loop over the same mix; parity of a served request
    against the reference and against the same integration run alone.  With
    cpu_s > 0, the CPU baseline of the mix: the reference on the first
    requests, one per host core, all at once (summed state-steps/s), and
    the CPU latency of every request run alone on one core."""
    import opf
    classes, dt = SERVE["classes"], SERVE["dt"]
    meshes = [opf.host_mesh(N) for (N, _, _) in classes]
    pool = int(pool_gb * 1e9)
    t_alone = _plain_step_seconds()
    sweep = []
    best = None
    for k, rate in enumerate(rates):
        reqs = _serve_requests(nreq, rate, SERVE["seed"] + k, meshes)
        srv, ids, polls, peak = _serve_once(reqs, pool, depth)
        lat = np.array([p["t_done"] - p["t_submit"] for p in polls])
        alone = np.array([r["nsteps"] * t_alone[r["cls"]] for r in reqs])
        slow = lat / alone
        span = max(p["t_done"] for p in polls) - min(p["t_submit"] for p in polls)
        steps = sum(r["nsteps"] for r in reqs)
        failed = sum(1 for p in polls if p["status"] != 0)
        row = dict(rate_per_s=rate if np.isfinite(rate) else "all at once", requests=nreq, state_steps=steps,
                   throughput=steps / span, p50_s=float(np.percentile(lat, 50)), p99_s=float(np.percentile(lat, 99)),
                   slowdown_p50=float(np.percentile(slow, 50)), slowdown_p99=float(np.percentile(slow, 99)),
                   peak_pool_gb=peak / 1e9, failed=failed)
        sweep.append(row)
        print(f"serving: rate {row['rate_per_s']}: {row['throughput']:.0f} state-steps/s, p50 {row['p50_s']:.2f} s, "
              f"p99 {row['p99_s']:.2f} s, slowdown p50 {row['slowdown_p50']:.2f}", file=sys.stderr, flush=True)
        if k == len(rates) - 1:
            best = (reqs, srv, ids, polls)
        else:
            srv.close()
    reqs, srv, ids, polls = best
    # parity: a served request against the same integration alone
    parity = {}
    j = next(k for k in range(len(reqs)) if reqs[k]["cls"] == 0 and polls[k]["status"] == 0)
    u = srv.result(ids[j], 0)
    srv.close()
    r = reqs[j]
    N, K, M = classes[0]
    one = opf.Context(N, K, M)
    one.setup(0, r["Re"], r["alpha"], dt)
    one.put_state(0, *r["state"][:3])
    one.run(r["nsteps"], corr_fixed=1)
    v = one.get_state(0)
    parity["alone_vs_in_mix_bitwise"] = bool(all(np.array_equal(u[k], v[k]) for k in range(3)))
    one.close()
    # the reference's (32,24,12) case served (one corrector per step, as the
    # reference's own run needed) against the reference's state after 100 steps
    gpath = os.path.join(REPO, "tests", "golden", "golden_c0.npz")
    if os.path.exists(gpath):
        with np.load(gpath) as g:
            gic, g100 = g["ic"], g["state_100"]
        srv = opf.Server(classes[:1], SERVE["block_slots"][:1], pool, depth=depth)
        rid = srv.submit(0, 2400.0, 1.25, dt, 100, tuple(gic), corr_fixed=1)
        while not srv.poll(rid)["done"]:
            time.sleep(0.005)
        u = srv.result(rid, 0)
        srv.close()
        parity["reference_c0_100_steps_rel_err"] = max(
            float(np.abs(u[k] - g100[k]).max() / np.abs(g100[k]).max()) for k in range(3))
    sat = max(sweep, key=lambda row: row["throughput"])
    mix_steps = sum(r["nsteps"] for r in reqs)
    plain_loop = mix_steps / sum(r["nsteps"] * t_alone[r["cls"]] for r in reqs)
    cpu = None
    exes = [os.path.join(REPO, "oracle", "_ref", e) for e in SERVE_EXES]
    if cpu_s > 0 and all(os.path.exists(e) for e in exes):
        cores = min(host_cores(), len(reqs))
        try:
            jobs = [(exes[rq["cls"]], rq["state"][:3], rq["Re"], rq["alpha"], dt) for rq in reqs[:cores]]
            tot, res = cpu_concurrent(jobs, cpu_s)
            sec_step = {}
            for rq, (n, sec) in zip(reqs[:cores], res):
                sec_step.setdefault(rq["cls"], []).append(sec / n)
            per = {c: float(np.mean(v)) for c, v in sec_step.items()}
            lat_cpu = np.array([rq["nsteps"] * per[rq["cls"]] for rq in reqs if rq["cls"] in per])
            cpu = dict(value=tot, unit="state-steps/s", cores=cores, kind="reference",
                       sample=f"reference Fortran (serial builds of the three sizes, MKL sequential, corrector "
                              f"to convergence), the first {cores} requests of the mix, one per core at once, "
                              f"about {cpu_s:.0f} s each; summed state-steps/s",
                       s_per_step={f"({classes[c][0]},{classes[c][1]},{classes[c][2]})": v
                                   for c, v in sorted(per.items())},
                       p50_s=float(np.percentile(lat_cpu, 50)), p99_s=float(np.percentile(lat_cpu, 99)),
                       latency_note="each request's horizon at its class's seconds per step on one core, "
                                    "no queueing")
        except Exception as e:                       # noqa: BLE001
            print(f"serving cpu baseline failed ({e})", file=sys.stderr)
    last = sweep[-1]
    return {"metric": "request latency p50/p99 (s) and served state-steps/s",
            "p50_s": last["p50_s"], "p99_s": last["p99_s"], "throughput": sat["throughput"],
            "unit": "state-steps/s",
            "config": {"workload": f"{nreq} requests per arrival rate, sizes {[list(c) for c in classes]} in ratio "
                                   f"5:3:2, Re~U[2000,5300], alpha in {{0.5,1.25}}, T~U[5,50] at dt={dt}, one "
                                   f"corrector per step, Poisson arrivals",
                       "rates_per_s": [r if np.isfinite(r) else "all at once" for r in rates],
                       "block_slots": list(SERVE["block_slots"]), "pool_gb": pool_gb, "depth": depth},
            "sweep": sweep,
            "plain_per_request_loop": plain_loop, "plain_s_per_step": t_alone,
            "speedup_vs_plain_loop": sat["throughput"] / plain_loop,
            "failed": sum(row["failed"] for row in sweep), "parity": parity, "cpu_baseline": cpu}


def load_traffic(kernel, workload):
    path = os.path.join(REPO, "profiles", f"traffic_{kernel}_{workload}.json")
    if os.path.exists(path):
        with open(path) as f:
            return json.load(f).get("bytes_per_launch")
    return None


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=1000)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--workload", default="c1", choices=sorted(WORKLOADS))
    ap.add_argument("--cpu-seconds", type=float, default=20.0)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--batch-states", type=int, default=512)
    ap.add_argument("--batch-steps", type=int, default=200)
    ap.add_argument("--no-batched", action="store_true")
    ap.add_argument("--serve-requests", type=int, default=24, help="requests per arrival rate")
    ap.add_argument("--serve-rates", default="2,4,8,inf", help="arrival rates per second (inf: all at once)")
    ap.add_argument("--serve-pool-gb", type=float, default=64.0)
    ap.add_argument("--serve-depth", type=int, default=3)
    ap.add_argument("--no-serving", action="store_true")
    ap.add_argument("--timing-steps", type=int, default=40)
    ap.add_argument("--calibrate-copy", type=int, default=0, metavar="BYTES",
                    help="only run a plain device copy of BYTES bytes five times (calibrates the "
                         "FETCH_SIZE / WRITE_SIZE counters of the traffic figures) and exit")
    args = ap.parse_args()
    if args.calibrate_copy > 0:
        import torch
        a = torch.ones(args.calibrate_copy, dtype=torch.uint8, device="cuda:0")
        b = torch.empty_like(a)
        for _ in range(5):
            b.copy_(a)
        torch.cuda.synchronize()
        print(json.dumps({"calibrate_copy_bytes": args.calibrate_copy, "copies": 5}))
        return
    if args.gpus != 1:
        print(json.dumps({"error": "this benchmark runs on one GPU only; --gpus must be 1 "
                                   "(multi-GPU sharding is a design, not a code path)"}))
        sys.exit(2)
    import opf

    name = args.workload
    wl = WORKLOADS[name]
    N, K, M, Re, alpha, dt, E0, seed, golden = wl
    ctx = opf.Context(N, K, M)
    ctx.setup(0, Re, alpha, dt)
    fields = make_ic(ctx, wl)
    ctx.put_state(0, *fields)

    # warmup, then the timed region (the library synchronises its stream on
    # both sides of opf_run)
    ctx.run(args.warmup, diag_every=10)
    t0 = time.perf_counter()
    ctx.run(args.steps, diag_every=10)
    t1 = time.perf_counter()
    secs = t1 - t0
    value = args.steps / secs
    diag = ctx.diag(0)

    # parity of the energy and friction velocity series with the reference
    parity = {"reference": golden, "checked_records": 0}
    gpath = os.path.join(REPO, "tests", "golden", golden) if golden else None
    ncorr_mean = 1.0
    if gpath and os.path.exists(gpath):
        with np.load(gpath) as g:
            rs = g["series"]
        rows = [r for r in diag if int(r[0]) < rs.shape[0]]
        if rows:
            d = np.array(rows)
            ref = rs[d[:, 0].astype(int)]
            dE = np.abs(d[:, 2] - ref[:, 2]) / ref[:, 2]
            dU = np.abs(d[:, 7] - ref[:, 7]) / ref[:, 7]
            parity.update(checked_records=len(rows), max_rel_dE=float(dE.max()),
                          max_rel_dutau=float(dU.max()),
                          ncorr_equal=bool(np.array_equal(d[:, 8].astype(int), ref[:, 8].astype(int))),
                          ok=bool(dE.max() <= 1e-10 and dU.max() <= 1e-10))
    if len(diag):
        ncorr_mean = float(np.mean(diag[:, 8][diag[:, 8] > 0])) if np.any(diag[:, 8] > 0) else 1.0

    # per-kernel durations with HIP events on the library's stream
    ctx.kernel_timing(True)
    ctx.run(args.timing_steps)
    kt = {}
    for k in ("zfwd", "theta", "zbwd", "plane", "step", "curl", "control"):
        ms, n = ctx.kernel_time(k)
        if n:
            kt[k] = dict(ms_total=ms, launches=n, us_avg=1000.0 * ms / n)
    ctx.kernel_timing(False)
    ab = alg_bytes(N, K, M)
    ab["step"] = (ab["step_pred"] + ncorr_mean * ab["step_corr"]) / (1.0 + ncorr_mean)
    dom = max(kt, key=lambda k: kt[k]["ms_total"])
    achieved = ab[dom] / (kt[dom]["us_avg"] * 1e-6) / 1e9
    ms_step = 1000.0 * secs / args.steps
    B_alg = alg_bytes_per_step(N, K, M, ncorr_mean)
    step_gbs = B_alg / (secs / args.steps) / 1e9

    batched = None
    ctx.close()
    if not args.no_batched:
        batched = batched_leg(args.batch_states, args.batch_steps,
                              0.0 if args.no_cpu_baseline else args.cpu_seconds / 4)

    serving = None
    if not args.no_serving:
        rates = [float(v) for v in args.serve_rates.split(",")]
        serving = serving_leg(args.serve_requests, rates, args.serve_pool_gb, args.serve_depth,
                              0.0 if args.no_cpu_baseline else args.cpu_seconds / 4)

    cpu = None
    if not args.no_cpu_baseline:
        cpu = cpu_baseline(name, wl, fields, args.cpu_seconds)

    out = {
        "metric": "state-steps/s plain vs batched, p50/p99 request latency, at dE<=1e-10",
        "value": value,
        "unit": "state-steps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic (seeded divergence-free perturbation of Hagen-Poiseuille flow)",
        "config": {"workload": f"plain single-state time step at "
                               f"(N,K,M)=({N},{K},{M}), Re={Re}, alpha={alpha}, dt={dt}, E0={E0}",
                   "N": N, "K": K, "M": M, "Re": Re, "alpha": alpha, "dt": dt,
                   "corrector": "iterated to convergence (main.f90:35-41)",
                   "mean_ncorr": ncorr_mean},
        "parity": parity,
        "roofline": {"bound": "hbm", "kernel": dom, "achieved": achieved, "peak": HBM_PEAK_GBS,
                     "unit": "GB/s", "frac": achieved / HBM_PEAK_GBS,
                     "traffic": load_traffic(dom, name),
                     "alg_bytes_per_launch": ab[dom], "us_per_launch": kt[dom]["us_avg"]},
        "step_roofline": {"B_alg_bytes": B_alg, "achieved_GBs": step_gbs,
                          "frac": step_gbs / HBM_PEAK_GBS},
        "kernels_us": {k: round(v["us_avg"], 3) for k, v in kt.items()},
        "batched": batched,
        "serving": serving,
        "cpu_baseline": cpu,
    }
    print(json.dumps(out))


if __name__ == "__main__":
    main()
