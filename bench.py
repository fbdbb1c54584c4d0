#!/usr/bin/env python3
"""Throughput of the null-collision Monte Carlo step on one MI355X.

Workload (default): the coupled relativistic avalanche in dry air (N2:O2:Ar =
0.781:0.210:0.009, 1 atm, 273 K), 10^7 initial electrons with kinetic energy log-uniform in
100 keV - 10 MeV, isotropic, from the origin, uniform E = 1 MV/m along -z, B = 0;
electrons, photons and positrons tracked with a 10 keV cut, populations capped at 2^27,
compaction every 8 steps, FP64 state, dt = 1 ps.  A step is one pt_advance (push,
null-collision selection, sampling, secondary append and the secondaries' own passes).

Metric: particle-steps/s = sum over timed steps of the active particles at step start,
divided by the wall time of the timed loop (inputs resident in HBM, tables uploaded).

Prints one JSON line.  `roofline` names what bounds the main advance kernel, the issue of
vector instructions: those it issues per second (counted by rocprofv3 over a short run of the
same workload) against one wave instruction per SIMD in four cycles.  Its `hbm` entry gives
the bytes the launches cannot do without (a launch takes its particles through several steps
and moves each one's state once, 165 B, and writes 93 B per appended secondary) over the
average launch duration measured with HIP events on the library's stream.  `cpu_baseline`
times the CPU restatement of the reference step (oracle/, OpenMP over the host cores) on a
bounded sample of the same workload.
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "particulator.jl_amd"))

HBM_PEAK_GBPS = 8000.0
# a launch reads each particle (10 FP64, uid, swarm, active flag: 93 B) and writes back
# position, momentum, t, s and r (9 FP64: 72 B), however many steps it advances it; an
# appended secondary writes a whole particle (93 B)
BYTES_PER_PARTICLE = 165.0
BYTES_PER_SECONDARY = 93.0
# one FP64 vector instruction of a wave takes a SIMD four cycles; 4 SIMDs a CU, 2.4 GHz at most
CLOCK_GHZ, CYCLES_PER_INSTRUCTION = 2.4, 4.0


def launch_bytes(psteps, secondaries, steps, launches):
    """bytes that the average of `launches` launches over `steps` steps has to move, with
    `psteps` particle-steps and `secondaries` in all"""
    return BYTES_PER_PARTICLE * psteps / max(steps, 1) + BYTES_PER_SECONDARY * secondaries / max(launches, 1)


def roofline(psteps, secondaries, steps, launches, avg_launch_ms, rate, traffic):
    valu = (traffic or {}).get("valu") or {}
    per_pstep, simds = valu.get("wave_instructions_per_particle_step"), valu.get("simds")
    nbytes = launch_bytes(psteps, secondaries, steps, launches)
    gbps = nbytes / (avg_launch_ms * 1e-3) / 1e9
    peak = simds * CLOCK_GHZ / CYCLES_PER_INSTRUCTION if simds else None
    achieved = per_pstep * rate / 1e9 if per_pstep else None
    return {"bound": "vector instruction issue", "achieved": achieved, "peak": peak,
            "unit": "1e9 wave instructions/s", "frac": achieved / peak if achieved and peak else None,
            "traffic": traffic["bytes"] if traffic else None, "kernel": "k_advance (in-place collisions)",
            "avg_launch_ms": avg_launch_ms, "steps_per_launch": steps / max(launches, 1),
            "hbm": {"algorithmic_bytes_per_launch": nbytes, "achieved": gbps, "peak": HBM_PEAK_GBPS, "unit": "GB/s",
                    "frac": gbps / HBM_PEAK_GBPS},
            "traffic_source": traffic}

WORKLOADS = {
    "avalanche": dict(n=10_000_000, e1=1e5, e2=1e7, loguniform=True, efield=1e6, dt=1e-12,
                      cap=1 << 27, compact_every=8, tracked=(1, 1, 1), horizon_steps=5000,
                      name="coupled relativistic avalanche, 1e7 e- log-uniform 0.1-10 MeV, "
                           "dry air 1 atm 273 K, E=1 MV/m, dt=1 ps, e-/photon/e+ tracked, "
                           "cap 2^27, compaction every 8 steps"),
    "sweep": dict(n=None, e1=1e6, e2=None, loguniform=False, efield=None, dt=1e-12, cap=1 << 28,
                  compact_every=8, tracked=(1, 0, 0), nswarm=256, count_range=(1000, 1_000_000),
                  field_range=(0.4e6, 4e6),
                  name="batched sweep, 256 swarms at E = 0.4-4 MV/m (log-spaced), U{1e3..1e6} e- each "
                       "at 1 MeV isotropic, dry air 1 atm 273 K, dt=1 ps, photons tallied, per-swarm "
                       "rate bounds, captured-graph replays with an autotuned launch"),
    "beam": dict(n=100_000_000, e1=1e7, dt=1e-9, caps=(1 << 23, 1 << 27, 1 << 22), steps=10,
                 dose=(300, 0.0, 3.0), name="photon pencil beam, 1e8 photons at 10 MeV along +z (1e-6 tilt) into "
                 "dry air 1 atm 273 K, no field, all secondaries tracked to 10 keV, dt = 1 ns; depth-dose "
                 "in 300 bins over 0-3 m, photon birth energies in 512 log bins over 10 keV-10 MeV"),
    "swarm": dict(n=10_000, e1=1e6, e2=None, loguniform=False, efield=1e6, dt=1e-12,
                  cap=1 << 20, compact_every=1, tracked=(1, 0, 0),
                  name="runaway swarm, 1e4 e- at 1 MeV, dry air 1 atm 273 K, E=1 MV/m, "
                       "dt=1 ps, photons tallied"),
}


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def cpu_model():
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline(wl, seed, nsample, nsteps):
    """Oracle (C, OpenMP) on a bounded window of the workload: the full initial population,
    a few steps, every host core this process may use (OMP_NUM_THREADS when the
    environment sets it, as a GPU box's CPU share does, else the affinity mask)."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import oracle as O
    import helpers as H
    O.build()
    affinity = len(os.sched_getaffinity(0))
    threads = int(os.environ.get("OMP_NUM_THREADS", "0") or 0) or affinity
    te, tg, tp = H.tables(efield=wl["efield"], dt=wl["dt"])
    caps = (nsample * 2, nsample // 4 + 1024, nsample // 64 + 1024)
    ow = H.make_oracle(te, tg, tp, seed, caps=caps, tracked=tuple(bool(x) for x in wl["tracked"]),
                       efield=(0.0, 0.0, -wl["efield"]), nthreads=threads)
    init = O.init_swarm(nsample, 0, seed, e1=wl["e1"], e2=wl["e2"], loguniform=wl["loguniform"])
    ow.add(0, init)
    del init
    ow.init()
    t, psteps = 0.0, 0
    log("cpu baseline: %d particles, %d steps, %d threads" % (nsample, nsteps, threads))
    t0 = time.perf_counter()
    for _ in range(nsteps):
        psteps += sum(int(O.lib().or_nactives(O.C.byref(ow.w.pop[s]))) for s in range(3)
                      if ow.bufs[s] is not None)
        ow.advance(t + wl["dt"])
        t += wl["dt"]
    el = time.perf_counter() - t0
    return {"value": psteps / el, "unit": "particle-steps/s", "cores": threads, "kind": "port",
            "cpu_model": cpu_model(), "host_cpus": os.cpu_count(), "affinity_cpus": affinity,
            "sample": "the full initial population (%d e- of the workload's distribution), its first %d steps "
                      "(%d particle-steps, %.1f s wall on %d OpenMP threads), reference-semantics C "
                      "restatement of the step (per-particle loop, static chunks, serial droplow!/repack! "
                      "each step)" % (nsample, nsteps, psteps, el, threads)}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=None,
                    help="timed steps (default: 300 avalanche, 40 sweep, 10 beam)")
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--workload", default="avalanche", choices=sorted(WORKLOADS))
    ap.add_argument("--n", type=int, default=None, help="override the initial particle count")
    ap.add_argument("--seed", type=int, default=2024)
    ap.add_argument("--rounds", type=int, default=None, help="collision rounds per step (0: history mode)")
    ap.add_argument("--block", type=int, default=None, help="threads per workgroup of the step kernels")
    ap.add_argument("--grid-mult", type=int, default=None)
    ap.add_argument("--defer-mask", type=lambda v: int(v, 0), default=None,
                    help="sampler kinds queued in collision rounds (bit = pt_proc_kind)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-traffic", action="store_true",
                    help="skip the two rocprofv3 counter passes that measure HBM traffic")
    ap.add_argument("--no-graph", action="store_true",
                    help="the learned variant steps from the host instead of replaying a captured graph")
    ap.add_argument("--no-unbatched", action="store_true",
                    help="sweep: skip the one-swarm-at-a-time plain run")
    ap.add_argument("--no-learned", action="store_true",
                    help="skip the learned-sampler + captured-graph + autotuned variant")
    ap.add_argument("--no-horizon", action="store_true",
                    help="skip the avalanche over all 5000 steps of its configuration")
    ap.add_argument("--no-sweep", action="store_true",
                    help="skip the batched-sweep leg of the default run")
    ap.add_argument("--cpu-sample", type=int, default=None,
                    help="initial particles of the CPU baseline (default: the workload's)")
    ap.add_argument("--cpu-steps", type=int, default=30)
    ap.add_argument("--copy-calibration", type=int, default=0, metavar="MIB",
                    help="only run a plain device-to-device copy of MIB MiB (to scale the HBM "
                         "byte counters of a profiler) and exit")
    args = ap.parse_args()
    args.steps_given = args.steps is not None
    if args.steps is None:
        args.steps = {"sweep": 40, "beam": 10}.get(args.workload, 300)
    if args.copy_calibration:
        import torch
        n = args.copy_calibration * (1 << 20) // 4
        a = torch.ones(n, dtype=torch.float32, device="cuda")
        b = torch.empty_like(a)
        torch.cuda.synchronize()
        b.copy_(a)
        torch.cuda.synchronize()
        print(json.dumps({"copy_bytes_read": 4 * n, "copy_bytes_written": 4 * n}))
        return
    if args.gpus != 1:
        print("bench.py measures one GPU only: this build has no multi-GPU path "
              "(run with --gpus 1)", file=sys.stderr)
        sys.exit(2)

    traffic = None
    if not args.no_traffic and args.workload == "avalanche":
        # before this process touches the GPU: the counter passes run as child processes
        try:
            traffic = pmc_traffic(args)
        except Exception as e:
            log("traffic passes failed: %r" % (e,))

    import particulator_hip as P
    from particulator_hip import air, co

    if args.workload == "sweep":
        return run_sweep(args, traffic)
    if args.workload == "beam":
        return run_beam(args)
    wl = dict(WORKLOADS[args.workload])
    n = args.n or wl["n"]
    cut = 1e4 * co.eV
    t_setup = time.perf_counter()
    te, tg, tp = air.build_tables(air.composition(), wl["efield"], wl["dt"], cut)
    pops = {}
    for name, tb, tr in (("electron", te, wl["tracked"][0]), ("photon", tg, wl["tracked"][1]),
                         ("positron", tp, wl["tracked"][2])):
        pops[name] = P.Population(wl["cap"], [], tb, cut, tracked=bool(tr))
    mp = P.MultiPopulation(seed=args.seed, **pops)
    mp.set_pusher(P.RK2Pusher(P.ElectromagneticField(P.HomogeneousField((0.0, 0.0, -wl["efield"])))))
    mp.init_particles(P.PT_ELECTRON, n, wl["e1"] * co.eV, (wl["e2"] or wl["e1"]) * co.eV,
                      loguniform=wl["loguniform"])
    mp.init()
    launch = mp.get_launch()
    for k, v in (("rounds", args.rounds), ("block", args.block), ("grid_mult", args.grid_mult),
                 ("defer_mask", args.defer_mask)):
        if v is not None:
            launch[k] = v
    launch["compact_every"] = wl["compact_every"]
    mp.set_launch(**launch)
    log("setup %.1f s, launch %s" % (time.perf_counter() - t_setup, launch))
    dt = wl["dt"]
    t = mp.run_steps(0.0, dt, args.warmup, compact_every=wl["compact_every"], check_every=args.warmup or 1)
    mp.work(reset=True)
    mp.profile(True)
    check(mp)
    t0 = time.perf_counter()
    t = mp.run_steps(t, dt, args.steps, compact_every=wl["compact_every"], check_every=args.steps)
    check(mp)
    el = time.perf_counter() - t0
    w = mp.work(reset=False)
    counts = [mp.count(s) for s in range(3)]
    psteps = w.particle_steps
    value = psteps / el
    adv_avg_ms = w.advance_ms / max(w.advance_launches, 1)
    log("timed %d steps in %.3f s: %.4g particle-steps/s; advance %.3f ms/launch, tail %.3f ms, "
        "compact %.3f ms total; populations %s; events/pstep %.2f; secondaries %d"
        % (args.steps, el, value, adv_avg_ms, w.tail_ms / max(w.advance_launches, 1), w.compact_ms,
           counts, w.events / max(psteps, 1), w.secondaries))
    out = {
        "metric": "particle-steps/s",
        "value": value,
        "unit": "particle-steps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": 1e3 * el / args.steps,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic (device-generated initial particles from a seeded Philox stream)",
        "config": {"workload": wl["name"], "initial_particles": n, "seed": args.seed,
                   "population_end": counts, "events_per_particle_step": w.events / max(psteps, 1)},
        "roofline": roofline(psteps, w.main_secondaries, args.steps, w.advance_launches, adv_avg_ms, value, traffic),
    }
    mp.close()
    nets = {}
    if not args.no_learned:
        try:
            out["learned_batched"], nets = learned_batched(args, wl, n, value)
        except Exception as e:  # the variant must not hide the plain figure
            out["learned_batched"] = {"value": None, "error": repr(e)}
    if not args.no_horizon:
        try:
            out["horizon"] = horizon(args, wl, n)
        except Exception as e:
            out["horizon"] = {"value": None, "error": repr(e)}
    if not args.no_sweep:
        try:
            # the sweep's own step counts (its steps cost ~37 ms each, and the one-swarm-at-a-
            # time form repeats them for each of its 256 contexts)
            sargs = argparse.Namespace(**vars(args))
            sargs.steps, sargs.warmup, sargs.n = min(args.steps, 40), min(args.warmup, 10), None
            out["sweep"] = sweep_leg(sargs, nets)
        except Exception as e:
            out["sweep"] = {"value": None, "error": repr(e)}
    if not args.no_cpu_baseline:
        try:
            out["cpu_baseline"] = cpu_baseline(wl, args.seed, args.cpu_sample or n, args.cpu_steps)
        except Exception as e:  # the CPU leg must not hide the GPU figure
            out["cpu_baseline"] = {"value": None, "error": repr(e)}
    print(json.dumps(out))


FETCH_SCALE = 2.0  # FETCH_SIZE reads 0.5 GiB for a 1 GiB device copy on this GPU
WRITE_SCALE = 1.0  # WRITE_SIZE reads 1 GiB for the same copy


VALU_COUNTERS = ("SQ_WAVES", "SQ_INSTS_VALU", "SQ_ACTIVE_INST_VALU", "SQ_THREAD_CYCLES_VALU", "SQ_WAVE_CYCLES",
                 "SQ_WAIT_ANY")


def pmc_pass(args, counters):
    """Per-dispatch values of `counters` for the main passes of the step's advance kernel,
    from one rocprofv3 counter pass over a short run of this workload (a child process)."""
    import shutil
    import sqlite3
    import subprocess
    import tempfile
    exe = shutil.which("rocprofv3") or "/opt/rocm/bin/rocprofv3"
    d = tempfile.mkdtemp(prefix="pt_pmc_", dir="/tmp")
    cmd = [exe, "--pmc"] + list(counters) + ["-d", d, "-o", "p", "--", sys.executable, os.path.abspath(__file__),
                                             "--workload", args.workload, "--steps", "16", "--warmup", "8",
                                             "--no-learned", "--no-cpu-baseline", "--no-traffic", "--no-horizon",
                                             "--no-sweep"]
    cmd += ["--n", str(args.n)] if args.n else []
    log("counter pass %s" % " ".join(counters))
    subprocess.run(cmd, timeout=240, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL, cwd="/tmp",
                   env=dict(os.environ, TMPDIR="/tmp"), check=False)
    dbs = [os.path.join(r, f) for r, _, fs in os.walk(d) for f in fs if f.endswith("_results.db")]
    if not dbs:
        raise RuntimeError("no results for %s" % (counters,))
    db = sqlite3.connect(dbs[0])
    out = {}
    for ctr in counters:
        rows = db.execute("select value from counters_collection where counter_name = ? and "
                          "kernel_name like '%k_advance<%, 0, false, false, false>%'", (ctr,)).fetchall()
        vals = [r[0] for r in rows]
        if not vals:
            raise RuntimeError("no %s samples for the advance kernel" % ctr)
        # the step's main pass (the short passes over overflow secondaries are left out)
        main = [v for v in vals if v >= 0.1 * max(vals)]
        out[ctr] = (sum(main) / len(main), len(main))
    db.close()
    shutil.rmtree(d, ignore_errors=True)
    return out


def pmc_traffic(args):
    """HBM bytes per launch of the step's advance kernel from two counter passes
    (FETCH_SIZE, then WRITE_SIZE, KiB per dispatch), scaled by what the counters read for a
    plain device copy of known size; and, from a third pass, its vector-instruction figures."""
    kib = {}
    for ctr in ("FETCH_SIZE", "WRITE_SIZE"):
        kib.update(pmc_pass(args, (ctr,)))
    fetch = kib["FETCH_SIZE"][0] * 1024 * FETCH_SCALE
    write = kib["WRITE_SIZE"][0] * 1024 * WRITE_SCALE
    out = {"bytes": fetch + write, "fetch_bytes": fetch, "write_bytes": write,
           "fetch_kib_raw": kib["FETCH_SIZE"][0], "write_kib_raw": kib["WRITE_SIZE"][0],
           "dispatches": kib["FETCH_SIZE"][1], "scale": {"FETCH_SIZE": FETCH_SCALE, "WRITE_SIZE": WRITE_SCALE},
           "note": "counter passes of a run of 24 steps of the same workload, several to a launch"}
    try:
        v = pmc_pass(args, VALU_COUNTERS)
        steps_per_launch = 24.0 / v["SQ_INSTS_VALU"][1]
        v = {k: x[0] for k, x in v.items()}
        n0 = args.n or WORKLOADS[args.workload]["n"]
        import torch
        simds = 4 * torch.cuda.get_device_properties(0).multi_processor_count
        # the grid is persistent (one wave per resident slot), so every SIMD holds
        # SQ_WAVES / simds waves for the whole pass and the wave-cycles of one SIMD sum to
        # that many times the pass's length
        waves_per_simd = v["SQ_WAVES"] / simds
        out["valu"] = {"wave_instructions_per_launch": v["SQ_INSTS_VALU"],
                       "wave_instructions_per_particle_step": v["SQ_INSTS_VALU"] / (n0 * steps_per_launch),
                       "lane_utilisation": v["SQ_THREAD_CYCLES_VALU"] / (64.0 * v["SQ_ACTIVE_INST_VALU"]),
                       "wait_fraction": v["SQ_WAIT_ANY"] / v["SQ_WAVE_CYCLES"],
                       "simds": simds, "waves_per_simd": waves_per_simd,
                       "simd_valu_busy": v["SQ_ACTIVE_INST_VALU"] * waves_per_simd / v["SQ_WAVE_CYCLES"],
                       "note": "the main passes of the same 24-step run: SQ_THREAD_CYCLES_VALU / "
                               "(64 SQ_ACTIVE_INST_VALU), SQ_WAIT_ANY / SQ_WAVE_CYCLES; simd_valu_busy = "
                               "share of each SIMD's time its vector unit issues = SQ_ACTIVE_INST_VALU x "
                               "waves per SIMD / SQ_WAVE_CYCLES"}
    except Exception as e:  # the byte figures stand without it
        out["valu"] = {"error": repr(e)}
    return out


def run_beam(args):
    """The photon pencil beam with its depth-dose and photon-energy tallies."""
    import numpy as np
    import particulator_hip as P
    from particulator_hip import air, co
    wl = WORKLOADS["beam"]
    n = args.n or wl["n"]
    steps = args.steps if args.steps_given else wl["steps"]
    cut, dt = 1e4 * co.eV, wl["dt"]
    te, tg, tp = air.build_tables(air.composition(), 1e6, 1e-12, cut)
    caps = list(wl["caps"])
    caps[1] = max(caps[1], int(1.1 * n))
    mp = P.MultiPopulation(seed=args.seed, tally_bins=512, tally_range=(1e4 * co.eV, 1e7 * co.eV),
                           dose=wl["dose"], tally_tracked=True,
                           electron=P.Population(caps[0], [], te, cut), photon=P.Population(caps[1], [], tg, cut),
                           positron=P.Population(caps[2], [], tp, cut))
    mp.set_pusher(P.RK2Pusher(P.ElectromagneticField(P.HomogeneousField((0.0, 0.0, 0.0)))))
    mp.init_beam(P.PT_PHOTON, n, wl["e1"] * co.eV)
    mp.init()
    # long steps: secondaries of several generations are born in a step
    mp.set_launch(**dict(mp.get_launch(), tail_passes=6))
    t = mp.run_steps(0.0, dt, args.warmup if args.steps_given else 1, compact_every=8, check_every=8)
    mp.work(reset=True)
    mp.profile(True)
    t0 = time.perf_counter()
    t = mp.run_steps(t, dt, steps, compact_every=8, check_every=steps)
    el = time.perf_counter() - t0
    w = mp.work(reset=False)
    hd, under, over, total = mp.dose()
    h1, c1, w1 = mp.tally(1)
    counts = [mp.count(s) for s in range(3)]
    value = w.particle_steps / el
    log("beam: %d steps in %.3f s: %.4g particle-steps/s, %.4g collision events/s; populations %s; "
        "dose %.4g J; photon births %d; advance %.1f ms/launch, last-workgroup tail %.1f ms/launch, secondaries "
        "advanced in their birth step %d" % (steps, el, value, w.events / el, counts, total, c1,
                                             w.advance_ms / max(w.advance_launches, 1),
                                             w.tail_ms / max(w.advance_launches, 1), w.tail_particles))
    peak = int(np.argmax(hd))
    out = {"metric": "particle-steps/s", "value": value, "unit": "particle-steps/s", "n_gpus": 1,
           "steps": steps, "warmup": 1, "ms_per_step": 1e3 * el / steps, "higher_is_better": True,
           "scaling": "weak", "vs_baseline": None, "dtype": "f64",
           "data": "synthetic (device-generated pencil beam, seeded Philox streams)",
           "config": {"workload": wl["name"], "initial_particles": n, "seed": args.seed, "population_end": counts,
                      "collision_events_per_s": w.events / el, "time_s": t},
           "tallies": {"dose_total_J": total, "dose_under_J": under, "dose_over_J": over,
                       "dose_peak_bin": peak, "dose_peak_J": float(hd[peak]),
                       "dose_first_bins_J": [float(v) for v in hd[:4]],
                       "photon_births": c1, "photon_birth_weight": w1}}
    print(json.dumps(out))
    mp.close()


def run_sweep(args, traffic):
    """The batched sweep as the bench line's workload."""
    r = sweep_leg(args, {})
    out = {
        "metric": "particle-steps/s", "value": r["batched_plain"], "unit": "particle-steps/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": r["ms_per_step"],
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f64",
        "data": "synthetic (device-generated initial particles from a seeded Philox stream)",
        "config": r["config"], "learned_batched": r["learned_batched"], "unbatched_plain": r["unbatched_plain"],
        "swarms": r["swarms"]}
    print(json.dumps(out))


def sweep_leg(args, nets):
    """Independent swarms of uneven sizes at different fields advanced together: one
    population with per-swarm fields and rate bounds, the launch chosen by the autotuner,
    steps replayed from a captured graph; then the same with the learned samplers (the
    networks in `nets`, trained and gated in another context of the same air, or trained
    here); and the plain GPU form, each swarm in its own context one after the other.
    Per-swarm growth rate and mean energy are reported."""
    import numpy as np
    import particulator_hip as P
    from particulator_hip import air, co, learned as LS
    wl = WORKLOADS["sweep"]
    ns = wl["nswarm"]
    rng = np.random.default_rng(args.seed)
    counts = rng.integers(wl["count_range"][0], wl["count_range"][1] + 1, size=ns)
    if args.n:
        counts = np.maximum(1, (counts * (args.n / counts.sum())).astype(np.int64))
    fields = wl["field_range"][0] * (wl["field_range"][1] / wl["field_range"][0]) ** (np.arange(ns) / (ns - 1))
    cut, dt = 1e4 * co.eV, wl["dt"]
    t_setup = time.perf_counter()
    te, tg, tp = air.swarm_tables(air.composition(), list(fields), dt, cut)
    cap = int(min(wl["cap"], max(1 << 20, 2 * counts.sum())))
    mp = P.MultiPopulation(seed=args.seed, nswarm=ns,
                           electron=P.Population(cap, [], te, cut, tracked=True),
                           photon=P.Population(1024, [], tg, cut, tracked=False),
                           positron=P.Population(1024, [], tp, cut, tracked=False))
    uid = 0
    for i in range(ns):
        mp.set_pusher(P.RK2Pusher(P.ElectromagneticField(P.HomogeneousField((0.0, 0.0, -fields[i])))), swarm=i)
        mp.init_particles(P.PT_ELECTRON, int(counts[i]), wl["e1"] * co.eV, swarm=i, uid0=uid)
        uid += int(counts[i])
    mp.init()
    s0 = mp.swarm_stats(0)
    log("sweep setup %.1f s: %d swarms, %d electrons, capacity %d" % (time.perf_counter() - t_setup, ns,
                                                                         counts.sum(), cap))
    t = 0.0
    best, trials, t = mp.autotune(t, dt, trial_steps=1)
    log("autotuned launch %s (%d trials)" % (best, len(trials)))
    t = mp.run_graph(t, dt, args.warmup, check_every=max(args.warmup, 1))

    def timed(label):
        nonlocal t
        mp.work(reset=True)
        mp.profile(True)
        t0 = time.perf_counter()
        t = mp.run_graph(t, dt, args.steps, check_every=args.steps)
        el = time.perf_counter() - t0
        w = mp.work(reset=False)
        mp.profile(False)
        log("%s: %d steps in %.3f s: %.4g particle-steps/s" % (label, args.steps, el, w.particle_steps / el))
        return w.particle_steps / el, el
    t_start = t
    v_plain, el = timed("plain")
    s1 = mp.swarm_stats(0)
    unb = None if args.no_unbatched else unbatched(args, wl, (te, tg, tp), counts, fields, int(round(t_start / dt)))
    # learned samplers: the gated networks of another context of the same air, else trained here
    if nets:
        for w, (params, emin, emax) in nets.items():
            LS.install(mp, w, params, emin, emax)
        gates = {LS.NAMES[w]: {"installed": 1, "trained_in": "the avalanche leg's context"} for w in nets}
    else:
        reps = {LS.NAMES[w]: LS.train(mp, w) for w in (LS.SB, LS.MOLLER)}
        gates = {k: {"ks_max": r["ks_max"], "installed": r["installed"]} for k, r in reps.items()}
    # the plain launch the tuner chose; the learned kinds join the deferred ones when it uses rounds
    lb = dict(best, defer_mask=best["defer_mask"] | (1 << 2) | (1 << 4)) if best["rounds"] > 0 else dict(best)
    mp.set_launch(**lb)
    v_learned, _ = timed("learned")
    T = t
    growth = np.log(np.maximum(s1[:, 0], 1) / np.maximum(s0[:, 0], 1)) / max(T - args.steps * dt, dt)
    emean = s1[:, 2] / np.maximum(s1[:, 1], 1e-300) / co.eV
    mp.close()
    return {
        "batched_plain": v_plain, "unit": "particle-steps/s", "ms_per_step": 1e3 * el / args.steps,
        "steps": args.steps,
        "config": {"workload": wl["name"], "swarms": ns, "initial_particles": int(counts.sum()),
                   "seed": args.seed, "launch": best},
        "learned_batched": {"value": v_learned, "ratio_to_batched_plain": v_learned / v_plain, "launch": lb,
                            "ratio_to_unbatched_plain": v_learned / unb["value"] if unb else None,
                            "gates": gates},
        "unbatched_plain": unb,
        "swarms": {"field_V_per_m": [float(fields[0]), float(fields[ns // 2]), float(fields[-1])],
                   "growth_rate_per_s": [float(growth[0]), float(growth[ns // 2]), float(growth[-1])],
                   "mean_energy_eV": [float(emean[0]), float(emean[ns // 2]), float(emean[-1])],
                   "time_s": T},
    }


def unbatched(args, wl, tables, counts, fields, presteps):
    """The plain GPU form of the sweep: each swarm alone in its own population (one run per
    field, as the reference runs a sweep), exact samplers, the default launch, steps from
    the host.  Each swarm first runs `presteps` untimed steps (the batched run's steps
    before its timed window), then the same timed steps; the figure is the summed
    particle-steps over the summed timed wall time."""
    import particulator_hip as P
    from particulator_hip import co
    te, tg, tp = tables
    cut, dt = 1e4 * co.eV, wl["dt"]
    psteps, el, uid = 0, 0.0, 0
    for i in range(len(counts)):
        n = int(counts[i])
        mp = P.MultiPopulation(seed=args.seed, electron=P.Population(
            max(1 << 16, 2 * n), [], te.with_ratebounds(te.ratebound[i:i + 1]), cut, tracked=True),
            photon=P.Population(1024, [], tg, cut, tracked=False),
            positron=P.Population(1024, [], tp.with_ratebounds(tp.ratebound[i:i + 1]), cut, tracked=False))
        mp.set_pusher(P.RK2Pusher(P.ElectromagneticField(P.HomogeneousField((0.0, 0.0, -fields[i])))))
        mp.init_particles(P.PT_ELECTRON, n, wl["e1"] * co.eV, uid0=uid)
        uid += n
        mp.init()
        t = mp.run_steps(0.0, dt, presteps, compact_every=8, check_every=max(presteps, 1))
        mp.work(reset=True)
        t0 = time.perf_counter()
        mp.run_steps(t, dt, args.steps, compact_every=8, check_every=args.steps)
        el += time.perf_counter() - t0
        psteps += mp.work(reset=False).particle_steps
        mp.close()
    log("unbatched plain: %d swarms one at a time, %d steps each: %.4g particle-steps/s"
        % (len(counts), args.steps, psteps / el))
    return {"value": psteps / el, "unit": "particle-steps/s", "seconds": el, "particle_steps": psteps,
            "untimed_steps_before": presteps,
            "note": "each swarm in its own population, exact samplers, default launch, host-stepped"}


def make_world(args, wl, n):
    import particulator_hip as P
    from particulator_hip import air, co
    cut = 1e4 * co.eV
    te, tg, tp = air.build_tables(air.composition(), wl["efield"], wl["dt"], cut)
    pops = {}
    for name, tb, tr in (("electron", te, wl["tracked"][0]), ("photon", tg, wl["tracked"][1]),
                         ("positron", tp, wl["tracked"][2])):
        pops[name] = P.Population(wl["cap"], [], tb, cut, tracked=bool(tr))
    mp = P.MultiPopulation(seed=args.seed, **pops)
    mp.set_pusher(P.RK2Pusher(P.ElectromagneticField(P.HomogeneousField((0.0, 0.0, -wl["efield"])))))
    mp.init_particles(P.PT_ELECTRON, n, wl["e1"] * co.eV, (wl["e2"] or wl["e1"]) * co.eV,
                      loguniform=wl["loguniform"])
    mp.init()
    return mp


def learned_batched(args, wl, n, plain_value):
    """The same workload with the learned bremsstrahlung and Moller samplers (trained on the
    device, gated at KS <= 0.01, evaluated on the matrix cores wherever those collisions are
    sampled), the launch shape, collision rounds and compaction cadence chosen by the
    autotuner, and the steps replayed from a captured graph.  Returns its throughput beside
    the plain figure."""
    import numpy as np
    from particulator_hip import learned as LS
    mp = make_world(args, wl, n)
    t = time.perf_counter()
    reps = {LS.NAMES[w]: LS.train(mp, w) for w in (LS.SB, LS.MOLLER)}
    train_s = time.perf_counter() - t
    installed = all(r["installed"] for r in reps.values())
    # the gated networks, for the sweep leg's contexts (same air, same samplers)
    nets = {w: (LS.get_params(mp, w), LS.defaults(w)["emin"], LS.defaults(w)["emax"])
            for w in (LS.SB, LS.MOLLER) if reps[LS.NAMES[w]]["installed"]}
    launch = mp.get_launch()
    # collision rounds, when the tuner tries them, carry the two learned kinds
    launch.update(defer_mask=(1 << 2) | (1 << 4))
    mp.set_launch(**launch)
    dt = wl["dt"]
    best, trials, tnow = mp.autotune(0.0, dt, trial_steps=4)
    mp.set_launch(**best)
    log("learned samplers trained in %.1f s (installed: %s); autotuned launch %s" % (train_s, installed, best))
    def steps(t, k, check):
        if args.no_graph:
            return mp.run_steps(t, dt, k, compact_every=best["compact_every"], check_every=check)
        return mp.run_graph(t, dt, k, check_every=check)
    tnow = steps(tnow, args.warmup, max(args.warmup, 1))
    mp.work(reset=True)
    mp.collision_counts(0, reset=True)
    mp.profile(True)
    t0 = time.perf_counter()
    tnow = steps(tnow, args.steps, args.steps)
    el = time.perf_counter() - t0
    w = mp.work(reset=False)
    value = w.particle_steps / el
    # what the networks can gain here: the share of the electrons' real collisions they
    # sample, and their samples/s against the rejection samplers they replace
    counts = mp.collision_counts(0)
    kinds = [type(pr).__name__ for pr in mp.get("electron").collisions.proc]
    real = float(sum(counts[1:1 + len(kinds)]))
    replaced = float(sum(counts[1 + i] for i, k in enumerate(kinds) if k in ("SeltzerBerger", "Moller")))
    rates = {}
    for wk in (LS.SB, LS.MOLLER):
        d = LS.defaults(wk)
        T = np.geomspace(d["emin"] * 1.01, d["emax"] * 0.99, 64)
        Z = np.tile(np.array([7, 8, 18], dtype=np.int32), 22)[:64]
        net, rej = LS.throughput(mp, wk, True, T, Z), LS.throughput(mp, wk, False, T, Z)
        rates[LS.NAMES[wk]] = {"network_samples_per_s": net, "rejection_samples_per_s": rej, "ratio": net / rej}
    log("learned+batched: %d steps in %.3f s: %.4g particle-steps/s (%.3fx plain); the networks sample %.2g of "
        "the real electron collisions; network/rejection samples/s %s"
        % (args.steps, el, value, value / plain_value, replaced / max(real, 1.0),
           {k: round(v["ratio"], 3) for k, v in rates.items()}))
    mp.close()
    return {"value": value, "unit": "particle-steps/s", "ratio_to_plain": value / plain_value,
            "replaced_collision_share": replaced / max(real, 1.0), "sampler_throughput": rates,
            "captured_graph": not args.no_graph,
            "graph_replay_ms_per_step": w.graph_ms / args.steps if not args.no_graph else None,
            "ms_per_step": 1e3 * el / args.steps, "launch": best, "learned_installed": installed,
            "training_s": train_s,
            "gates": {k: {"ks_max": r["ks_max"], "ks_mean": r["ks_mean"], "ks_noise": r["ks_noise"],
                          "installed": r["installed"], "samples": r["samples"],
                          "data_ms": r["gen_ms"], "train_ms": r["train_ms"], "gate_ms": r["eval_ms"]}
                      for k, r in reps.items()},
            "autotune_trials": len(trials)}, nets


def horizon(args, wl, n):
    """The avalanche over its full length: every step of the configuration (5000 x 1 ps)
    from the initial particles, host-stepped with compaction every 8 steps, timed as a
    whole; particle-steps/s, step times at the start and the end, end populations."""
    mp = make_world(args, wl, n)
    dt, total, chunk = wl["dt"], wl["horizon_steps"], 500
    mp.work(reset=True)
    t, done, psteps, first, last = 0.0, 0, 0, None, None
    t0 = time.perf_counter()
    while done < total:
        k = min(chunk, total - done)
        c0 = time.perf_counter()
        t = mp.run_steps(t, dt, k, compact_every=wl["compact_every"], check_every=k)
        ms = 1e3 * (time.perf_counter() - c0) / k
        first = ms if first is None else first
        last = ms
        done += k
        log("horizon: %d / %d steps, %.3f ms/step, populations %s" % (done, total, ms,
                                                                     [mp.count(s) for s in range(3)]))
    el = time.perf_counter() - t0
    check(mp)
    w = mp.work(reset=False)
    pops = [mp.get(s).nactives() for s in ("electron", "photon", "positron")]
    mp.close()
    return {"steps": total, "seconds": el, "value": w.particle_steps / el, "unit": "particle-steps/s",
            "ms_per_step_first_500": first, "ms_per_step_last_500": last, "time_s": t,
            "population_end_active": pops, "secondaries": w.secondaries,
            "note": "all 5000 steps of the configuration from t = 0 in a fresh context (host-stepped, "
                    "compaction every 8), capacity flags checked at the end"}


def check(mp):
    rc, flags = mp.flags()
    if rc != 0:
        raise SystemExit("device error flags %s" % flags)


if __name__ == "__main__":
    main()
