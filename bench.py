"""Benchmark: a 32-qubit random grid circuit on one MI355X.

One step = one full circuit (|0..0> preparation plus every fused pass) on a
complex64 state resident in HBM.  The circuit is the 4x8 grid, 20 cycles,
seed 0 construction of qsim_amd/circuits.py, fused by qsim's
MultiQubitGateFuser (or the blocked-pass planner) and applied by qsim's own
apply loop over the gfx950 kernels.  The paths run on the same circuit:

  plain-fp32-vector  max_fused_size 4, FP32 vector kernels (qsim's method)
  fp32-mfma          max_fused_size 4, exact-FP32 MFMA for the k=4 passes
  bf16-k6            max_fused_size 6, fused matrices built in FP64 on the
                     host, split-BF16 MFMA for k>=5 passes
  fp16-k5, fp16-k6   max_fused_size 5 / 6, FP64-built fused matrices, FP16
                     MFMA with a power-of-two scale per matrix and per group
                     for k>=5 passes
  blocked-13         cache-blocked passes over 13 tile qubits (5 lowest + 8
                     chosen), gates fused to <= 4 qubits in FP64 inside each
                     pass, FP16 MFMA with a power-of-two scale per tile on
                     the LDS-resident tile
  blocked-14         the same over 14 tile qubits (4 lowest + 10 chosen; one
                     128 KiB tile per CU, fewer passes)
  blocked-14-bf16    blocked-14 on the split-BF16 product instead of FP16
  learned            the partition the learned planner picks for this
                     circuit with the committed cost model
                     (qsim_amd/data/cost_model.json), among qsim's fuser at
                     max_fused_size 2..6 x gate methods and blocked passes

Each path's fidelity F = |<psi64|psi>|^2 / (<psi64|psi64> <psi|psi>) is
measured on the same construction at 28 qubits against a complex128 run of
the same circuit on the GPU (FP64 gate matrices and FP64 vector kernels;
that path is checked against the CPU FP64 oracle by the tests), with the
norm drift |<psi|psi> - 1| beside it.  `value` is the learned planner's
pick when it meets 1 - F <= 1e-6 with a norm drift <= 1e-5, else the
fastest path that does.  Beside the headline, the batched trajectory engine
runs its own workload (1024 noisy trajectories of 18/20/22 qubits), and the
20-qubit grid circuit runs eagerly and as one captured graph.

Prints one JSON line with the roofline of that path's dominant gate kernel
(HIP events around every pass inside the timed region) and qsim's own
AVX/OpenMP CPU path timed on a bounded sample of the same circuit.

    python bench.py [--gpus 1] [--steps 3] [--warmup 1] [--qubits 32]
                    [--cycles 20] [--paths a,b,c] [--cpu-passes P | --no-cpu]
                    [--no-fidelity]
"""

from __future__ import annotations

import argparse
import json
import os
import sys
import tempfile
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBPS = 8000.0
METRIC = ("32q circuit time + HBM GB/s, learned/MFMA vs plain FP32 fusion "
          "at F>=1-1e-6")

# name -> (partition, max_fused_size or tile qubits, FP64 fused matrices or
# low tile qubits, gate method, blocked-pass arithmetic)
PATHS = {
    "plain-fp32-vector": ("mqubit", 4, False, 1, "f16"),
    "fp32-mfma": ("mqubit", 4, False, 0, "f16"),
    "bf16-k6": ("mqubit", 6, True, 2, "f16"),
    "fp16-k5": ("mqubit", 5, True, 3, "f16"),
    "fp16-k6": ("mqubit", 6, True, 3, "f16"),
    "blocked-13": ("blocked", 13, 5, 0, "f16"),
    "blocked-14": ("blocked", 14, 4, 0, "f16"),
    "blocked-14-bf16": ("blocked", 14, 4, 0, "bf16"),
    # the learned planner's pick (qsim_amd/data/cost_model.json)
    "learned": ("learned", 0, 0, 0, "f16"),
}
# The fusion sweep of the 30-qubit workload: qsim's fuser at
# max_fused_size k with qsim's FP32 fused matrices on the FP32 kernels
# (vector kernels below k = 4, exact-FP32 MFMA from k = 4).
for _k in range(2, 7):
    PATHS[f"fp32-k{_k}"] = ("mqubit", _k, False, 0, "f16")
SWEEP_PATHS = [f"fp32-k{k}" for k in range(2, 7)]

# HBM bytes per amplitude per launch from rocprofv3 FETCH_SIZE / WRITE_SIZE
# runs, scaled by what the counters read for a copy of known size (reads x 2,
# writes x 1); profiles/gate_passes_32q_blocked_vs_fused.md ("The 14-qubit pass
# with IO waves" for GateBlockF16IoKernel).
MEASURED_HBM_BYTES_PER_AMP = {"GateBlockF16IoKernel": 16.00,
                              "GateBlockKernel": 16.04}

# MFMA flops issued per amplitude per 4-qubit op of a blocked pass: a batch
# of 32 groups (512 amplitudes) takes 2 K blocks x (3 FP16 or 4 split-BF16
# products) MFMAs of 32 x 32 x 16.
BLOCK_FLOPS_PER_AMP_OP = {"GateBlockF16IoKernel": 6 * 2 * 32 * 32 * 16 / 512.0,
                          "GateBlockF16Kernel": 6 * 2 * 32 * 32 * 16 / 512.0,
                          "GateBlockKernel": 8 * 2 * 32 * 32 * 16 / 512.0}
# Dense MFMA peak of MI355X, fp16 and bf16 alike.
MFMA_F16_PEAK_TFLOPS = 2500.0


def log(*a):
    print(*a, file=sys.stderr, flush=True)


_MODEL = None


def fuse(circ, name):
    """Partitions the circuit for path `name`; returns (passes, gate method,
    planner pick or None)."""
    global _MODEL
    from qsim_amd import costmodel, driver
    part, a, b, method, arith = PATHS[name]
    circ.set_block_arith(arith)
    if part == "learned":
        if _MODEL is None:
            _MODEL = costmodel.CostModel.load()
        chosen, cands = circ.plan_learned(_MODEL)
        return circ.num_passes, cands[chosen]["method"], cands[chosen]
    if part == "blocked":
        return circ.fuse_blocked(a, b), method, None
    return circ.fuse(a, driver.FUSER_MQUBIT, f64_matrices=b), method, None


def available_paths():
    from qsim_amd import costmodel
    return [p for p in PATHS if p not in SWEEP_PATHS and
            (PATHS[p][0] != "learned" or os.path.exists(costmodel.MODEL_PATH))]


def kernel_family(circ, i, qubits, method, n, arith="f16"):
    """The gate kernel a pass runs (qsim_amd/csrc: gate_kernels.hip,
    mfma_kernels.hip, f16_kernels.hip and block_kernels.hip dispatch).
    Blocked passes of unitary gates run the FP16 kernels (14 tile qubits:
    GateBlockF16IoKernel) unless the split-BF16 arithmetic is asked for."""
    from qsim_amd import driver
    if circ.pass_kind(i) == driver.PASS_BLOCKED:
        if arith != "f16":
            return "GateBlockKernel"
        return "GateBlockF16IoKernel" if len(qubits) == 14 else "GateBlockF16Kernel"
    k = len(qubits)
    low = bool(qubits) and min(qubits) < 5
    if method != 1 and 4 <= k <= 6 and n >= k + 5:
        if method == 2 and k >= 5:
            if n >= 11:
                return "GateBf16RowSetKernel" if low else "GateBf16RowRegKernel"
            return "GateBf16TileKernel" if low else "GateBf16RegKernel"
        if method == 3 and k >= 5 and n >= 12:
            return "GateF16SetKernel" if low else "GateF16RegKernel"
        if method == 0 and k >= 5 and n >= 11:
            return "GateF32RowSetKernel" if low else "GateF32RowRegKernel"
        if k == 4:
            return "GateMfmaLaneKernel"
        return "GateMfmaTileKernel" if low else "GateMfmaRegKernel"
    if n >= k + 6 and (k == 4 or (k < 4 and low)):
        return "GateLaneKernel"
    return "GateTileKernel" if low else "GateRegKernel"


def run_path(args, text, name):
    import qsim_amd
    from qsim_amd import driver

    part, kmax, f64m, _, arith = PATHS[name]
    circ = driver.Circuit(text)
    t0 = time.time()
    npass, method, pick = fuse(circ, name)
    fuse_s = time.time() - t0
    if pick is not None:
        log(f"[{name}] planner pick: {pick}")
        part = "blocked" if pick["blocked"] else "mqubit"
        kmax = pick["a"]
        f64m = pick["b"] if pick["blocked"] else True
    passes = circ.passes()
    n = circ.num_qubits
    block_ops = [len(circ.block_info(i)) if
                 circ.pass_kind(i) == driver.PASS_BLOCKED else 0
                 for i in range(npass)]
    log(f"[{name}] {circ.num_gates} gates -> {npass} passes "
        f"(k histogram {np.bincount([len(q) for q, _ in passes]).tolist()}, "
        f"{sum(block_ops)} fused gates in blocked passes), "
        f"fuse {fuse_s:.3f}s")
    qsim_amd.set_gate_method(method)
    ss = qsim_amd.StateSpace(np.float32)
    st = ss.create(n)
    if st is None:
        raise RuntimeError("cannot allocate the state")
    try:
        for w in range(args.warmup):
            ss.set_state_zero(st)
            circ.run(st)
            qsim_amd.synchronize()
        qsim_amd.synchronize()
        qsim_amd.PassTimer.start(npass * args.steps + 16)
        qsim_amd.Timer.record(0)
        t_wall = time.time()
        for _ in range(args.steps):
            ss.set_state_zero(st)
            circ.run(st)
        qsim_amd.Timer.record(1)
        qsim_amd.synchronize()
        wall = time.time() - t_wall
        total_ms = qsim_amd.Timer.elapsed_ms(0, 1)
        pass_ms = qsim_amd.PassTimer.stop(npass * args.steps + 16)
        norm = ss.norm(st)
    finally:
        qsim_amd.set_gate_method(0)
        st.free()
    log(f"[{name}] {args.steps} circuits in {total_ms:.1f} ms "
        f"(wall {wall:.3f}s), {len(pass_ms)} passes timed, norm {norm:.9f}")
    if args.pass_times and len(pass_ms) == npass * args.steps:
        # Median over the timed circuits of each pass, with its qubits (the
        # tile qubits of a blocked pass) and fused gates.
        med = np.median(np.asarray(pass_ms).reshape(args.steps, npass), 0)
        for i, ((q, _), ms) in enumerate(zip(passes, med)):
            log(f"[{name}] pass {i}: {float(ms):.3f} ms, qubits {list(q)}, "
                f"fused gates {block_ops[i] or 1}")

    bytes_per_pass = 16.0 * (1 << n)   # every complex64 read and written once
    fams = [kernel_family(circ, i, q, method, n, arith)
            for i, (q, _) in enumerate(passes)] * args.steps
    per_fam = {}
    flops = {}
    for i, (f, ms) in enumerate(zip(fams, pass_ms)):
        per_fam.setdefault(f, []).append(float(ms))
        flops.setdefault(f, []).append(
            BLOCK_FLOPS_PER_AMP_OP.get(f, 0.0) * block_ops[i % npass]
            * (1 << n))
    fam_stats = {}
    for f, v in per_fam.items():
        avg = float(np.mean(v))
        fam_stats[f] = {"passes": len(v), "avg_ms": avg,
                        "total_ms": float(np.sum(v)),
                        "achieved_gbps": bytes_per_pass / (avg * 1e-3) / 1e9}
        if f in BLOCK_FLOPS_PER_AMP_OP:
            tf = float(np.sum(flops[f])) / (float(np.sum(v)) * 1e-3) / 1e12
            fam_stats[f]["mfma_tflops"] = tf
            fam_stats[f]["mfma_frac"] = tf / MFMA_F16_PEAK_TFLOPS
            fam_stats[f]["avg_ops_per_pass"] = (
                float(np.mean([o for o in block_ops if o])))
    dominant = max(fam_stats, key=lambda f: fam_stats[f]["total_ms"])
    d = fam_stats[dominant]
    per_k = {}
    for (q, _), ms in zip(passes * args.steps, pass_ms):
        per_k.setdefault(len(q), []).append(float(ms))
    k_stats = {str(k): {"passes": len(v), "avg_ms": float(np.mean(v)),
                        "gbps": bytes_per_pass / (float(np.mean(v)) * 1e-3) / 1e9}
               for k, v in sorted(per_k.items())}
    return {
        "name": name, "partition": part, "planner_pick": pick,
        "max_fused_size": kmax if part == "mqubit" else 4,
        "fp64_matrices": bool(f64m) if part == "mqubit" else True,
        "tile_qubits": kmax if part == "blocked" else None,
        "low_tile_qubits": f64m if part == "blocked" else None,
        "num_qubits": n, "num_gates": circ.num_gates, "passes": npass,
        "circuit_s": total_ms / args.steps / 1e3, "wall_s": wall,
        "final_norm": norm, "fuse_s": fuse_s,
        # host planning (fusion or the learned pick) plus one circuit
        "plan_plus_circuit_s": fuse_s + total_ms / args.steps / 1e3,
        "pass_ms_sum": float(np.sum(pass_ms)) / args.steps,
        "hbm_gbps_avg_pass": bytes_per_pass / (float(np.mean(pass_ms)) * 1e-3) / 1e9,
        "gate_passes_per_s": npass / (total_ms / args.steps / 1e3),
        "kernels": fam_stats, "per_k": k_stats,
        "roofline": {
            "bound": "hbm", "kernel": dominant,
            "achieved": d["achieved_gbps"], "peak": HBM_PEAK_GBPS,
            "unit": "GB/s", "frac": d["achieved_gbps"] / HBM_PEAK_GBPS,
            "traffic": (MEASURED_HBM_BYTES_PER_AMP[dominant] * (1 << n)
                        if dominant in MEASURED_HBM_BYTES_PER_AMP else None),
            "bytes_per_launch": bytes_per_pass,
            "avg_launch_ms": d["avg_ms"],
        },
    }


def _rel_diff64(ss64, a, b):
    """||a - b|| / ||b|| of two complex128 states on the device; a is
    overwritten with a - b (b is negated and restored, exactly)."""
    nb = ss64.norm(b)
    ss64.multiply(-1.0, b)
    ss64.add(b, a)
    ss64.multiply(-1.0, b)
    return float(np.sqrt(ss64.norm(a) / nb))


def fidelities(args, names, picks=None):
    """1 - F (normalised states) and the norm drift of each path at
    --fidelity-qubits qubits against the complex128 run (FP64 fused
    matrices, FP64 kernels; the tests pin that run to qsim's
    SimulatorBasic<double> at 28 qubits within 1e-12), and each path's
    relative L2 distance from the unfused complex64 run of the same circuit
    (every gate its own FP32 pass, as QSimRunner would apply the circuit
    without fusion).  A path with a planner pick in `picks` (the learned
    planner's choice at the benchmark size) is measured with that same
    partition kind, not re-planned at the smaller size."""
    import qsim_amd
    from qsim_amd import circuits, driver

    nq = args.fidelity_qubits
    text = circuits.grid_circuit(nq, args.cycles, args.seed)
    ss64 = qsim_amd.StateSpace(np.float64)
    ref = ss64.create(nq)
    ss64.set_state_zero(ref)
    c64 = driver.Circuit(text)
    c64.fuse(4, driver.FUSER_MQUBIT, f64_matrices=True)
    c64.run(ref)
    out = {}
    ss32 = qsim_amd.StateSpace(np.float32)
    tmp = ss64.create(nq)
    unfused = ss64.create(nq)
    cu = driver.Circuit(text)
    cu.fuse(1, driver.FUSER_NONE)
    st = ss32.create(nq)
    try:
        ss32.set_state_zero(st)
        cu.run(st)
        ss64.copy(st, unfused)
    finally:
        st.free()
    log(f"unfused complex64 run at {nq}q: {cu.num_passes} passes")
    for name in names:
        c = driver.Circuit(text)
        pick = (picks or {}).get(name)
        if pick is not None:
            c.apply_candidate(pick)
            method = pick["method"]
        else:
            _, method, _ = fuse(c, name)
        qsim_amd.set_gate_method(method)
        st = ss32.create(nq)
        try:
            ss32.set_state_zero(st)
            c.run(st)
            ss64.copy(st, tmp)       # complex64 -> complex128 on the device
        finally:
            qsim_amd.set_gate_method(0)
            st.free()
        ip = ss64.inner_product(ref, tmp)
        n64 = ss64.norm(ref)
        n32 = ss64.norm(tmp)
        f_raw = abs(ip) ** 2
        f = f_raw / (n64 * n32)
        rel_unfused = _rel_diff64(ss64, tmp, unfused)
        out[name] = {"qubits": nq, "one_minus_F": 1.0 - f,
                     "norm_drift": abs(n32 - 1.0),
                     "one_minus_F_unnormalised": 1.0 - f_raw, "norm": n32,
                     "rel_l2_vs_unfused": rel_unfused}
        log(f"[{name}] {nq}q: 1-F = {1.0 - f:.3e}, norm drift "
            f"{abs(n32 - 1.0):.3e} (1-|<psi64|psi>|^2 = {1.0 - f_raw:.3e}), "
            f"rel-L2 vs unfused {rel_unfused:.2e}")
    ref.free()
    tmp.free()
    unfused.free()
    return out


def host_cores():
    """Threads for the CPU baseline: every CPU this process may run on (its
    affinity set), capped by OMP_NUM_THREADS where the host sets it (the
    GPU host gives each GPU's jobs a share of its cores that way); and the
    counts behind the choice."""
    aff = len(os.sched_getaffinity(0))
    omp = int(os.environ.get("OMP_NUM_THREADS", "0") or 0)
    threads = min(aff, omp) if omp > 0 else aff
    return threads, {"affinity_cpus": aff, "machine_cpus": os.cpu_count(),
                     "omp_num_threads": omp or None}


def run_cpu_baseline(args, circuit_file):
    """qsim's own CPU path on the same circuit file: QSimRunner::Run with
    MultiQubitGateFuser at max_fused_size 4 (lib/run_qsim.h:225-289) on the
    simulator lib/simmux.h selects for the host (SimulatorAVX512 where the
    CPU has AVX-512, else SimulatorAVX), every core of the process's share.
    The whole circuit is timed unless --cpu-passes P bounds it to the first
    P fused passes (then scaled by the pass count)."""
    import oracle
    threads, cores = host_cores()
    if args.cpu_threads:
        threads = args.cpu_threads
    p = args.cpu_passes if args.cpu_passes > 0 else None
    log(f"cpu baseline: qsim QSimRunner on the host's widest SIMD simulator, "
        f"{threads} threads ({cores}), "
        + (f"first {p} passes" if p else "full circuit"))
    t0 = time.time()
    info = oracle.run_reference(circuit_file, mode="avx", max_fused=4,
                                threads=threads, passes=p, timeout=1800,
                                widest_simd=True)
    wall = time.time() - t0
    if p:
        per_pass = info["sim_s"] / max(1, min(p, info["fused_ops"]))
        per_circuit = per_pass * info["fused_ops"]
        sample = (f"first {p} of {info['fused_ops']} fused passes "
                  f"(MultiQubitGateFuser k=4) of the same "
                  f"{info['num_qubits']}q circuit; seconds per pass x passes "
                  f"per circuit")
    else:
        per_circuit = info["sim_s"]
        sample = (f"full circuit: QSimRunner::Run (MultiQubitGateFuser k=4, "
                  f"{info['fused_ops']} fused passes, fusion included) of the "
                  f"same {info['num_qubits']}q circuit file")
    log(f"cpu baseline: {info['simulator']} {info['sim_s']:.2f}s "
        f"({info['fused_ops']} passes/circuit), process wall {wall:.1f}s")
    return {
        "value": per_circuit, "unit": "s/circuit", "cores": threads,
        "kind": "reference",
        "sample": (f"{sample} on qsim's {info['simulator']} (oracle/_ref), "
                   f"{threads} OpenMP threads"),
        "simulator": info["simulator"], "host": cores,
        "sample_s": info["sim_s"], "passes_per_circuit_cpu": info["fused_ops"],
    }


def run_grid30(args):
    """The 30-qubit workload (5 x 6 grid, 20 cycles, seed 0, 8 GiB of
    complex64): qsim's fuser swept over max_fused_size 2..6 on the FP32
    kernels, each pass's HBM GB/s, and qsim's own CPU path (QSimRunner with
    MultiQubitGateFuser k = 4 on the host's widest SIMD simulator, every
    core of the process's share) on the whole circuit.  Reported beside the
    headline."""
    from qsim_amd import circuits
    n, cycles = 30, 20
    text = circuits.grid_circuit(n, cycles, 0)
    out = {"workload": "30q random grid circuit 5x6, 20 cycles, seed 0, "
                       "complex64, qsim fuser k=2..6, FP32 kernels",
           "per_k": {}}
    for name in SWEEP_PATHS:
        r = run_path(args, text, name)
        out["per_k"][name.split("-k")[1]] = {
            "passes": r["passes"], "circuit_s": r["circuit_s"],
            "hbm_gbps_avg_pass": r["hbm_gbps_avg_pass"],
            "frac_of_hbm_peak": r["hbm_gbps_avg_pass"] / HBM_PEAK_GBPS,
            "kernels": r["kernels"], "final_norm": r["final_norm"]}
    if not args.no_cpu:
        with tempfile.TemporaryDirectory() as tmp:
            cf = os.path.join(tmp, "grid30.txt")
            with open(cf, "w") as f:
                f.write(text)
            try:
                out["cpu_baseline"] = run_cpu_baseline(args, cf)
            except Exception as e:  # reported, never silently replaced
                log(f"30q cpu baseline failed: {e!r}")
                out["cpu_baseline"] = {"value": None, "error": repr(e)}
    return out


def run_trajectories(args):
    """The batched noisy-trajectory engine on its own workload: 1024
    trajectories of the grid circuit at 18, 20 and 22 qubits (341-342 each),
    12 cycles, depolarising p = 1e-3 after every gate and amplitude damping
    gamma = 5e-3 per qubit per cycle; one launch per batch, graph-replayed.
    Reported beside the headline number, not as it."""
    from qsim_amd import trajectories
    sizes = [18, 20, 22]
    ntraj = args.trajectories
    b = trajectories.TrajectoryBatch(sizes, 12, p_depol=1e-3, gamma_damp=5e-3)
    circuit_of = [i % 3 for i in range(ntraj)]
    reps = list(range(ntraj))
    b.plan(circuit_of, reps, 4)
    threads, plan, tune = b.autotune(log=log)
    plan_s = b.plan(circuit_of, reps, plan)  # host planning of the pick
    b.run(threads, use_graph=True)
    times = []
    for _ in range(3):
        t0 = time.time()
        b.run(threads, use_graph=True)
        times.append(time.time() - t0)
    best = min(times)
    zz_mean = float(np.mean([np.mean(b.zz(t)) for t in range(ntraj)]))
    kernel = "tiled" if threads == trajectories.TILED else f"{threads} threads"
    log(f"trajectories: {ntraj} in {best * 1e3:.1f} ms "
        f"({ntraj / best:.0f}/s), {kernel}, "
        f"{trajectories.describe_plan(plan)}, host plan {plan_s:.2f}s")
    out = {"workload": "grid circuit 18/20/22 qubits, 12 cycles, "
                       "depolarise 1e-3 + amplitude damping 5e-3",
           "trajectories": ntraj, "batch_ms": best * 1e3,
           "trajectories_per_s": ntraj / best,
           "trajectories_per_s_with_host_planning": ntraj / (best + plan_s),
           "kernel": kernel, "plan": trajectories.describe_plan(plan),
           "host_plan_s": plan_s,
           "autotune": tune, "mean_zz": zz_mean}
    b.free()
    if not args.no_cpu:
        try:
            out["cpu_baseline"] = trajectories_cpu(args, sizes)
        except Exception as e:  # reported, never silently replaced
            out["cpu_baseline"] = {"value": None, "error": repr(e)}
    return out


def run_small_circuit(args):
    """The 20-qubit grid circuit (4x5, 14 cycles, seed 0, max_fused_size 2:
    qsim's own CPU-runnable case) run eagerly, one pass at a time from the
    host, and as one captured graph with every matrix resident on the
    device.  At 8 MiB of state this workload is bound by per-pass host work
    and launch latency, not by HBM; reported beside the headline."""
    import qsim_amd
    from qsim_amd import circuits, driver
    n, cycles = 20, 14
    c = driver.Circuit(circuits.grid_circuit(n, cycles, 0))
    c.fuse(2)
    ss = qsim_amd.StateSpace(np.float32)
    st = ss.create(n)

    def timed(fn, reps=20):
        ss.set_state_zero(st)
        fn()
        qsim_amd.synchronize()
        best = float("inf")
        for _ in range(reps):
            ss.set_state_zero(st)
            qsim_amd.synchronize()
            t0 = time.perf_counter()
            fn()
            qsim_amd.synchronize()
            best = min(best, time.perf_counter() - t0)
        return best

    eager = timed(lambda: c.run(st))
    want = st.to_numpy()
    ss.set_state_zero(st)
    g = c.capture(st)
    graph = timed(g.launch)
    same = bool(np.array_equal(st.to_numpy(), want))
    g.free()
    st.free()
    log(f"20q grid circuit (k=2, {c.num_passes} passes): eager "
        f"{eager * 1e3:.2f} ms, graph {graph * 1e3:.2f} ms, identical {same}")
    return {"workload": "20q random grid circuit 4x5, 14 cycles, seed 0, "
                        "complex64, max_fused_size 2",
            "passes": c.num_passes, "eager_ms": eager * 1e3,
            "graph_ms": graph * 1e3, "graph_speedup": eager / graph,
            "graph_identical_to_eager": same}


def stream_ceiling(n):
    """GB/s of the backend's plainest in-place pass (ScaleKernel: each
    complex64 amplitude read and written once, grid-stride) on an n-qubit
    state: the practical ceiling a gate pass is held against, beside the
    nominal 8 TB/s.  Best of 5 after a warm-up, from HIP events."""
    import qsim_amd
    ss = qsim_amd.StateSpace(np.float32)
    st = ss.create(n)
    ss.set_state_uniform(st)
    ss.multiply(1.0, st)
    best = float("inf")
    for _ in range(5):
        qsim_amd.Timer.record(0)
        ss.multiply(1.0, st)
        qsim_amd.Timer.record(1)
        best = min(best, qsim_amd.Timer.elapsed_ms(0, 1))
    st.free()
    gbps = 16.0 * (1 << n) / (best * 1e-3) / 1e9
    log(f"stream ceiling (ScaleKernel, {n}q): {best:.2f} ms = {gbps:.0f} GB/s")
    return {"kernel": "ScaleKernel", "ms": best, "achieved": gbps,
            "frac_of_peak": gbps / HBM_PEAK_GBPS}


def trajectories_cpu(args, sizes):
    """qsim's QuantumTrajectorySimulator (oracle/_ref) on a sample of the
    batch: 4 trajectories per size, scaled to the batch's mix."""
    import oracle
    from qsim_amd import circuits
    threads, cores = host_cores()
    if args.cpu_threads:
        threads = args.cpu_threads
    per = 4
    total = 0.0
    with tempfile.TemporaryDirectory() as tmp:
        for n in sizes:
            f = os.path.join(tmp, f"g{n}.txt")
            with open(f, "w") as fh:
                fh.write(circuits.grid_circuit(n, 12, 0))
            rows, cols = circuits.grid_shape(n)
            _, s = oracle.run_reference_trajectories(
                f, rows, cols, 0, per, 1e-3, 5e-3, max_fused=4,
                threads=threads, widest_simd=True)
            total += s["sim_s"] / per
    per_traj = total / len(sizes)
    return {"value": 1.0 / per_traj, "unit": "trajectories/s",
            "cores": threads, "host": cores, "kind": "reference",
            "sample": f"{per} trajectories per size on qsim's "
                      f"QuantumTrajectorySimulator + SimulatorAVX, "
                      f"{threads} OpenMP threads"}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--qubits", type=int, default=32)
    ap.add_argument("--cycles", type=int, default=20)
    ap.add_argument("--seed", type=int, default=0)
    ap.add_argument("--paths", default="",
                    help="comma-separated subset of " + ",".join(PATHS) +
                    " (default: all; 'learned' needs the trained model)")
    ap.add_argument("--fidelity-qubits", type=int, default=28)
    ap.add_argument("--no-fidelity", action="store_true")
    ap.add_argument("--cpu-passes", type=int, default=0,
                    help="bound the CPU baseline to the first P fused passes "
                         "(default 0: the whole circuit)")
    ap.add_argument("--cpu-threads", type=int, default=0)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--pmc-calibration", action="store_true",
                    help="only run two state-scaling passes over a 30-qubit "
                         "complex64 state (8 GiB read + 8 GiB written each): "
                         "the known-size reference for HBM counters")
    ap.add_argument("--trajectories", type=int, default=1024,
                    help="size of the trajectory batch reported beside the "
                         "headline (0: skip)")
    ap.add_argument("--pass-times", action="store_true",
                    help="log each pass's median time, qubits and fused "
                         "gates (stderr)")
    ap.add_argument("--no-grid30", action="store_true",
                    help="skip the 30-qubit fusion sweep and its CPU run")
    ap.add_argument("--no-small", action="store_true",
                    help="skip the 20-qubit eager vs captured-graph line")
    args = ap.parse_args()

    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU; --gpus {args.gpus} is not "
              "supported (sharding across GPUs is a design note only).",
              file=sys.stderr)
        sys.exit(2)

    import qsim_amd
    from qsim_amd import circuits
    name, mem, cus = qsim_amd.device_info()
    log(f"device: {name}, {mem / 2**30:.0f} GiB, {cus} CUs")
    if args.pmc_calibration:
        ss = qsim_amd.StateSpace(np.float32)
        st = ss.create(30)
        ss.set_state_uniform(st)
        for _ in range(2):
            ss.multiply(1.0, st)    # ScaleKernel: 16 * 2^30 bytes each
        qsim_amd.synchronize()
        st.free()
        log("pmc calibration: 2 ScaleKernel passes over 2^30 amplitudes")
        return
    text = circuits.grid_circuit(args.qubits, args.cycles, args.seed)
    rows, cols = circuits.grid_shape(args.qubits)
    names = [p for p in args.paths.split(",") if p] or available_paths()
    results = {p: run_path(args, text, p) for p in names}

    fid = {}
    if not args.no_fidelity:
        fid = fidelities(args, names,
                         {p: results[p]["planner_pick"] for p in names
                          if results[p].get("planner_pick")})
        for p in names:
            results[p]["fidelity"] = fid[p]

    def ok(p):
        return not fid or (fid[p]["one_minus_F"] <= 1e-6 and
                           fid[p]["norm_drift"] <= 1e-5)
    eligible = [p for p in names if ok(p)] or names
    # The headline is the learned planner's pick when it meets the bar (it
    # is what a caller gets); otherwise the fastest path that does.
    if "learned" in eligible:
        best = "learned"
    else:
        best = min(eligible, key=lambda p: results[p]["circuit_s"])
    b = results[best]

    cpu = None
    if not args.no_cpu:
        with tempfile.TemporaryDirectory() as tmp:
            cf = os.path.join(tmp, "circuit.txt")
            with open(cf, "w") as f:
                f.write(text)
            try:
                cpu = run_cpu_baseline(args, cf)
            except Exception as e:  # reported, never silently replaced
                log(f"cpu baseline failed: {e!r}")
                cpu = {"value": None, "error": repr(e)}

    grid30 = None
    if not args.no_grid30:
        try:
            grid30 = run_grid30(args)
        except Exception as e:  # reported beside the headline, never hidden
            log(f"30q sweep failed: {e!r}")
            grid30 = {"error": repr(e)}

    traj = None
    if args.trajectories > 0:
        try:
            traj = run_trajectories(args)
        except Exception as e:  # reported beside the headline, never hidden
            log(f"trajectory batch failed: {e!r}")
            traj = {"error": repr(e)}

    ceiling = None
    try:
        ceiling = stream_ceiling(args.qubits)
        b["roofline"]["stream_ceiling"] = ceiling
        b["roofline"]["frac_of_stream_ceiling"] = (
            b["roofline"]["achieved"] / ceiling["achieved"])
    except Exception as e:  # reported beside the headline, never hidden
        log(f"stream ceiling failed: {e!r}")

    small = None
    if not args.no_small:
        try:
            small = run_small_circuit(args)
        except Exception as e:  # reported beside the headline, never hidden
            log(f"small circuit failed: {e!r}")
            small = {"error": repr(e)}

    plain = results.get("plain-fp32-vector")
    out = {
        "metric": METRIC,
        "value": b["circuit_s"],
        "unit": "s/circuit",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": b["circuit_s"] * 1e3,
        "higher_is_better": False,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {
            "workload": (f"{args.qubits}q random grid circuit {rows}x{cols}, "
                         f"{args.cycles} cycles, seed {args.seed}, complex64, "
                         f"path {best}"),
            "num_qubits": args.qubits, "cycles": args.cycles,
            "method": best, "partition": b["partition"],
            "planner_pick": b["planner_pick"],
            "max_fused_size": b["max_fused_size"],
            "tile_qubits": b["tile_qubits"],
            "num_gates": b["num_gates"], "fused_passes": b["passes"],
        },
        "gate_passes_per_s": b["gate_passes_per_s"],
        "hbm_gbps_avg_pass": b["hbm_gbps_avg_pass"],
        "speedup_vs_plain_fp32_k4": (plain["circuit_s"] / b["circuit_s"]
                                     if plain else None),
        "fidelity": fid.get(best),
        "paths": {p: {k: v for k, v in r.items() if k != "roofline"}
                  for p, r in results.items()},
        "roofline": b["roofline"],
        "cpu_baseline": cpu,
        "grid30_fusion_sweep": grid30,
        "trajectory_batch": traj,
        "small_circuit": small,
    }
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
