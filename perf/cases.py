"""The work that programs built on this framework have it do, as cases that
can be timed and compared: every case goes through the public entry points
(qsim_amd.Simulator, StateSpace, PreparedBlock, the gate queue, and the C ABI's
trajectory batch) on states that live on the GPU.

    listed()            the cases, dicts of plain values
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs on the GPU, made from the seed alone
    run(state)          one pass, and its outputs
    work(case)          bytes and flops one pass cannot do without
    exact(case, seed)   the outputs in 64 bits, by torch alone
"""

import ctypes
import math
import random

import numpy as np
import torch

import qsim_amd
from qsim_amd import circuits
from qsim_amd.trajectories import grid_pairs


def listed():
    return [
        # A small circuit gate by gate from |0>, as interactive use and the
        # tests have it: 1- and 2-qubit gates, bound by calls and launches.
        {"name": "circuit_12q", "kind": "circuit", "n": 12, "cycles": 4},
        # The 20-qubit workload after fusion to k <= 4 qubits.
        {"name": "fused_20q", "kind": "gates", "n": 20, "bits": 32,
         "kmin": 1, "kmax": 4, "count": 24},
        # A large fused circuit, every size of fused gate, any qubits.
        {"name": "fused_29q", "kind": "gates", "n": 29, "bits": 32,
         "kmin": 1, "kmax": 4, "count": 12},
        # Wider fusion (max_fused_size 5 and 6) with the default arithmetic.
        {"name": "fused_wide_28q", "kind": "gates", "n": 28, "bits": 32,
         "kmin": 5, "kmax": 6, "count": 6},
        # Double precision, fused gates of every size.
        {"name": "fused_double_27q", "kind": "gates", "n": 27, "bits": 64,
         "kmin": 1, "kmax": 5, "count": 10},
        # Controlled gates: 1..3 controls, high and low.
        {"name": "controlled_27q", "kind": "controlled", "n": 27, "bits": 32,
         "count": 12},
        # The largest: cache-blocked passes of the 32-qubit workload,
        # prepared once as a driver does.
        {"name": "blocked_32q", "kind": "blocked", "n": 32, "tile": 14,
         "low": 4, "ops": 5, "passes": 3},
        # The same through the gate queue, as the learned fuser's gates
        # reach it: passes are built as the gates come in.
        {"name": "queue_25q", "kind": "queue", "n": 25, "tile": 14, "low": 4,
         "ops": 6, "passes": 4},
        # An energy (1-, 2- and 4-qubit terms), the norm, and the overlap
        # with another state.
        {"name": "observables_27q", "kind": "observables", "n": 27,
         "bits": 32, "terms": 9},
        # Bitstrings of a final state.
        {"name": "sample_28q", "kind": "sample", "n": 28, "samples": 20000},
        # A measurement in mid-circuit: outcome and collapsed state.
        {"name": "measure_26q", "kind": "measure", "n": 26, "bits": 32,
         "qubits": 2},
        # A batch of noisy trajectories of uneven sizes, one launch.
        {"name": "trajectories", "kind": "trajectories", "n": 16, "step": 2,
         "count": 300, "tile": 14, "low": 4, "passes": 4, "ops": 5},
    ]


def draw(rng):
    kind = rng.choice(["circuit", "gates", "gates", "gates", "controlled",
                       "blocked", "blocked", "queue", "observables", "sample",
                       "measure", "trajectories"])
    if kind == "circuit":
        return {"kind": kind, "n": rng.randint(10, 18),
                "cycles": rng.randint(2, 8)}
    if kind == "gates":
        bits = rng.choice([32, 32, 64])
        kmin = rng.choice([1, 1, 2, 3, 4, 5])
        return {"kind": kind, "n": rng.randint(14, 29 if bits == 32 else 27),
                "bits": bits, "kmin": kmin, "kmax": rng.randint(kmin, 6),
                "count": rng.randint(3, 10)}
    if kind == "controlled":
        return {"kind": kind, "n": rng.randint(14, 29),
                "bits": rng.choice([32, 32, 64]), "count": rng.randint(4, 12)}
    if kind == "blocked":
        tile = rng.choice([11, 12, 13, 13, 14, 14, 14])
        return {"kind": kind, "n": rng.randint(18, 31), "tile": tile,
                "low": rng.randint(3, 6), "ops": rng.randint(1, 7),
                "passes": rng.randint(1, 4)}
    if kind == "queue":
        return {"kind": kind, "n": rng.randint(18, 28),
                "tile": rng.choice([13, 14]), "low": rng.choice([4, 5]),
                "ops": rng.randint(2, 7), "passes": rng.randint(2, 5)}
    if kind == "observables":
        return {"kind": kind, "n": rng.randint(16, 29),
                "bits": rng.choice([32, 32, 64]), "terms": rng.randint(3, 12)}
    if kind == "sample":
        return {"kind": kind, "n": rng.randint(12, 30),
                "samples": int(round(10 ** rng.uniform(2, 4.7)))}
    if kind == "measure":
        return {"kind": kind, "n": rng.randint(14, 28),
                "bits": rng.choice([32, 32, 64]), "qubits": rng.randint(1, 6)}
    return {"kind": kind, "n": rng.randint(14, 17), "step": rng.randint(0, 2),
            "count": rng.randint(40, 300), "tile": rng.choice([13, 14]),
            "low": rng.choice([4, 5]), "passes": rng.randint(2, 5),
            "ops": rng.randint(2, 7)}


# ---- inputs ----------------------------------------------------------------


def _rng(case, seed):
    return random.Random(1_000_003 * int(seed) + case["n"])


def _amplitudes(n, bits, seed):
    """A normalised state with the amplitudes of a random circuit's output
    (complex Gaussian), interleaved, on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    dtype = torch.float32 if bits == 32 else torch.float64
    t = torch.empty(2 << n, dtype=dtype, device="cuda")
    t.normal_(generator=gen)
    norm = torch.linalg.vector_norm(t, dtype=torch.float64).item()
    return t.mul_(1.0 / norm)


def _wrap(t, n):
    fp = np.float32 if t.dtype == torch.float32 else np.float64
    return qsim_amd.State(n, fp, ptr=t.data_ptr(), owner=False)


def _unitary(rng, k):
    g = np.random.default_rng(rng.getrandbits(63))
    d = 1 << k
    q, r = np.linalg.qr(g.normal(size=(d, d)) + 1j * g.normal(size=(d, d)))
    ph = np.diagonal(r)
    return q * (ph / np.abs(ph))


def _hermitian(rng, k):
    """A Hermitian term with spectral norm 1: U diag(+-1) U^dagger."""
    u = _unitary(rng, k)
    s = np.array([1.0 if i % 2 else -1.0 for i in range(1 << k)])
    return (u * s) @ u.conj().T


def _matrix(u, bits):
    """The interleaved matrix a caller passes, in the state's precision."""
    return np.ascontiguousarray(u.astype(
        np.complex64 if bits == 32 else np.complex128)).view(
            np.float32 if bits == 32 else np.float64).reshape(-1)


def _qubits(rng, n, k):
    return sorted(rng.sample(range(n), k))


_S = math.sqrt(0.5)
_GATES_1Q = {
    "x_1_2": np.array([[0.5 + 0.5j, 0.5 - 0.5j], [0.5 - 0.5j, 0.5 + 0.5j]]),
    "y_1_2": np.array([[0.5 + 0.5j, -0.5 - 0.5j], [0.5 + 0.5j, 0.5 + 0.5j]]),
    "hz_1_2": np.array([[0.5 + 0.5j, -1j * _S], [_S, 0.5 + 0.5j]]),
}


def _fsim(theta, phi):
    c, s = math.cos(theta), -1j * math.sin(theta)
    return np.array([[1, 0, 0, 0], [0, c, s, 0], [0, s, c, 0],
                     [0, 0, 0, np.exp(-1j * phi)]])


def _circuit_gates(case, seed):
    rows, cols = circuits.grid_shape(case["n"])
    _, ops = circuits.grid_circuit_ops(rows, cols, case["cycles"], int(seed))
    return [(list(q), _GATES_1Q[name] if len(q) == 1 else _fsim(*prm))
            for _, name, q, prm in ops]


def _plain_gates(case, seed):
    rng = _rng(case, seed)
    span = case["kmax"] - case["kmin"] + 1
    gates = []
    for i in range(case["count"]):
        k = case["kmin"] + i % span
        gates.append((_qubits(rng, case["n"], k), _unitary(rng, k)))
    return gates


def _controlled_gates(case, seed):
    """(targets, controls, control values, matrix): 1- and 2-qubit gates with
    1..3 controls."""
    rng = _rng(case, seed)
    gates = []
    for i in range(case["count"]):
        k, c = 1 + i % 2, 1 + i % 3
        both = rng.sample(range(case["n"]), k + c)
        gates.append((sorted(both[:k]), sorted(both[k:]), rng.getrandbits(c),
                      _unitary(rng, k)))
    return gates


def _blocked_passes(case, seed):
    """[(tile qubits, [(qubits, matrix), ...]), ...]: a planner's passes, the
    `low` lowest qubits and chosen higher ones, gates fused to 3 or 4 qubits."""
    rng = _rng(case, seed)
    passes = []
    for _ in range(case["passes"]):
        high = rng.sample(range(case["low"], case["n"]),
                          case["tile"] - case["low"])
        tile = list(range(case["low"])) + sorted(high)
        gates = []
        for i in range(case["ops"]):
            k = 3 if i % 5 == 4 else 4
            gates.append((sorted(rng.sample(tile, k)), _unitary(rng, k)))
        passes.append((tile, gates))
    return passes


def _terms(case, seed):
    rng = _rng(case, seed)
    terms = []
    for i in range(case["terms"]):
        k = (1, 2, 4)[i % 3]
        terms.append((_qubits(rng, case["n"], k), _hermitian(rng, k)))
    return terms


def _measured(case, seed):
    rng = _rng(case, seed)
    return _qubits(rng, case["n"], case["qubits"]), rng.uniform(0.02, 0.98)


# ---- trajectory batches (include/qsim_hip.h, qsim_hip_traj_*) --------------

_OP = np.dtype([("kind", "u4"), ("k", "u4"), ("q", "u4", 4), ("moff", "u4"),
                ("moff2", "u4"), ("r", "f8"), ("cp", "f8"), ("slot", "u4"),
                ("pad", "u4")])
_DESC = np.dtype([("num_qubits", "u4"), ("num_pairs", "u4"),
                  ("state_offset", "u8"), ("op_begin", "u8"),
                  ("op_end", "u8"), ("pair_offset", "u4"), ("pad", "u4")])
_GATE, _CHANNEL, _TILE_PASS, _KRAUS = 0, 1, 2, 3
_GAMMA = 0.05  # amplitude damping


def _trajectory_plans(case, seed):
    """Per trajectory (largest first) its steps: ("pass", tile, gates) and
    ("damp", qubit, draw), matrices FP32.  Trajectories of one size share
    their circuit; each has a Pauli error folded into one gate (a
    depolarising channel the host decided) and amplitude-damping channels
    whose draw only the state decides."""
    rng = _rng(case, seed)
    sizes = [case["n"] + case["step"] * i for i in (2, 1, 0)]
    base = {}
    for n in sorted(set(sizes), reverse=True):
        tb = min(case["tile"], n)
        steps = []
        for _ in range(case["passes"]):
            tile = list(range(case["low"])) + sorted(rng.sample(
                range(case["low"], n), tb - case["low"]))
            steps.append((tile, [
                (sorted(rng.sample(tile, 4)),
                 _unitary(rng, 4).astype(np.complex64))
                for _ in range(case["ops"])]))
        base[n] = steps
    paulis = [np.array([[0, 1], [1, 0]]), np.array([[0, -1j], [1j, 0]]),
              np.array([[1, 0], [0, -1]])]
    plans = []
    for t in range(case["count"]):
        n = sizes[t * 3 // case["count"]]
        steps = []
        hit = rng.randrange(case["passes"]), rng.randrange(case["ops"])
        err = paulis[rng.randrange(3)]
        for p, (tile, gates) in enumerate(base[n]):
            gates = list(gates)
            if p == hit[0]:
                q, u = gates[hit[1]]
                full = np.kron(np.eye(8), err)  # on the lowest gate qubit
                gates[hit[1]] = (q, (full @ u).astype(np.complex64))
            steps.append(("pass", tile, gates))
            if p % 2 == t % 2:
                steps.append(("damp", rng.randrange(n),
                              1.0 - _GAMMA * rng.uniform(0.02, 0.98)))
        plans.append((n, steps))
    return plans


def _damping():
    k0 = np.diag([1.0, math.sqrt(1 - _GAMMA)]).astype(np.complex64)
    k1 = np.array([[0, math.sqrt(_GAMMA)], [0, 0]], np.complex64)
    return [(k0, 1.0 - _GAMMA), (k1, 0.0)]


class _Batch:
    """A prepared trajectory batch; owns its handle."""

    def __init__(self, plans):
        mats, offs, total = [], {}, 0

        def put(m):
            nonlocal total
            key = m.tobytes()
            if key not in offs:
                offs[key] = total
                mats.append(_matrix(m, 32))
                total += mats[-1].size
            return offs[key]

        def gate(kind, qs, m, **more):
            o = np.zeros((), _OP)
            o["kind"], o["k"] = kind, len(qs)
            o["q"][:len(qs)] = qs
            o["moff"] = put(m)
            for name, v in more.items():
                o[name] = v
            return o

        ops, descs, pairs, slots = [], [], [], 0
        kraus = _damping()
        for n, steps in plans:
            begin = len(ops)
            damped = False
            for step in steps:
                if step[0] == "pass":
                    _, tile, gates = step
                    o = np.zeros((), _OP)
                    mask = sum(1 << q for q in tile)
                    o["kind"], o["k"] = _TILE_PASS, len(gates)
                    o["q"][:2] = mask & 0xFFFFFFFF, mask >> 32
                    ops.append(o)
                    ops += [gate(_GATE, q, m) for q, m in gates]
                else:
                    _, q, r = step
                    o = np.zeros((), _OP)
                    o["kind"], o["k"], o["moff2"] = _CHANNEL, len(kraus), 1
                    o["q"][0], o["slot"] = q, slots
                    o["r"], o["cp"] = r, sum(b for _, b in kraus)
                    o["pad"] = 1 if damped else 0
                    ops.append(o)
                    ops += [gate(_KRAUS, [q], m, r=b,
                                 moff2=put(m.conj().T @ m)) for m, b in kraus]
                    slots += 1
                    damped = True
            zz = grid_pairs(n)
            descs.append((n, len(zz), 0, begin, len(ops), len(pairs),
                          1 if damped else 0))
            pairs += zz
        self.num_pairs, self.slots = len(pairs), slots
        ops = np.stack(ops).astype(_OP)
        descs = np.array(descs, _DESC)
        mats = np.concatenate(mats).astype(np.float32)
        pr = np.asarray(pairs, np.uint32).reshape(-1)
        h = ctypes.c_void_p()
        qsim_amd._check(qsim_amd.lib().qsim_hip_traj_prepare(
            descs.ctypes.data, len(descs), ops.ctypes.data, len(ops),
            mats.ctypes.data, mats.size,
            pr.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)),
            self.num_pairs, slots, ctypes.byref(h)))
        self.h = h

    def run(self):
        """<Z_a Z_b> of every trajectory's pairs and the Kraus choices."""
        lib = qsim_amd.lib()
        qsim_amd._check(lib.qsim_hip_traj_run(self.h, 1, 0))
        zz = np.zeros(self.num_pairs, np.float64)
        dec = np.zeros(self.slots, np.int32)
        qsim_amd._check(lib.qsim_hip_traj_results(
            self.h, zz.ctypes.data_as(ctypes.POINTER(ctypes.c_double)),
            self.num_pairs, dec.ctypes.data, self.slots))
        return zz, dec

    def __del__(self):
        if getattr(self, "h", None):
            qsim_amd.lib().qsim_hip_traj_free(self.h)
            self.h = None


# ---- prepare and run -------------------------------------------------------


def prepare(case, seed):
    kind, n = case["kind"], case["n"]
    bits = case.get("bits", 32)
    s = {"case": case, "sim": qsim_amd.Simulator(),
         "ss": qsim_amd.StateSpace(np.float32 if bits == 32 else np.float64)}
    if kind == "trajectories":
        s["batch"] = _Batch(_trajectory_plans(case, seed))
        return s
    if kind == "circuit":
        s["amps"] = torch.zeros(2 << n, dtype=torch.float32, device="cuda")
        s["gates"] = [(q, _matrix(u, 32))
                      for q, u in _circuit_gates(case, seed)]
    else:
        s["amps"] = _amplitudes(n, bits, seed)
    s["state"] = _wrap(s["amps"], n)
    if kind == "gates":
        s["gates"] = [(q, _matrix(u, bits)) for q, u in _plain_gates(case, seed)]
    elif kind == "controlled":
        s["gates"] = [(q, c, v, _matrix(u, bits))
                      for q, c, v, u in _controlled_gates(case, seed)]
    elif kind == "blocked":
        s["passes"] = [
            s["sim"].prepare_gate_block(
                n, tile, [(q, _matrix(u, 64)) for q, u in gates])
            for tile, gates in _blocked_passes(case, seed)]
    elif kind == "queue":
        s["gates"] = [(q, _matrix(u, 32))
                      for _, gates in _blocked_passes(case, seed)
                      for q, u in gates]
    elif kind == "observables":
        s["terms"] = [(q, _matrix(u, bits)) for q, u in _terms(case, seed)]
        s["other_amps"] = _amplitudes(n, bits, seed + 500_000)
        s["other"] = _wrap(s["other_amps"], n)
    elif kind == "sample":
        s["seed"] = int(seed) & 0x7FFFFFFF
    elif kind == "measure":
        s["qubits"], s["u"] = _measured(case, seed)
    # The inputs are written on torch's stream, the default one, which is the
    # library's too.
    return s


def run(s):
    case, sim, ss = s["case"], s["sim"], s["ss"]
    kind = case["kind"]
    if kind == "trajectories":
        return s["batch"].run()
    st = s["state"]
    if kind == "circuit":
        ss.set_state_zero(st)
        for q, m in s["gates"]:
            sim.apply_gate(q, m, st)
        return s["amps"]
    if kind == "gates":
        for q, m in s["gates"]:
            sim.apply_gate(q, m, st)
        return s["amps"]
    if kind == "controlled":
        for q, c, v, m in s["gates"]:
            sim.apply_controlled_gate(q, c, v, m, st)
        return s["amps"]
    if kind == "blocked":
        for p in s["passes"]:
            p.run(st)
        return s["amps"]
    if kind == "queue":
        qsim_amd.set_gate_queue(case["tile"], case["low"])
        for q, m in s["gates"]:
            sim.apply_gate(q, m, st)
        qsim_amd.flush()
        qsim_amd.set_gate_queue(0)
        return s["amps"]
    if kind == "observables":
        vals = [sim.expectation_value(q, m, st) for q, m in s["terms"]]
        vals.append(ss.inner_product(s["other"], st))
        return {"energy": np.array([[v.real, v.imag] for v in vals]),
                "norm": ss.norm(st)}
    if kind == "sample":
        # Indices below 2^63: the signed view has the same values.
        return ss.sample(st, case["samples"], s["seed"]).view(np.int64)
    mask, bits = ss.measure(s["qubits"], lambda norm: s["u"] * norm, st)
    return {"bits": bits, "state": s["amps"]}


# ---- what a pass cannot do without -----------------------------------------


def work(case):
    kind, n = case["kind"], case["n"]
    amp = 8 if case.get("bits", 32) == 32 else 16
    size = float(1 << n)
    if kind == "circuit":
        gates = _circuit_gates(case, 0)
        return {"bytes": size * amp * (1 + 2 * len(gates)),
                "flops": sum(8.0 * (1 << len(q)) * size for q, _ in gates)}
    if kind == "gates":
        span = case["kmax"] - case["kmin"] + 1
        ks = [case["kmin"] + i % span for i in range(case["count"])]
        return {"bytes": 2 * amp * size * len(ks),
                "flops": sum(8.0 * (1 << k) * size for k in ks)}
    if kind == "controlled":
        touched = [(1 + i % 2, size / (1 << (1 + i % 3)))
                   for i in range(case["count"])]
        return {"bytes": sum(2.0 * amp * a for _, a in touched),
                "flops": sum(8.0 * (1 << k) * a for k, a in touched)}
    if kind in ("blocked", "queue"):
        return {"bytes": 2.0 * amp * size * case["passes"],
                "flops": 8.0 * 16 * size * case["ops"] * case["passes"]}
    if kind == "observables":
        ks = [(1, 2, 4)[i % 3] for i in range(case["terms"])]
        return {"bytes": amp * size * (len(ks) + 3),
                "flops": sum((8.0 * (1 << k) + 8) * size for k in ks)
                + 12 * size}
    if kind == "sample":
        return {"bytes": amp * size + 8.0 * case["samples"],
                "flops": 4 * size}
    if kind == "measure":
        return {"bytes": 2.0 * amp * size, "flops": 6 * size}
    byt = flo = 0.0
    for t in range(case["count"]):
        m = float(1 << (case["n"] + case["step"] * (2 - t * 3 // case["count"])))
        # Every tile pass streams the state once; the pairs read it once.
        byt += 16 * m * case["passes"] + 8 * m
        flo += 8 * 16 * m * case["ops"] * case["passes"]
    return {"bytes": byt, "flops": flo}


# ---- 64 bits ---------------------------------------------------------------


def _split(psi, n, qubits):
    """psi viewed with a dimension of its own for each of `qubits`; the view
    and {qubit: dimension}."""
    shape, where, top = [], {}, n
    for q in sorted(qubits, reverse=True):
        shape.append(1 << (top - q - 1))
        where[q] = len(shape)
        shape.append(2)
        top = q
    shape.append(1 << top)
    return psi.view(shape), where


def _groups(psi, n, qs, cqs=(), cvals=0, most=26):
    """Views of psi, targets first (highest qubit first), that together hold
    every amplitude the gate touches, in pieces of at most 2^most."""
    free = [q for q in range(n - 1, -1, -1) if q not in qs and q not in cqs]
    cut = free[:max(0, n - len(cqs) - most)]
    v, where = _split(psi, n, list(qs) + list(cqs) + cut)
    for piece in range(1 << len(cut)):
        idx = [slice(None)] * v.dim()
        for i, q in enumerate(cut):
            idx[where[q]] = (piece >> i) & 1
        for i, q in enumerate(cqs):
            idx[where[q]] = (cvals >> i) & 1
        gone = {where[q] for q in list(cqs) + cut}
        left = [d for d in range(v.dim()) if d not in gone]
        first = [left.index(where[q]) for q in sorted(qs, reverse=True)]
        rest = [d for d in range(len(left)) if d not in first]
        yield v[tuple(idx)].permute(first + rest)


def _rounded(u, bits):
    """The matrix as passed to the call, in 64 bits."""
    m = u.astype(np.complex64) if bits == 32 else u
    return torch.from_numpy(m.astype(np.complex128)).cuda()


def _apply(psi, n, qs, u, cqs=(), cvals=0):
    d = 1 << len(qs)
    for w in _groups(psi, n, qs, cqs, cvals):
        w.copy_((u @ w.reshape(d, -1)).reshape(w.shape))


def _expect(psi, n, qs, u):
    d, total = 1 << len(qs), 0j
    for w in _groups(psi, n, qs):
        g = w.reshape(d, -1)
        total += torch.sum(g.conj() * (u @ g)).item()
    return total


def _psi64(case, seed, bits):
    t = _amplitudes(case["n"], bits, seed)
    return torch.view_as_complex(t.double().view(-1, 2))


def _real(psi):
    return torch.view_as_real(psi).reshape(-1)


def _exact_trajectory(n, steps):
    psi = torch.zeros(1 << n, dtype=torch.complex128, device="cuda")
    psi[0] = 1
    kraus = _damping()
    for step in steps:
        if step[0] == "pass":
            for q, m in step[2]:
                _apply(psi, n, q, _rounded(m, 32))
            continue
        _, q, r = step
        v, where = _split(psi, n, [q])
        p = v.abs().square().sum(dim=(0, 2))
        p0, p1 = (p / p.sum()).tolist()
        keep = p0 * abs(kraus[0][0][0, 0]) ** 2 + p1 * abs(kraus[0][0][1, 1]) ** 2
        pick = 0 if r < keep else 1
        _apply(psi, n, [q], _rounded(kraus[pick][0], 32))
    prob = psi.abs().square()
    prob = prob / prob.sum()
    out = []
    for a, b in grid_pairs(n):
        v, where = _split(prob, n, [a, b])
        m = v.sum(dim=[d for d in range(v.dim()) if d not in where.values()])
        out.append(m[0, 0] + m[1, 1] - m[0, 1] - m[1, 0])
    return torch.stack(out)


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    bits = case.get("bits", 32)
    if kind == "sample":
        return None  # whole numbers only
    if kind == "trajectories":
        zz = [_exact_trajectory(n, steps)
              for n, steps in _trajectory_plans(case, seed)]
        return torch.cat(zz), None
    if kind == "circuit":
        psi = torch.zeros(1 << n, dtype=torch.complex128, device="cuda")
        psi[0] = 1
        for q, u in _circuit_gates(case, seed):
            _apply(psi, n, q, _rounded(u, 32))
        return _real(psi)
    psi = _psi64(case, seed, bits)
    if kind == "gates":
        for q, u in _plain_gates(case, seed):
            _apply(psi, n, q, _rounded(u, bits))
    elif kind == "controlled":
        for q, c, v, u in _controlled_gates(case, seed):
            _apply(psi, n, q, _rounded(u, bits), c, v)
    elif kind in ("blocked", "queue"):
        for _, gates in _blocked_passes(case, seed):
            for q, u in gates:
                _apply(psi, n, q, _rounded(u, 64 if kind == "blocked" else 32))
    elif kind == "observables":
        vals = [_expect(psi, n, q, _rounded(u, bits))
                for q, u in _terms(case, seed)]
        vals.append(torch.vdot(_psi64(case, seed + 500_000, bits), psi).item())
        return {"energy": np.array([[v.real, v.imag] for v in vals]),
                "norm": float(torch.linalg.vector_norm(psi).item() ** 2)}
    else:
        qubits, u = _measured(case, seed)
        cum = torch.cumsum(psi.abs().square(), 0)
        r = u * cum[-1].item()
        k = int(torch.searchsorted(cum, r, right=True).item())
        mask = sum(1 << q for q in qubits)
        idx = torch.arange(1 << n, device="cuda")
        psi = torch.where((idx & mask) == (k & mask), psi, 0)
        psi = psi / torch.linalg.vector_norm(psi)
        return {"bits": None, "state": _real(psi)}
    return _real(psi)
