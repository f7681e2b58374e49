"""Trajectory batches built directly on the C ABI (qsim_hip_traj_*): the
tiled batch (many workgroups a trajectory) against the per-gate kernel (one
workgroup a trajectory) and against FP64 numpy."""

import ctypes

import numpy as np
import pytest
import torch

import qsim_amd
from helpers import random_matrix, to_interleaved

pytestmark = pytest.mark.gpu

OP = np.dtype([("kind", "u4"), ("k", "u4"), ("q", "u4", 4), ("moff", "u4"),
               ("moff2", "u4"), ("r", "f8"), ("cp", "f8"), ("slot", "u4"),
               ("pad", "u4")])
DESC = np.dtype([("num_qubits", "u4"), ("num_pairs", "u4"),
                 ("state_offset", "u8"), ("op_begin", "u8"), ("op_end", "u8"),
                 ("pair_offset", "u4"), ("pad", "u4")])
GATE, CHANNEL, TILE_PASS, KRAUS = 0, 1, 2, 3
TILED = 1


class Batch:
    def __init__(self):
        self.ops, self.mats, self.descs, self.pairs = [], [], [], []
        self.floats = self.slots = 0

    def put(self, m):
        a = to_interleaved(np.asarray(m), np.float32)
        self.mats.append(a)
        self.floats += a.size
        return self.floats - a.size

    def op(self, kind, qs=(), **more):
        o = np.zeros((), OP)
        o["kind"], o["k"] = kind, len(qs)
        o["q"][:len(qs)] = qs
        for name, v in more.items():
            o[name] = v
        self.ops.append(o)

    def gate(self, qs, u):
        self.op(GATE, qs, moff=self.put(u))

    def tile_pass(self, tile, gates):
        mask = sum(1 << q for q in tile)
        self.op(TILE_PASS, moff=0)
        self.ops[-1]["k"] = len(gates)
        self.ops[-1]["q"][:2] = mask & 0xFFFFFFFF, mask >> 32
        for qs, u in gates:
            self.gate(qs, u)

    def channel(self, qs, kraus, r, normalise):
        """kraus: [(qubits, matrix, bound, unitary)]."""
        self.op(CHANNEL, r=r, cp=sum(k[2] for k in kraus), slot=self.slots,
                pad=int(normalise), moff2=len(qs))
        self.ops[-1]["k"] = len(kraus)
        self.ops[-1]["q"][:len(qs)] = qs
        self.slots += 1
        for kq, m, bound, unitary in kraus:
            full = embed(m, kq, qs)
            self.op(KRAUS, kq, moff=self.put(m) if len(kq) else 0,
                    moff2=self.put(full.conj().T @ full), r=bound,
                    pad=int(unitary))

    def trajectory(self, n, build, normalise, pairs):
        begin = len(self.ops)
        build(self)
        self.descs.append((n, len(pairs), 0, begin, len(self.ops),
                           len(self.pairs), int(normalise)))
        self.pairs += pairs

    def prepare(self):
        descs, ops = np.array(self.descs, DESC), np.stack(self.ops).astype(OP)
        mats = np.concatenate(self.mats).astype(np.float32)
        pr = np.asarray(self.pairs, np.uint32).reshape(-1)
        h = ctypes.c_void_p()
        qsim_amd._check(qsim_amd.lib().qsim_hip_traj_prepare(
            descs.ctypes.data, len(descs), ops.ctypes.data, len(ops),
            mats.ctypes.data, mats.size,
            pr.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)),
            len(self.pairs), self.slots, ctypes.byref(h)))
        return h

    def run(self, threads, graph=0, repeats=1):
        lib = qsim_amd.lib()
        h = self.prepare()
        zz = np.zeros(len(self.pairs), np.float64)
        dec = np.zeros(self.slots, np.int32)
        states = [np.zeros(2 << n, np.float32) for n, *_ in self.descs]
        try:
            for _ in range(repeats):
                qsim_amd._check(lib.qsim_hip_traj_run(h, threads, graph))
            qsim_amd._check(lib.qsim_hip_traj_results(
                h, zz.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), len(zz),
                dec.ctypes.data, len(dec)))
            for t, s in enumerate(states):
                qsim_amd._check(lib.qsim_hip_traj_state(h, t, s.ctypes.data))
        finally:
            qsim_amd._check(lib.qsim_hip_traj_free(h))
        return zz, dec, states


def embed(m, kq, qs):
    """A Kraus operator over the channel's qubits."""
    m = np.asarray(m, np.complex128)
    if list(kq) == list(qs):
        return m
    if not len(kq):
        return np.eye(1 << len(qs), dtype=np.complex128)
    return np.kron(np.eye(2), m) if kq[0] == qs[0] else np.kron(m, np.eye(2))


def amplitude_damping(q, gamma):
    k0 = np.diag([1, np.sqrt(1 - gamma)])
    k1 = np.array([[0, np.sqrt(gamma)], [0, 0]])
    return [([q], k0, 1 - gamma, False), ([q], k1, 0.0, False)]


def two_qubit_channel(qs, rng):
    """A unitary operator, an identity, one on a single qubit, and a
    non-unitary pair on both qubits that completes them."""
    u = random_matrix(2, rng)
    a = np.diag([1, 1, 1, np.sqrt(0.5)])
    b = np.zeros((4, 4))
    b[0, 3] = np.sqrt(0.5)
    s = np.sqrt(0.7)
    return [(list(qs), np.sqrt(0.1) * u, 0.1, True),
            ([], np.eye(1), 0.1, True),
            ([qs[1]], np.sqrt(0.1) * np.diag([1, -1]), 0.1, True),
            (list(qs), s * a, 0.7 * 0.5, False),
            (list(qs), s * b, 0.0, False)]


def random_batch(sizes, tile_bits, rng):
    b = Batch()
    for i, n in enumerate(sizes):
        def build(b, n=n, i=i):
            damped = False
            for step in range(3):
                tb = min(tile_bits, n)
                if tb >= 9:
                    low = 4 if n > 4 else 3
                    high = sorted(rng.choice(np.arange(low, n), tb - low,
                                             replace=False).tolist())
                    tile = list(range(low)) + high
                    gates = [(sorted(rng.choice(tile, k, replace=False).tolist()),
                              random_matrix(k, rng))
                             for k in rng.integers(1, 5, size=1 + (i + step) % 6)]
                    b.tile_pass(tile, gates)
                for k in rng.integers(1, min(n, 4) + 1, size=(i + step) % 3):
                    b.gate(sorted(rng.choice(n, k, replace=False).tolist()),
                           random_matrix(k, rng))
                if (i + step) % 2:
                    q = int(rng.integers(n))
                    b.channel([q], amplitude_damping(q, 0.3),
                              1 - 0.3 * rng.uniform(0.05, 0.95), damped)
                    damped = True
                elif i % 3 == 0:
                    qs = sorted(rng.choice(n, 2, replace=False).tolist())
                    b.channel(qs, two_qubit_channel(qs, rng),
                              float(rng.uniform(0.65, 0.999)), damped)
                    damped = True
        pairs = [tuple(rng.choice(n, 2, replace=False).tolist())
                 for _ in range((0, 3, 16, 17, 40)[i % 5])]
        b.trajectory(n, build, True, pairs)
    return b


def apply(psi, n, qs, m):
    """m, row and column bit j on qubit qs[j], over psi in FP64."""
    k = len(qs)
    axes = [n - 1 - q for q in reversed(qs)]
    v = np.moveaxis(psi.reshape((2,) * n), axes, range(k))
    v = (m @ v.reshape(1 << k, -1)).reshape((2,) * n)
    return np.moveaxis(v, range(k), axes).reshape(-1)


def replay(b):
    """The batch's streams in FP64 numpy: pair values, choices, states."""
    mats = np.concatenate(b.mats).astype(np.float64)

    def mat(off, k):
        m = mats[off:off + (2 << 2 * k)].reshape(1 << k, 1 << k, 2)
        return m[..., 0] + 1j * m[..., 1]

    zz, dec, states = [], np.full(b.slots, -1, np.int32), []
    for n, num_pairs, _, begin, end, first_pair, normalise in b.descs:
        psi = np.zeros(1 << n, np.complex128)
        psi[0] = 1
        i = begin
        while i < end:
            o = b.ops[i]
            k = int(o["k"])
            if o["kind"] == GATE:
                psi = apply(psi, n, o["q"][:k].tolist(), mat(int(o["moff"]), k))
            elif o["kind"] == CHANNEL:
                # lib/qtrajectory.h:330-370: the non-unitary operators in
                # turn until the draw falls below the running sum.
                nq = int(o["moff2"])
                norm = np.vdot(psi, psi).real if o["pad"] & 1 else 1.0
                cp, best, at, pick = float(o["cp"]), 0.0, 0, -1
                for j in range(k):
                    c = b.ops[i + 1 + j]
                    if c["pad"] & 1:
                        continue
                    kk = apply(psi, n, o["q"][:nq].tolist(),
                               mat(int(c["moff2"]), nq))
                    prob = np.vdot(psi, kk).real / norm
                    if prob > best:
                        best, at = prob, j
                    cp += prob - float(c["r"])
                    if o["r"] < cp or j == k - 1:
                        pick = j if o["r"] < cp else at
                        break
                dec[o["slot"]] = pick
                if pick >= 0 and b.ops[i + 1 + pick]["k"]:
                    c = b.ops[i + 1 + pick]
                    ck = int(c["k"])
                    psi = apply(psi, n, c["q"][:ck].tolist(),
                                mat(int(c["moff"]), ck))
                psi = psi / np.sqrt(norm)
                i += k
            i += 1
        p = np.abs(psi) ** 2
        idx = np.arange(1 << n)
        for qa, qb in b.pairs[first_pair:first_pair + num_pairs]:
            sign = 1 - 2 * (((idx >> qa) ^ (idx >> qb)) & 1)
            zz.append((p * sign).sum() / p.sum())
        if normalise:
            psi = psi / np.sqrt(p.sum())
        states.append(np.stack([psi.real, psi.imag], 1).reshape(-1))
    return np.array(zz), dec, states


@pytest.mark.parametrize("threads", [256, 1024, TILED])
@pytest.mark.parametrize("tile_bits,sizes", [
    (14, [17, 14, 9, 4]), (13, [15, 13, 11, 10]), (10, [12, 10, 6])])
def test_batch_matches_numpy(tile_bits, sizes, threads):
    b = random_batch(sizes, tile_bits, np.random.default_rng(sum(sizes)))
    zz, dec, states = replay(b)
    zt, dt, st = b.run(threads)
    np.testing.assert_array_equal(dt, dec)
    np.testing.assert_allclose(zt, zz, atol=1e-5, rtol=0)
    for n, x, y in zip(sizes, st, states):
        assert np.linalg.norm(x - y) < 1e-5, n


@pytest.mark.parametrize("tile_bits,sizes", [
    (14, [18, 17, 16, 15, 14, 13, 10, 9, 6, 4]),
    (13, [17, 15, 14, 13, 12, 9, 8]),
    (11, [16, 14, 12, 11, 10]),
    (14, [14, 4]),
    (9, [9, 9, 9])])
def test_tiled_batch_matches_per_gate_kernel(tile_bits, sizes):
    # Uneven sizes, streams of different lengths, one chunk and several per
    # trajectory, gates outside passes, channels of every operator kind.
    # Bars: those of the tiled kernel against qsim's simulator (1e-5).
    b = random_batch(sizes, tile_bits, np.random.default_rng(31 * tile_bits))
    zz, dec, states = b.run(512)
    for graph, repeats in ((0, 1), (1, 3)):
        zt, dt, st = b.run(TILED, graph, repeats)
        np.testing.assert_array_equal(dt, dec)
        np.testing.assert_allclose(zt, zz, atol=1e-5, rtol=0)
        for n, (x, y) in zip(sizes, zip(st, states)):
            assert np.linalg.norm(x - y) < 1e-5, n
            assert abs(np.linalg.norm(x) - 1) < 1e-5


def test_long_chunks_match_per_gate_kernel():
    # Above 24 qubits a chunk has more than 2^14 amplitudes: four rounds of
    # the final sums here, channels on one and two qubits, 17 pairs.
    sizes = [9, 10, 11, 26]
    b = random_batch(sizes, 14, np.random.default_rng(26))
    zz, dec, states = b.run(512)
    zt, dt, st = b.run(TILED)
    np.testing.assert_array_equal(dt, dec)
    np.testing.assert_allclose(zt, zz, atol=1e-5, rtol=0)
    for n, x, y in zip(sizes, st, states):
        assert np.linalg.norm(x - y) < 1e-5, n


def test_batch_memory_follows_its_streams():
    # 8000 gates on 24 qubits: 1024 sweep chunks a gate.  Beyond the state and
    # the operations (64 bytes a gate), a batch takes a few bytes a gate, not
    # a few a chunk, before it is run tiled and after.
    n, gates = 24, 8000
    u = random_matrix(1, np.random.default_rng(3))
    b = Batch()
    moff = b.put(u)

    def build(b):
        for i in range(gates):
            b.op(GATE, [i % n], moff=moff)
    b.trajectory(n, build, False, [(0, n - 1)])
    lib = qsim_amd.lib()
    free0 = torch.cuda.mem_get_info()[0]
    h = b.prepare()
    try:
        limit = (8 << n) + 64 * gates + (16 << 20)
        assert free0 - torch.cuda.mem_get_info()[0] < limit
        qsim_amd._check(lib.qsim_hip_traj_run(h, TILED, 0))
        assert free0 - torch.cuda.mem_get_info()[0] < limit + (16 << 20)
    finally:
        qsim_amd._check(lib.qsim_hip_traj_free(h))
