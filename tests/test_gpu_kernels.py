"""Parity of the HIP kernels (through the C ABI) with the CPU oracle.

Bar: complex64 results within 1e-6 relative L2 (per pass) / 1e-5 (whole
circuits) of the oracle's FP32 result, complex128 within 1e-12; sampled
bitstrings and measured bits identical for identical draws.
"""

import threading
import time

import numpy as np
import pytest

import oracle
import qsim_amd
from helpers import (dense_gate, expectation2_circuit, from_interleaved,
                     gate_op, known_answers, pauli_string_matrix,
                     random_matrix, random_state, reference_runs, rel_l2,
                     to_interleaved)
from qsim_amd import circuits

pytestmark = pytest.mark.gpu

DTYPES = [np.float32, np.float64]
TOL = {np.float32: 1e-6, np.float64: 1e-12}


@pytest.fixture(scope="module")
def ss32():
    return qsim_amd.StateSpace(np.float32)


@pytest.fixture(scope="module")
def sim():
    return qsim_amd.Simulator()


def upload(a, n, dtype):
    st = qsim_amd.State(n, dtype)
    st.from_numpy(a)
    return st


def test_device_is_gfx950():
    name, mem, cus = qsim_amd.device_info()
    print("device:", name, mem, cus, flush=True)
    assert "gfx950" in name


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("test", ["TestApplyGate1", "TestApplyGate2",
                                  "TestApplyGate3", "TestApplyGate5"])
def test_known_answer_apply_gate(test, dtype, sim):
    t = known_answers()["apply_gate"][test]
    n = t["num_qubits"]
    ss = qsim_amd.StateSpace(dtype)
    st = ss.create(n)
    ss.set_state_zero(st)
    checks = 0
    for step in t["steps"]:
        if "apply" in step:
            for spec in step["apply"]:
                qs, m, cqs, cmask = gate_op(spec, dtype)
                sim.apply_controlled_gate(qs, cqs, cmask, m, st)
        else:
            i, re, im = step["check"]
            a = ss.get_ampl(st, i)
            assert abs(a.real - re) < 1e-6 and abs(a.imag - im) < 1e-6
            checks += 1
    assert checks > 0
    assert abs(ss.norm(st) - 1) < 1e-6


@pytest.mark.parametrize("dtype", DTYPES)
def test_known_answer_controlled_circuit(dtype, sim):
    t = known_answers()["controlled_circuit"]
    n = t["num_qubits"]
    ss = qsim_amd.StateSpace(dtype)
    st = ss.create(n)
    ss.set_state_zero(st)
    for spec in t["gates"]:
        qs, m, cqs, cmask = gate_op(spec, dtype)
        sim.apply_controlled_gate(qs, cqs, cmask, m, st)
    s = st.to_numpy()
    exp = np.array(t["expected"])
    got = np.stack([s[0:2 * len(exp):2], s[1:2 * len(exp):2]], axis=1)
    assert np.max(np.abs(got - exp)) < 1e-6
    # Same gates twice give bit-identical states (the fixture's determinism
    # check, tests/simulator_testfixture.h:739-765).
    st2 = ss.create(n)
    ss.set_state_zero(st2)
    for spec in t["gates"]:
        qs, m, cqs, cmask = gate_op(spec, dtype)
        sim.apply_controlled_gate(qs, cqs, cmask, m, st2)
    np.testing.assert_array_equal(st2.to_numpy(), s)


@pytest.mark.parametrize("dtype", DTYPES)
def test_multi_qubit_gates_closed_form(dtype, sim):
    # tests/simulator_testfixture.h:1146-1213 up to 10 + log2(64) qubits.
    ss = qsim_amd.StateSpace(dtype)
    for n in range(2, 17):
        st = ss.create(n)
        size = 1 << n
        inorm = np.sqrt(1.0 / size)
        for q in range(1, min(6, n - 1) + 1):
            size1 = 1 << q
            size2 = size1 * size1
            m = np.arange(1, 2 * size2 + 1, dtype=dtype)
            for k in range(0, n - q + 1):
                ss.set_state_uniform(st)
                sim.apply_gate(list(range(k, k + q)), m, st)
                s = st.to_numpy()
                j = (np.arange(size) >> k) & (size1 - 1)
                er = size2 * (1 + 2 * j) * inorm
                ei = er + size1 * inorm
                assert np.max(np.abs(s[0::2] / er - 1)) < 1e-6, (n, q, k)
                assert np.max(np.abs(s[1::2] / ei - 1)) < 1e-6, (n, q, k)


def _target_sets(n, k, rng):
    """Low, high, mixed and random target sets (exercises both kernels)."""
    sets = set()
    if k == 0:
        return [[]]
    sets.add(tuple(range(k)))
    sets.add(tuple(range(n - k, n)))
    for _ in range(4):
        sets.add(tuple(sorted(rng.choice(n, size=k, replace=False).tolist())))
    return [list(s) for s in sets]


@pytest.mark.parametrize("dtype", DTYPES)
def test_apply_gate_vs_oracle(dtype, sim):
    rng = np.random.default_rng(11)
    for n in list(range(1, 13)) + [14, 17, 20]:
        for k in range(0, min(n, 6) + 1):
            for qs in _target_sets(n, k, rng):
                u = random_matrix(k, rng, unitary=bool(rng.integers(2)))
                m = to_interleaved(u, dtype)
                s = random_state(n, rng, dtype)
                st = upload(s, n, dtype)
                sim.apply_gate(qs, m, st)
                oracle.apply_gate(n, s, qs, m)
                err = rel_l2(st.to_numpy(), s)
                assert err < TOL[dtype], (n, k, qs, err)


@pytest.mark.parametrize("dtype", DTYPES)
def test_apply_gate_f64_matrix_on_f32_state(dtype, sim):
    # Matrices may arrive in FP64 (host-built fused matrices).
    rng = np.random.default_rng(12)
    n = 12
    for k in range(1, 7):
        qs = sorted(rng.choice(n, size=k, replace=False).tolist())
        u = random_matrix(k, rng)
        s = random_state(n, rng, np.float32)
        st = upload(s, n, np.float32)
        sim.apply_gate(qs, to_interleaved(u, np.float64), st)
        oracle.apply_gate(n, s, qs, to_interleaved(u, np.float32))
        assert rel_l2(st.to_numpy(), s) < 1e-6


@pytest.mark.parametrize("dtype", DTYPES)
def test_controlled_gate_vs_oracle(dtype, sim):
    rng = np.random.default_rng(13)
    for n in (2, 3, 5, 7, 9, 12, 16, 19):
        for _ in range(12):
            k = int(rng.integers(0, min(4, n - 1) + 1))
            nc = int(rng.integers(1, min(n - k, 5) + 1))
            perm = rng.permutation(n)
            qs = sorted(perm[:k].tolist())
            cqs = sorted(perm[k:k + nc].tolist())
            cvals = int(rng.integers(0, 1 << nc))
            u = random_matrix(k, rng)
            m = to_interleaved(u, dtype)
            s = random_state(n, rng, dtype)
            st = upload(s, n, dtype)
            sim.apply_controlled_gate(qs, cqs, cvals, m, st)
            oracle.apply_controlled_gate(n, s, qs, cqs, cvals, m)
            err = rel_l2(st.to_numpy(), s)
            assert err < TOL[dtype], (n, qs, cqs, cvals, err)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("controls", [(), (0,), (1, 2), (2,), (3,), (5,),
                                      (0, 4), (2, 5, 7), (1, 3, 4, 5, 9)])
def test_lane_kernel_edges(dtype, controls, sim):
    # The smallest state the lane kernel takes (6 + k + controls it skips),
    # one qubit less (the tile kernel) and one more, targets packed at the
    # bottom, at the top and alternating; amplitudes outside the controls'
    # subspace keep their bits.
    rng = np.random.default_rng(77 + len(controls))
    for k in range(0, 5):
        for n in range(5 + k + len(controls), 8 + k + len(controls)):
            free = [q for q in range(n) if q not in controls]
            if len(free) < k or any(c >= n for c in controls):
                continue
            for qs in {tuple(free[:k]), tuple(free[len(free) - k:]),
                       tuple(free[::2][:k])}:
                qs = list(qs)
                vals = int(rng.integers(0, 1 << len(controls)))
                m = to_interleaved(random_matrix(k, rng), dtype)
                s = random_state(n, rng, dtype)
                st = upload(s, n, dtype)
                sim.apply_controlled_gate(qs, list(controls), vals, m, st)
                got = st.to_numpy()
                want = s.copy()
                oracle.apply_controlled_gate(n, want, qs, list(controls), vals,
                                             m)
                assert rel_l2(got, want) < TOL[dtype], (n, qs)
                idx = np.arange(1 << n)
                out = np.zeros(1 << n, bool)
                for i, c in enumerate(controls):
                    out |= ((idx >> c) & 1) != ((vals >> i) & 1)
                np.testing.assert_array_equal(got.reshape(-1, 2)[out],
                                              s.reshape(-1, 2)[out])


@pytest.mark.parametrize("dtype,n,qs,controls", [
    (np.float32, 23, [19, 20, 21, 22], []),
    (np.float32, 24, [19, 21, 22, 23], []),
    (np.float64, 22, [18, 19, 20, 21], []),
    (np.float64, 23, [18, 20, 21, 22], [5]),
    (np.float32, 17, [9, 16], [1]),
    (np.float32, 18, [16, 17], [0, 2]),
    (np.float32, 20, [7, 18], [1, 9])])
def test_lane_kernel_far_members(dtype, n, qs, controls, sim):
    # Workgroups in runs of 32 per XCD: members 4 MiB apart, and two targets
    # with a control below qubit 3, at the smallest grids (a multiple of 256
    # workgroups, and one below it).
    rng = np.random.default_rng(n)
    m = to_interleaved(random_matrix(len(qs), rng), dtype)
    s = random_state(n, rng, dtype)
    st = upload(s, n, dtype)
    cvals = (1 << len(controls)) - 1
    sim.apply_controlled_gate(qs, controls, cvals, m, st)
    oracle.apply_controlled_gate(n, s, qs, controls, cvals, m)
    assert rel_l2(st.to_numpy(), s) < TOL[dtype]


@pytest.mark.parametrize("qs,controls", [([16, 27], [1]), ([17, 24], [0, 2]),
                                         ([13, 24], [2]), ([14, 27], [2, 20]),
                                         ([14, 27], [2, 12])])
def test_two_far_targets_with_a_low_control(qs, controls, sim, ss32):
    # 28 qubits, both sides of the line between the tile and the lane kernel.
    # Uniform amplitudes: each target pattern gets its row sum.
    n, rng = 28, np.random.default_rng(28)
    u = random_matrix(2, rng, unitary=False)
    st = ss32.create(n)
    ss32.set_state_uniform(st)
    cvals = (1 << len(controls)) - 2
    sim.apply_controlled_gate(qs, controls, cvals, to_interleaved(u, np.float32),
                              st)
    a = float(np.float32(2.0**-14))
    for i in rng.integers(0, 1 << n, 3000).tolist():
        want = a
        if all((i >> c) & 1 == (cvals >> b) & 1 for b, c in enumerate(controls)):
            want = a * u[((i >> qs[0]) & 1) | ((i >> qs[1]) & 1) << 1].sum()
        assert abs(ss32.get_ampl(st, i) - want) < 1e-6 * a * 4, i


@pytest.mark.parametrize("n", [10, 13, 20, 21])
def test_four_qubit_gates_around_the_small_state_kernel(n, sim):
    # complex64 k = 4 without a target below qubit 5: up to 20 qubits 32 groups
    # a wave, above it the lane kernel (which also takes target 4 at any size).
    rng = np.random.default_rng(n)
    for qs in ([5, 6, 7, 8], [6, 7, 8, 9], list(range(n - 4, n)), [4, 6, 7, 9]):
        m = to_interleaved(random_matrix(4, rng), np.float32)
        s = random_state(n, rng, np.float32)
        st = upload(s, n, np.float32)
        sim.apply_gate(qs, m, st)
        oracle.apply_gate(n, s, qs, m)
        assert rel_l2(st.to_numpy(), s) < 1e-6, qs


@pytest.mark.parametrize("k", [5, 6])
@pytest.mark.parametrize("n", [9, 10, 11, 12, 16, 22])
def test_complex128_wide_gates(n, k, sim):
    # Below, at and above one set (2^10, 2^11 amplitudes), and enough sets
    # for several per workgroup (2^22: the double-buffered loop); the targets
    # that end in lanes, members and copies alike.
    rng = np.random.default_rng(n + k)
    for qs in (list(range(k)), list(range(n - k, n)),
               sorted(rng.choice(n, k, replace=False).tolist()),
               [0] + list(range(n - k + 1, n)),
               [0, 2, 4] + list(range(n - k + 3, n))):
        if len(set(qs)) < k:
            continue
        m = to_interleaved(random_matrix(k, rng), np.float64)
        s = random_state(n, rng, np.float64)
        st = upload(s, n, np.float64)
        sim.apply_gate(qs, m, st)
        oracle.apply_gate(n, s, qs, m)
        assert rel_l2(st.to_numpy(), s) < 1e-14, (n, qs)


@pytest.mark.parametrize("dtype", DTYPES)
def test_expectation_value_vs_oracle(dtype, sim):
    rng = np.random.default_rng(14)
    for n in (1, 2, 4, 6, 9, 13, 18):
        for k in range(1, min(n, 6) + 1):
            for qs in _target_sets(n, k, rng)[:3]:
                u = random_matrix(k, rng, unitary=False)
                m = to_interleaved(u, dtype)
                s = random_state(n, rng, dtype)
                st = upload(s, n, dtype)
                got = sim.expectation_value(qs, m, st)
                ref = oracle.expectation_value(n, s, qs, m)
                tol = 2e-6 if dtype == np.float32 else 1e-12
                assert abs(got - ref) < tol, (n, k, qs, got, ref)


@pytest.mark.parametrize("dtype", DTYPES)
def test_expectation_value_many_chunks(dtype, sim):
    # 24 qubits: more chunks (lane and MFMA kernels) and groups than one round
    # of the grid holds, targets in the lanes and above.
    n, rng = 24, np.random.default_rng(41)
    s = random_state(n, rng, dtype)
    st = upload(s, n, dtype)
    for k in range(1, 5):
        for qs in (list(range(k)), [6 + 4 * b for b in range(k)],
                   [2] + [n - k + 1 + b for b in range(k - 1)]):
            m = to_interleaved(random_matrix(k, rng, unitary=False), dtype)
            got = sim.expectation_value(qs, m, st)
            ref = oracle.expectation_value(n, s, qs, m)
            assert abs(got - ref) < (2e-6 if dtype == np.float32 else 1e-12), qs


def test_expectation_value2_known_answer(sim):
    exp = known_answers()["expectation2"]["expected_real"]
    n, ops = expectation2_circuit()
    for dtype in DTYPES:
        ss = qsim_amd.StateSpace(dtype)
        st = ss.create(n)
        ss.set_state_zero(st)
        for spec in ops:
            qs, m, _, _ = gate_op(spec, dtype)
            sim.apply_gate(qs, m, st)
        for k in range(1, 7):
            pm = to_interleaved(pauli_string_matrix(k), dtype)
            total = 0j
            for i in range(n - k + 1):
                total += (0.1 + 0.2 * i) * sim.expectation_value(
                    list(range(i, i + k)), pm, st)
            assert abs(total.real - exp[k - 1]) < 1e-6
            assert abs(total.imag) < 1e-8


@pytest.mark.parametrize("dtype", DTYPES)
def test_reductions_vs_oracle(dtype):
    rng = np.random.default_rng(15)
    ss = qsim_amd.StateSpace(dtype)
    for n in (0, 1, 3, 8, 11, 16, 21):
        a = random_state(n, rng, dtype) * dtype(1.3)
        b = random_state(n, rng, dtype)
        sa, sb = upload(a, n, dtype), upload(b, n, dtype)
        tol = 1e-12
        assert abs(ss.norm(sa) - oracle.norm(n, a)) < tol
        assert abs(ss.inner_product(sa, sb) - oracle.inner_product(n, a, b)) < tol
        assert abs(ss.real_inner_product(sa, sb)
                   - oracle.real_inner_product(n, a, b)) < tol
    # Size mismatch -> NaN (lib/statespace_cuda.h:219-223).
    assert np.isnan(ss.real_inner_product(upload(a, n, dtype), ss.create(n - 1)))


@pytest.mark.parametrize("dtype", DTYPES)
def test_sample_identical_to_oracle(dtype):
    rng = np.random.default_rng(16)
    ss = qsim_amd.StateSpace(dtype)
    for n in (1, 2, 5, 9, 12, 13, 16, 20):
        s = random_state(n, rng, dtype)
        st = upload(s, n, dtype)
        norm = oracle.serial_norm(n, s)
        for num, seed in ((1, 3), (1000, 0), (20000, 9)):
            draws = oracle.generate_random_values(num, seed, norm)
            got = ss.sample_with_draws(st, draws[:-1])
            ref = oracle.sample_with_draws(n, s, draws)
            np.testing.assert_array_equal(got, ref)
        got = ss.sample(st, 1000, 5)
        np.testing.assert_array_equal(got, oracle.sample(n, s, 1000, 5))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n", [21, 23])
def test_sample_over_several_spans(n, dtype):
    # 2 and 8 spans of 1024 sample blocks: the outer prefix sums and their
    # search.
    rng = np.random.default_rng(n)
    ss = qsim_amd.StateSpace(dtype)
    s = random_state(n, rng, dtype)
    st = upload(s, n, dtype)
    draws = oracle.generate_random_values(20000, 9, oracle.serial_norm(n, s))
    np.testing.assert_array_equal(ss.sample_with_draws(st, draws[:-1]),
                                  oracle.sample_with_draws(n, s, draws))
    np.testing.assert_array_equal(ss.sample(st, 1000, 5),
                                  oracle.sample(n, s, 1000, 5))


def test_sample_over_more_spans_than_a_workgroup(ss32):
    # 29 qubits: 512 spans, two rounds of the outer scan.  Uniform amplitudes:
    # a draw in the middle of amplitude j finds j.
    n = 29
    st = ss32.create(n)
    ss32.set_state_uniform(st)
    p = float(np.float32(1 / np.sqrt(1 << n))) ** 2
    j = np.unique(np.random.default_rng(5).integers(0, 1 << n, 20000))
    j[[0, -1]] = 0, (1 << n) - 1
    np.testing.assert_array_equal(ss32.sample_with_draws(st, (j + 0.5) * p), j)
    draws = oracle.generate_random_values(1000, 3, ss32.norm(st))[:-1] / p
    got = ss32.sample(st, 1000, 3)
    far = np.abs(draws - np.round(draws)) > 1e-3
    np.testing.assert_array_equal(got[far], np.floor(draws)[far])
    assert far.mean() > 0.9


def test_long_sampling_leaves_other_threads_their_turn(ss32):
    # 30 million draws take about a second of host time; norms on another
    # thread do not wait for them.
    n, num = 10, 30_000_000
    s = random_state(n, np.random.default_rng(6))
    st = upload(s, n, np.float32)
    took = []

    def sample():
        t = time.perf_counter()
        bits = ss32.sample(st, num, 4)
        took.append(time.perf_counter() - t)
        took.append(np.bincount(bits.astype(np.int64), minlength=1 << n))
    th = threading.Thread(target=sample)
    th.start()
    longest = 0.0
    while th.is_alive():
        t = time.perf_counter()
        ss32.norm(st)
        longest = max(longest, time.perf_counter() - t)
    th.join()
    assert longest < 0.5 * took[0], (longest, took[0])
    p = np.abs(from_interleaved(s)) ** 2
    assert np.abs(took[1] / num - p / p.sum()).max() < 6 * np.sqrt(p.max() / num)


def test_sample_draws_past_the_end(ss32):
    # Draws at or beyond the total map to 2^n - 1 (lib/statespace_basic.h:227-229).
    n = 10
    rng = np.random.default_rng(17)
    s = random_state(n, rng, np.float32)
    st = upload(s, n, np.float32)
    total = oracle.serial_norm(n, s)
    draws = np.array([0.0, total * 0.5, total, total * 2])
    got = ss32.sample_with_draws(st, draws)
    ref = oracle.sample_with_draws(n, s, np.append(draws, total * 2))
    np.testing.assert_array_equal(got, ref)
    assert got[-1] == (1 << n) - 1


@pytest.mark.parametrize("dtype", DTYPES)
def test_measurement_vs_oracle(dtype):
    rng = np.random.default_rng(18)
    ss = qsim_amd.StateSpace(dtype)
    for n in (3, 10, 14, 18):
        s = random_state(n, rng, dtype)
        st = upload(s, n, dtype)
        pn = ss.partial_norms(st)
        assert abs(pn.sum() - oracle.norm(n, s)) < 1e-12
        c = from_interleaved(s)
        p = np.abs(c.astype(np.complex64 if dtype == np.float32 else np.complex128)) ** 2
        csum = np.cumsum(p.astype(np.float64))
        for trial in range(20):
            qubits = sorted(rng.choice(n, size=int(rng.integers(1, n + 1)),
                                       replace=False).tolist())
            mask = sum(1 << q for q in qubits)
            r_total = rng.uniform(0, csum[-1])
            res = ss.virtual_measure(qubits, lambda norm: r_total * norm / csum[-1], st)
            k_ref = int(np.searchsorted(csum, r_total * pn.sum() / csum[-1], side="right"))
            k_ref = min(k_ref, (1 << n) - 1)
            # Allow the boundary index only when the draw sits on a rounding tie.
            assert res[1] == (k_ref & mask) or abs(csum[k_ref] - r_total) < 1e-12
        mask, bits = 0b101, 0b100
        ss.collapse(st, mask, bits)
        oracle.collapse(n, s, mask, bits)
        assert rel_l2(st.to_numpy(), s) < TOL[dtype] * 4


def test_measurement_of_a_long_range(ss32):
    # 23 qubits: ranges of 8192 amplitudes, two narrowing steps of eight loads
    # in flight.  Amplitudes are whole numbers times 2^-22: squares and sums
    # are exact, so every index is.
    n, rng = 23, np.random.default_rng(23)
    s = np.zeros(2 << n, np.float32)
    s[0::2] = rng.integers(-2000, 2001, 1 << n) * 2.0**-22
    st = upload(s, n, np.float32)
    p = (s[0::2] * s[0::2]).astype(np.float64)
    pn = ss32.partial_norms(st)
    part = (1 << n) // len(pn)
    np.testing.assert_array_equal(pn, p.reshape(-1, part).sum(axis=1))
    for m in (0, 1, 511, 1023):
        csum = np.cumsum(p[m * part:(m + 1) * part])
        for r in rng.uniform(0, csum[-1], 50):
            k = ss32.find_measured_bits(st, m, r, (1 << n) - 1)
            assert k == m * part + np.searchsorted(csum, r, side="right")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,mask,bits", [
    (6, 0b111000, 0b101000), (12, 0b1000, 0b1000), (13, 0b1, 0),
    (13, 0b1000000000100, 0b100), (16, 0b1011000010001000, 0b11000000001000),
    (16, 0xffff, 0x1234), (16, 0xfff8, 0x1230), (19, 0x60000, 0x20000),
    (14, 0b11000, 0b100)])
def test_collapse_masks(n, mask, bits, dtype):
    # Measured qubits whose zero half is skipped (from qubit 3, complex128 2),
    # those that are only tested, both, all; the last wants a bit outside the
    # mask, which no amplitude has.
    rng = np.random.default_rng(n)
    ss = qsim_amd.StateSpace(dtype)
    s = random_state(n, rng, dtype)
    st = upload(s, n, dtype)
    ss.collapse(st, mask, bits)
    if bits & ~mask:
        assert not st.to_numpy().any()
    else:
        oracle.collapse(n, s, mask, bits)
        assert rel_l2(st.to_numpy(), s) < TOL[dtype] * 4


@pytest.mark.parametrize("n", [14, 18])
def test_states_aligned_to_an_amplitude(n, sim, ss32):
    # A complex64 state 8 bytes off a 16-byte boundary, as a caller's buffer
    # may be: the kernels that load 16 bytes give what they give on it.
    rng = np.random.default_rng(n)
    s, t = random_state(n, rng), random_state(n, rng)
    room = [ss32.create(n + 1) for _ in range(2)]
    assert all(r.ptr % 16 == 0 for r in room)
    results = []
    for shift in (0, 8):
        a, b = (qsim_amd.State(n, np.float32, ptr=r.ptr + shift, owner=False)
                for r in room)
        a.from_numpy(s)
        b.from_numpy(t)
        rng = np.random.default_rng(1)
        out = [ss32.norm(a), ss32.inner_product(a, b), ss32.partial_norms(a),
               ss32.sample(a, 1000, 2)]
        for tb in (9, 13, 14):
            tile = list(range(4)) + list(range(n - tb + 4, n))
            gates = []
            for k in (1, 2, 3, 4, 4):
                qs = sorted(rng.choice(tile, k, replace=False).tolist())
                gates.append((qs, to_interleaved(random_matrix(k, rng),
                                                 np.float64)))
            sim.apply_gate_block(tile, gates, a)
        for k in (1, 2, 3, 4, 5, 6):
            for qs in (list(range(k)), list(range(n - k, n))):
                m = to_interleaved(random_matrix(k, rng), np.float32)
                sim.apply_gate(qs, m, a)
                out.append(sim.expectation_value(qs, m, a))
        out.append(a.to_numpy())
        ss32.collapse(a, 0b1010010, 0b10)
        out += [a.to_numpy(), b.to_numpy()]
        results.append(out)
    for x, y in zip(*results):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("n,run", [(18, 64), (24, 64), (24, 1024)])
def test_measured_index_has_probability(n, run):
    # Draws at the sums ahead of runs of zeros, to the last bits of rounding:
    # whichever way they round, the index found is the last amplitude of the
    # run before or the first of the next one, never a zero.
    rng = np.random.default_rng(n + run)
    ss = qsim_amd.StateSpace(np.float64)
    size = 1 << n
    c = rng.normal(size=size) * ((np.arange(size) // run) % 2 == 0)
    c /= np.sqrt(np.sum(c * c))
    a = np.zeros(2 * size)
    a[0::2] = c
    st = upload(a, n, np.float64)
    parts = len(ss.partial_norms(st))
    part = size // parts
    for m in range(0, parts, max(1, parts // 64)):
        p = c[m * part:(m + 1) * part] ** 2
        # The last runs of a part have no run after them.
        for b in range(run, part - run, 2 * run):
            total = p[:b].sum()
            for ulps in range(-4, 5):
                r = total + ulps * np.spacing(total)
                k = ss.find_measured_bits(st, m, r, size - 1) - m * part
                assert k in (b - 1, b + run), (m, b, ulps, k)


@pytest.mark.parametrize("dtype", DTYPES)
def test_state_fills_and_elementwise(dtype):
    ss = qsim_amd.StateSpace(dtype)
    rng = np.random.default_rng(19)
    n = 13
    st = ss.create(n)
    ss.set_state_zero(st)
    s = st.to_numpy()
    assert s[0] == 1 and np.count_nonzero(s) == 1
    ss.set_state_uniform(st)
    s = st.to_numpy()
    assert np.all(s[0::2] == dtype(1.0 / np.sqrt(1 << n))) and not s[1::2].any()
    ss.set_all_zeros(st)
    assert not st.to_numpy().any()
    a = random_state(n, rng, dtype)
    b = random_state(n, rng, dtype)
    sa, sb = upload(a, n, dtype), upload(b, n, dtype)
    assert ss.add(sa, sb)
    np.testing.assert_array_equal(sb.to_numpy(), (a + b).astype(dtype))
    ss.multiply(0.37, sa)
    np.testing.assert_array_equal(sa.to_numpy(), a * dtype(0.37))
    for exclude in (False, True):
        sc = upload(a, n, dtype)
        ss.bulk_set_ampl(sc, 0b110, 0b010, complex(0.25, -0.5), exclude)
        ref = from_interleaved(a).copy()
        sel = ((np.arange(1 << n) & 0b110) == 0b010) != exclude
        ref[sel] = complex(0.25, -0.5)
        np.testing.assert_array_equal(from_interleaved(sc.to_numpy()), ref)
    ss.set_ampl(sa, 77, complex(1.5, -2.5))
    assert ss.get_ampl(sa, 77) == complex(1.5, -2.5)
    sd = ss.create(n)
    assert ss.copy(sa, sd)
    np.testing.assert_array_equal(sd.to_numpy(), sa.to_numpy())
    assert not ss.copy(sa, ss.create(n + 1))
    assert not ss.add(sa, ss.create(n + 1))


def test_grid20_circuit_vs_oracle_and_reference(ss32, sim):
    # The 20-qubit / 14-cycle grid circuit, gate by gate on the GPU.
    txt = circuits.grid_circuit(20, 14, seed=0)
    c = oracle.Circuit(txt, np.float32)
    s_or, _ = c.run()
    st = ss32.create(20)
    ss32.set_state_zero(st)
    n, ops = circuits.grid_circuit_ops(4, 5, 14, 0)
    for t, name, qs, prm in ops:
        q, m = oracle.gate_matrix(name, list(qs), list(prm), np.float32)
        sim.apply_gate(q, m, st)
    s = st.to_numpy()
    assert rel_l2(s, s_or) < 1e-5
    g = reference_runs()["grid20"]
    amps = g["avx"]["amplitudes"]
    cplx = from_interleaved(s)
    for i, (re, im) in amps.items():
        assert abs(cplx[int(i)] - complex(re, im)) < 1e-6
    # Identical draws on the identical state: identical bitstrings.
    bits = ss32.sample(st, 1000, 0)
    np.testing.assert_array_equal(bits, oracle.sample(20, s, 1000, 0))
    # Against the reference's own, independently evolved FP32 state the
    # cumulative sums differ by ~1e-9, which moves a few of 1000 draws across
    # an amplitude boundary (each such flip lands on a neighbouring index).
    ref_bits = np.array(g["samples_seed0"], dtype=np.uint64)
    flips = np.flatnonzero(bits != ref_bits)
    print(f"grid20: {len(flips)} of 1000 samples differ from the reference's "
          f"independently evolved state", flush=True)
    assert len(flips) <= 10


def test_large_state_round_trip(sim):
    # 27 qubits: gates followed by their inverses restore the state; the norm
    # is preserved by every pass (size-independent properties).
    n = 27
    rng = np.random.default_rng(20)
    ss = qsim_amd.StateSpace(np.float32)
    st = ss.create(n)
    ss.set_state_uniform(st)
    ref = ss.create(n)
    ss.set_state_uniform(ref)
    gates = []
    for k in (1, 2, 3, 4, 5, 6, 2, 3):
        qs = sorted(rng.choice(n, size=k, replace=False).tolist())
        gates.append((qs, random_matrix(k, rng)))
    for qs, u in gates:
        sim.apply_gate(qs, to_interleaved(u, np.float32), st)
        assert abs(ss.norm(st) - 1) < 1e-5
    for qs, u in reversed(gates):
        sim.apply_gate(qs, to_interleaved(u.conj().T, np.float32), st)
    ip = ss.inner_product(ref, st)
    assert abs(ip - 1) < 1e-5


def test_error_paths(ss32, sim):
    st = ss32.create(5)
    with pytest.raises(qsim_amd.QsimHipError) as e:
        sim.apply_gate(list(range(7)), np.zeros(2 << 14, np.float32), ss32.create(8))
    assert e.value.code == -4
    with pytest.raises(qsim_amd.QsimHipError) as e:
        sim.apply_gate([3, 1], np.zeros(32, np.float32), st)
    assert e.value.code == -1
    with pytest.raises(qsim_amd.QsimHipError):
        sim.apply_gate([5], np.zeros(8, np.float32), st)
    with pytest.raises(qsim_amd.QsimHipError):
        sim.apply_controlled_gate([1], [1], 1, np.zeros(8, np.float32), st)
    # Allocation beyond the device -> Null (None), not an exception.
    assert qsim_amd.StateSpace(np.float64).create(40) is None


@pytest.mark.parametrize("method", [qsim_amd.METHOD_VECTOR, qsim_amd.METHOD_AUTO])
def test_fp32_methods_vs_oracle(method, sim):
    # FP32 vector kernels and FP32 MFMA (k >= 4) meet the same 1e-6 bar, for
    # low, high, mixed and random targets.
    rng = np.random.default_rng(21)
    qsim_amd.set_gate_method(method)
    try:
        for n in (9, 10, 11, 12, 13, 16, 19):
            for k in (4, 5, 6):
                if k + 5 > n:
                    continue
                for qs in _target_sets(n, k, rng):
                    u = random_matrix(k, rng)
                    m = to_interleaved(u, np.float32)
                    s = random_state(n, rng, np.float32)
                    st = upload(s, n, np.float32)
                    sim.apply_gate(qs, m, st)
                    oracle.apply_gate(n, s, qs, m)
                    err = rel_l2(st.to_numpy(), s)
                    assert err < 1e-6, (method, n, k, qs, err)
    finally:
        qsim_amd.set_gate_method(qsim_amd.METHOD_AUTO)


@pytest.mark.parametrize("k", [5, 6])
def test_vector_method_complex128_wide_gates(k, sim):
    # METHOD_VECTOR names the vector kernels in both precisions.  The FP64
    # matrix-unit kernel returns the same bits, so its time tells which ran:
    # at 20 qubits with low targets 16 (k = 5) and 26 us (k = 6) against 39 and
    # 355 us.
    n, qs = 20, list(range(k))
    rng = np.random.default_rng(k)
    m = to_interleaved(random_matrix(k, rng), np.float64)
    s = random_state(n, rng, np.float64)
    ms, got = {}, {}
    for method in (qsim_amd.METHOD_VECTOR, qsim_amd.METHOD_AUTO):
        st = upload(s, n, np.float64)
        qsim_amd.set_gate_method(method)
        try:
            sim.apply_gate(qs, m, st)
            got[method] = st.to_numpy()
            qsim_amd.PassTimer.start(32)
            for _ in range(20):
                sim.apply_gate(qs, m, st)
            ms[method] = np.median(qsim_amd.PassTimer.stop(32))
        finally:
            qsim_amd.set_gate_method(qsim_amd.METHOD_AUTO)
    oracle.apply_gate(n, s, qs, m)
    for method, a in got.items():
        assert rel_l2(a, s) < 1e-14, method
    assert ms[qsim_amd.METHOD_VECTOR] > 1.5 * ms[qsim_amd.METHOD_AUTO], ms


def test_vector_method_expectation_values(sim):
    # The 4-qubit complex64 kernels add their FP64 sums in different orders:
    # over amplitudes of many magnitudes (sums that round) the last bits tell
    # which ran.
    n, rng = 16, np.random.default_rng(40)
    s = random_state(n, rng, np.float32) * np.exp2(rng.uniform(-60, 0, 2 << n))
    s = (s / np.linalg.norm(s)).astype(np.float32)
    st = upload(s, n, np.float32)
    differ = 0
    for qs in _target_sets(n, 4, rng):
        m = to_interleaved(random_matrix(4, rng, unitary=False), np.float32)
        ref = oracle.expectation_value(n, s, qs, m)
        auto = sim.expectation_value(qs, m, st)
        qsim_amd.set_gate_method(qsim_amd.METHOD_VECTOR)
        try:
            vector = sim.expectation_value(qs, m, st)
        finally:
            qsim_amd.set_gate_method(qsim_amd.METHOD_AUTO)
        assert abs(auto - ref) < 2e-6 and abs(vector - ref) < 2e-6, qs
        differ += auto != vector
    assert differ > 0


def test_bf16x3_mfma_accuracy(sim):
    # Split-BF16 x3 products carry ~2^-16 relative error per product: per pass
    # the state stays within 5e-5 relative L2 of the FP64 result.
    rng = np.random.default_rng(22)
    qsim_amd.set_gate_method(qsim_amd.METHOD_MFMA_BF16X3)
    try:
        for n in (11, 12, 16, 20):
            for k in (5, 6):
                for qs in _target_sets(n, k, rng):
                    u = random_matrix(k, rng)
                    s = random_state(n, rng, np.float64)
                    st = upload(s.astype(np.float32), n, np.float32)
                    sim.apply_gate(qs, to_interleaved(u, np.float64), st)
                    oracle.apply_gate(n, s, qs, to_interleaved(u, np.float64))
                    err = rel_l2(st.to_numpy(), s)
                    assert err < 5e-5, (n, k, qs, err)
    finally:
        qsim_amd.set_gate_method(qsim_amd.METHOD_AUTO)


def test_fp16x2_mfma_accuracy(sim):
    # FP16 with a power-of-two scale per matrix and per group, matrix and
    # amplitudes in two fp16 parts each (22 bits), FP32 accumulation: per
    # pass the state stays within 1e-6 relative L2 of the FP64 result, for
    # low, high, mixed and random targets (LDS-tile and register paths).
    rng = np.random.default_rng(23)
    qsim_amd.set_gate_method(qsim_amd.METHOD_MFMA_FP16X2)
    try:
        for n in (11, 12, 13, 16, 20):
            for k in (5, 6):
                for qs in _target_sets(n, k, rng):
                    u = random_matrix(k, rng)
                    s = random_state(n, rng, np.float64)
                    st = upload(s.astype(np.float32), n, np.float32)
                    sim.apply_gate(qs, to_interleaved(u, np.float64), st)
                    oracle.apply_gate(n, s, qs, to_interleaved(u, np.float64))
                    err = rel_l2(st.to_numpy(), s)
                    assert err < 1e-6, (n, k, qs, err)
    finally:
        qsim_amd.set_gate_method(qsim_amd.METHOD_AUTO)


@pytest.mark.parametrize("method,bar", [
    (qsim_amd.METHOD_AUTO, 1e-6),           # exact FP32, row blocks
    (qsim_amd.METHOD_MFMA_BF16X3, 5e-5),    # split-BF16, row blocks
    (qsim_amd.METHOD_MFMA_FP16X2, 1e-6)])   # FP16 with scaling
def test_k56_row_block_kernels_over_many_sets(sim, method, bar):
    # At 22 qubits every k = 5, 6 kernel has more sets of groups than
    # workgroups (2048 against at most 4 per CU), so each workgroup runs
    # its double-buffered loop: the next set's loads in flight while the
    # current one is computed, for low (LDS set) and high (register)
    # targets.
    rng = np.random.default_rng(24)
    n = 22
    qsim_amd.set_gate_method(method)
    try:
        for k in (5, 6):
            for qs in ([0, 1, 2, 3, 4, 5][:k], [3, 7, 11, 15, 19, 21][:k],
                       [5, 9, 12, 14, 17, 20][:k]):
                u = random_matrix(k, rng)
                s = random_state(n, rng, np.float64)
                st = upload(s.astype(np.float32), n, np.float32)
                sim.apply_gate(qs, to_interleaved(u, np.float64), st)
                oracle.apply_gate(n, s, qs, to_interleaved(u, np.float64))
                err = rel_l2(st.to_numpy(), s)
                print(f"method {method} k={k} qs={qs} relL2 {err:.2e}",
                      flush=True)
                assert err < bar, (method, k, qs, err)
    finally:
        qsim_amd.set_gate_method(qsim_amd.METHOD_AUTO)


@pytest.mark.parametrize("scale", [1e-30, 1e-3, 1.0, 1e3, 1e30])
def test_fp16x2_scaling_over_magnitudes(sim, scale):
    # The per-group scale keeps fp16's 5-bit exponent out of the way: groups
    # of very different size in one state (one group all zero, one tiny, the
    # rest at `scale`), and non-unitary matrices scaled by 1e-3 and 1e3.
    rng = np.random.default_rng(24)
    n = 14
    qsim_amd.set_gate_method(qsim_amd.METHOD_MFMA_FP16X2)
    try:
        for k, qs in ((5, [0, 3, 6, 9, 12]), (6, [5, 6, 7, 8, 9, 13]),
                      (6, [0, 1, 2, 3, 4, 5])):
            for mscale in (1e-3, 1.0, 1e3):
                u = random_matrix(k, rng) * mscale
                s = random_state(n, rng, np.float64) * scale
                s[: 2 << k] = 0.0           # a zero group (low targets)
                s[2 << k: 4 << k] *= 1e-20  # a tiny one
                s = s.astype(np.float32).astype(np.float64)
                st = upload(s.astype(np.float32), n, np.float32)
                sim.apply_gate(qs, to_interleaved(u, np.float64), st)
                oracle.apply_gate(n, s, qs, to_interleaved(u, np.float64))
                err = rel_l2(st.to_numpy(), s)
                assert err < 1e-6, (k, qs, mscale, err)
    finally:
        qsim_amd.set_gate_method(qsim_amd.METHOD_AUTO)
