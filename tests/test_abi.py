"""The C ABI library loads and exports every symbol include/qsim_hip.h declares
(no GPU needed; no compute is called)."""

import os
import re
from array import array

import numpy as np
import pytest

import qsim_amd

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def header_functions(path):
    text = open(path).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(qsim_hip_\w+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    names = header_functions(os.path.join(ROOT, "include", "qsim_hip.h"))
    assert len(names) > 30
    dll = qsim_amd.load_library()
    missing = [n for n in names if not hasattr(dll, n)]
    assert not missing, missing


def test_python_signatures_cover_header():
    names = header_functions(os.path.join(ROOT, "include", "qsim_hip.h"))
    declared = {s[0] for s in qsim_amd.SIGNATURES}
    assert set(names) == declared


def test_min_size_needs_no_gpu():
    dll = qsim_amd.load_library()
    assert dll.qsim_hip_min_size(0) == 64
    assert dll.qsim_hip_min_size(20) == 2 << 20
    assert dll.qsim_hip_num_partial_norms(30) == 1024


def test_library_is_gfx950_code():
    # The shared object carries a gfx950 code object (offload bundle).
    data = open(qsim_amd.LIB_PATH, "rb").read()
    assert b"gfx950" in data


@pytest.mark.parametrize("qs", [
    [], [0, 1], (2, 5), range(3), [0, True], [1.0], [np.int64(3)],
    [np.int64(-1)], [-1], [1 << 32], [np.int64(1 << 32)], ["0", "1"], "01", 5,
    None, [None], [[0, 1]], {0, 1}, {0: 1}, b"\0\1\2\3", bytes(8),
    bytearray([0, 1]), memoryview(bytes([0, 1])), array("I", [0, 1]),
    array("b", [0, 1]), np.array([0, 1]), np.array([-1]), np.array([1 << 32]),
    np.array([0.0, 1.0]), np.array([[0, 1]]), np.array([[3]]),
    np.array([True]), np.array(3), np.array([3], dtype=object)], ids=repr)
def test_qubit_lists_as_numpy_takes_them(qs):
    # A gate call's qubits are what numpy makes of them as uint32, and what it
    # refuses is refused.
    try:
        ref = np.asarray(qs, dtype=np.uint32).reshape(-1)
    except Exception as e:
        with pytest.raises(type(e)):
            qsim_amd._qubits(qs)
        return
    owner, addr, count = qsim_amd._qubits(qs)
    assert count == len(ref)
    np.testing.assert_array_equal(np.frombuffer(owner, np.uint32) if count
                                  else np.empty(0, np.uint32), ref)
    assert np.asarray(owner).ctypes.data == addr or count == 0
