"""Programs that start from |0...0> or from the identity matrix without either being
in the vector: on the CPU model of the passes (every tile, address and load as the
kernels take them), against the same program over a vector that holds the start.  Both
run the same operations on the same numbers: the results are equal, also where the
vector held NaN before.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from quict_amd import _native as nat
from quict_amd import workloads
from quict_amd.core import CX, Circuit, H, Rz, X
from quict_amd.simulation.gate_compiler import compile_gates

HERE = os.path.dirname(os.path.abspath(__file__))
P, I = ctypes.c_void_p, ctypes.c_int


@pytest.fixture(scope="module")
def emu():
    subprocess.check_call(["make", "-s", "-C", os.path.join(HERE, "planner")])
    lib = ctypes.CDLL(os.path.join(HERE, "planner", "_build", "libplanner_wires.so"))
    lib.wires_apply.argtypes = [P, I, P, I, I, I, I, I, P]
    lib.wires_run.argtypes = [P, I, I, P, I, I, I, I, I, P]
    lib.wires_last_error.restype = ctypes.c_char_p
    return lib


def circuit(name, n):
    c = Circuit(n)
    if name == "few":  # most qubits are never touched; flips before and after
        X | c(n - 1)
        H | c(0)
        CX | c([0, n - 2])
        X | c(1)
        Rz(0.3) | c(0)
        return c
    if name == "flips":
        for q in range(n):
            X | c(q)
        H | c(n // 2)
        for q in range(0, n - 1, 2):
            CX | c([q, q + 1])
        return c
    return workloads.random_mix_circuit(n, int(name), n + 1)


@pytest.mark.parametrize("RB,TB,L", [(4, 8, 4), (4, 7, 4), (4, 8, 3)])
@pytest.mark.parametrize("name", ["few", "flips", "3", "40", "300"])
@pytest.mark.parametrize("n,identity", [(3, False), (12, False), (13, False), (16, False), (5, True), (7, True),
                                        (8, True)])
def test_start_that_is_not_in_the_vector(emu, n, identity, name, RB, TB, L):
    recs, keep = compile_gates(circuit(name, n).gates, n)
    bits = 2 * n if identity else n
    want = np.zeros(1 << bits, dtype=np.complex128)
    if identity:
        want[:: (1 << n) + 1] = 1
    else:
        want[0] = 1
    got = np.full(1 << bits, np.nan + 1j * np.nan)
    st, st3 = np.zeros(8, dtype=np.int32), np.zeros(3, dtype=np.int64)
    gates = nat.gate_array_ptr(recs)
    assert emu.wires_apply(want.ctypes.data, bits, gates, len(recs), RB, TB, L, 16, st.ctypes.data) == 0
    assert emu.wires_run(got.ctypes.data, bits, identity, gates, len(recs), RB, TB, L, 16, st3.ctypes.data) == 0, \
        emu.wires_last_error()
    assert np.array_equal(got, want)
    if not identity and bits > RB + TB and st3[0]:
        assert st3[1] < st3[2]  # some tiles are known to be empty
