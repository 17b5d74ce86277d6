"""How large the planner's programs become (quict_amd/csrc/qsim_wire_plan.hpp), on the
CPU model, which also runs them."""
import ctypes
import random

import numpy as np
import pytest

from quict_amd import _native as nat
from quict_amd.core import Circuit, H, Unitary, X
from quict_amd.simulation.gate_compiler import compile_gates
from test_wire_planner import check, emu  # noqa: F401  (the fixture)


def plan(lib, recs, n):
    """The plan's counts: passes, fused passes, ops, ..."""
    st = np.zeros(8, dtype=np.int32)
    rc = lib.wires_apply(None, n, nat.gate_array_ptr(recs), len(recs), 4, 8, 4, 16, st.ctypes.data_as(ctypes.c_void_p))
    assert rc == 0, lib.wires_last_error()
    return st


def tables(n, count, seed=1):
    rng, r = random.Random(seed), np.random.RandomState(seed)
    c = Circuit(n)
    for _ in range(count):
        Unitary(np.diag(np.exp(1j * r.uniform(0, 6, 8)))) | c(rng.sample(range(n), 3))
    return compile_gates(c.gates, n)


def test_a_pass_takes_as_many_tables_as_it_stages(emu):  # noqa: F811
    """Three-qubit diagonal gates that all commute: those that wait for another pass do
    not use up the tables of this one.  The planner of whole gates takes 12 passes."""
    recs, keep = tables(20, 200)
    assert plan(emu, recs, 20)[0] <= 12
    recs, keep = tables(15, 200)
    check(emu, recs, 15)


def all_ones_phase(n, k, hadamards):
    """X on k qubits, a phase on all of them, X again; with Hadamard gates around: a
    Grover diffusion."""
    c = Circuit(n)
    args = list(range(n - k, n))
    m = np.eye(1 << k, dtype=complex)
    m[-1, -1] = np.exp(0.7j)
    for g in [H, X] if hadamards else [X]:
        for q in args:
            g | c(q)
    Unitary(m) | c(args)
    for g in [X, H] if hadamards else [X]:
        for q in args:
            g | c(q)
    return c


@pytest.mark.parametrize("hadamards", [False, True])
@pytest.mark.parametrize("k", [3, 4, 6, 8, 10])
def test_a_phase_under_flips_stays_one_phase(emu, k, hadamards):  # noqa: F811
    n = 14
    recs, keep = compile_gates(all_ones_phase(n, k, hadamards).gates, n)
    # a phase, at most a flip or a rotation with two phases on either side of it per
    # qubit, relayouts between them
    assert plan(emu, recs, n)[2] <= 8 * k
    check(emu, recs, n)
