"""How large the planner's programs become (quict_amd/csrc/qsim_wire_plan.hpp), on the
CPU model, which also runs them."""
import ctypes
import random

import numpy as np

from quict_amd import _native as nat
from quict_amd.core import Circuit, Unitary
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
