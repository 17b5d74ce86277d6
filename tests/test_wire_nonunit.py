"""Diagonal gates and exchanges whose entries are far from modulus 1, on the CPU model
of the planned passes: nothing may be divided by such an entry.  Every amplitude keeps
its relative precision: 8 roundings of half a unit in its last place a gate."""
import ctypes

import numpy as np
import pytest

from quict_amd import _native as nat
from test_wire_planner import emu  # noqa: F401  (the fixture)

X = (nat.GATE_XPERM, 0, [1, 1])
CASES = {
    "diag": [(nat.GATE_DIAG, 0, [1e-200, 1], [3])],
    "diag denormal ratio": [(nat.GATE_DIAG, 0, [1e-160, 1], [3])],
    "diag, again and again": [(nat.GATE_DIAG, 0, [1e-30, 1], [3])] * 12,
    "controlled diag": [(nat.GATE_DIAG, 2, [1e-200, 1j], [1, 7, 3])],
    "two-target diag": [(nat.GATE_DIAG, 0, [1e-200, 1, 1, 1e-200], [3, 9])],
    "exchange": [(nat.GATE_XPERM, 0, [1e-200, 1], [3])],
    "controlled exchange": [(nat.GATE_XPERM, 1, [1, 1e-200], [11, 3])],
    "swap": [(nat.GATE_SWAP, 0, [1e-200, 1], [3, 9])],
    "phase under a flip": [X + ([3],), (nat.GATE_PHASE, 1, [1e-200], [3, 9]), X + ([3],)],
    "diag under flips": [X + ([3],), X + ([1],), (nat.GATE_DIAG, 1, [1e-200, 1], [1, 3]), X + ([1],)],
}


def records(name):
    gates = CASES[name]
    recs = np.zeros(len(gates), dtype=nat.QS_GATE_DTYPE)
    for rec, (kind, nc, m, bits) in zip(recs, gates):
        rec["kind"], rec["ncontrols"], rec["ntargets"] = kind, nc, len(bits) - nc
        rec["bits"][: len(bits)] = bits
        rec["m"][: 2 * len(m)] = np.array(m, dtype=complex).view(np.float64)
    return recs


@pytest.mark.parametrize("shape", [16, 8])
@pytest.mark.parametrize("n", [12, 14])
@pytest.mark.parametrize("name", list(CASES))
def test_entries_far_from_one(emu, name, n, shape):  # noqa: F811
    recs = records(name)
    rng = np.random.RandomState(1)
    v = rng.randn(1 << n) + 1j * rng.randn(1 << n)
    v /= np.linalg.norm(v)
    ref, st, P = v.copy(), np.zeros(8, dtype=np.int32), ctypes.c_void_p
    emu.cpu_apply_gates(ref.ctypes.data_as(P), n, nat.gate_array_ptr(recs), len(recs), 1)
    assert emu.wires_apply(v.ctypes.data_as(P), n, nat.gate_array_ptr(recs), len(recs), 4, 8, 4, shape,
                           st.ctypes.data_as(P)) == 0, emu.wires_last_error()
    assert np.all(np.abs(v - ref) <= 8 * 2.0 ** -53 * len(recs) * np.abs(ref))
