"""Records made for a whole circuit at once against records made gate by gate, and
uniform draws made in one call against draws one by one.

Tolerance of the payloads: closed forms of a matrix entry from another library's sin
and cos, each within one unit in the last place (2.3e-16 for values up to 1), at most
two factors: 1e-15.  Everything else is equal.
"""
import random

import numpy as np
import pytest

from quict_amd import _native as nat
from quict_amd.core import Circuit
from quict_amd.core import noise as qn
from quict_amd.core.gate import GATE_TYPE_TO_CLASS
from quict_amd.core.gate_type import GateType
from quict_amd.simulation import gate_compiler as gc
from quict_amd.simulation.density_matrix import program_records
from quict_amd.simulation.uniforms import uniforms

N = 9
ANGLES = [0, 0.0, 1, np.float64(0.3), np.pi, 2 * np.pi, 4 * np.pi, -2.5, 1e-300, 1e9]


def circuit(gates, seed, single):
    rng = random.Random(seed)
    types = [t for t, c in GATE_TYPE_TO_CLASS.items()
             if t not in (GateType.measure, GateType.reset, GateType.perm, GateType.perm_fx, GateType.unitary)]
    c = Circuit(N)
    for _ in range(gates):
        g = GATE_TYPE_TO_CLASS[rng.choice(types)]()
        if g.type == GateType.barrier:
            continue
        q = rng.sample(range(N), g.controls + g.targets)
        if g.params:
            g = g(*[rng.choice(ANGLES + [rng.uniform(-7, 7)]) for _ in range(g.params)])
        g | c(q)
    if single:
        c.convert_precision()
    return c


@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("kw", [{}, {"dagger": True}, {"conj": True, "row_offset": 3}])
def test_a_circuit_at_once_equals_gate_by_gate(single, kw):
    c = circuit(400, 5, single)
    got, keep = gc.compile_gates(c.gates, N, **kw)
    want, held = np.zeros(len(c.gates), dtype=nat.QS_GATE_DTYPE), []
    k = 0
    for g in c.gates:
        k += gc.compile_gate(g, N, want[k], held, **kw)
    want = want[:k]
    assert len(got) == k and len(keep) == len(held)
    for f in ("kind", "ncontrols", "ntargets", "bits"):
        assert np.array_equal(got[f], want[f])
    tol = 1e-15 if not single else 2.0 ** -23  # (a rounding to 32 bits can fall either way)
    assert np.max(np.abs(got["m"] - want["m"])) <= tol
    assert np.array_equal(got["big"] != 0, want["big"] != 0)
    for a, b in zip(keep, held):
        assert np.array_equal(a, b)


def test_classes_that_read_their_attributes_otherwise():
    class Shifted(GATE_TYPE_TO_CLASS[GateType.h]):
        @property
        def targs(self):
            return [q + 1 for q in self._targs]

    g = Shifted()
    g._targs = [2]
    recs, _ = gc.compile_gates([g], N)
    assert recs["bits"][0, 0] == N - 1 - 3


def test_errors_pass_through():
    g = GATE_TYPE_TO_CLASS[GateType.rx]()
    g._targs, g._pargs = [0], ["x"]
    with pytest.raises((TypeError, ValueError)):
        gc.compile_gates([g], N)
    assert len(gc.compile_gates([], N)[0]) == 0


@pytest.mark.parametrize("single", [False, True])
def test_noisy_programs_made_at_once(single):
    """Channels whose Kraus operators are multiplied out together give the bits that
    they give one by one: the records of a noisy circuit are equal."""
    nm = qn.NoiseModel()
    nm.add(qn.DepolarizingError(0.05, 2), ["cx", "cz"])
    nm.add(qn.DampingError(0.1, 0.05, 0.2), ["h", "rx", "ry", "u1"])
    nm.add(qn.BitflipError(0.1), ["h", "s"], [0, 1])
    nm.add(qn.BitflipError(0.1).tensor(qn.PhaseflipError(0.2)), ["crz"])
    c = circuit(150, 8, single)
    (a, keep_a), (b, keep_b) = (program_records(nm.transpile(c, True, lazy=lazy).gates, N) for lazy in (False, True))
    for f in ("kind", "ncontrols", "ntargets", "bits", "m"):
        assert np.array_equal(a[f], b[f])
    wide = [[np.ctypeslib.as_array((nat.ctypes.c_double * (2 * 4 ** int(r["ntargets"]))).from_address(int(r["big"])))
             for r in x if r["big"]] for x in (a, b)]
    assert len(wide[0]) == len(wide[1]) and all(np.array_equal(x, y) for x, y in zip(*wide))
    # the channel's own Kraus operators are there when asked for
    eager, lazy = ([g for g in nm.transpile(c, True, lazy=z).gates if hasattr(g, "noise_matrix")] for z in (False, True))
    for x, y in zip(eager, lazy):
        assert x._precision == y._precision and all(np.array_equal(k, l) for k, l in zip(x.noise_matrix, y.noise_matrix))


@pytest.mark.parametrize("count", [0, 1, 2, 63, 1000, 20480])
def test_draws_in_one_call(count, monkeypatch):
    random.seed(count)
    want, after = [random.random() for _ in range(count)], random.random()
    random.seed(count)
    got = uniforms(count)
    assert got.dtype == np.float64 and got.tolist() == want and random.random() == after
    monkeypatch.setattr(random, "random", lambda: 0.25)  # a replaced generator is asked
    assert uniforms(count).tolist() == [0.25] * count
