"""Channels that compute their Kraus operators after a gate in their own way: the
density-matrix simulator's program holds what they return."""
import numpy as np

from quict_amd.core import CX, Circuit, H
from quict_amd.core.noise import BitflipError, NoiseModel
from quict_amd.simulation.density_matrix import program_records


class Twice(BitflipError):
    """Applies the gate twice."""

    def apply_to_gate(self, matrix):
        return [k @ matrix @ matrix for k in self.kraus]


def test_an_overridden_apply_to_gate_is_used():
    c = Circuit(3)
    for q in range(3):
        H | c(q)
    CX | c([0, 1])
    nm = NoiseModel()
    nm.add_noise_for_all_qubits(Twice(0.2), ["h"])
    eager, keep = program_records(nm.transpile(c, True).gates, 3)
    lazy, keep2 = program_records(nm.transpile(c, True, lazy=True).gates, 3)
    assert np.array_equal(eager["m"], lazy["m"])
