"""Simulators that override where a run starts."""
import numpy as np
import pytest

from quict_amd import workloads
from quict_amd.simulation import DensityMatrixSimulator, StateVectorSimulator

pytestmark = pytest.mark.gpu


class LastState(StateVectorSimulator):
    def initial_state_vector(self, all_zeros=False):
        super().initial_state_vector(all_zeros)
        self._vector[0], self._vector[-1] = 0, 1


class LastMatrix(DensityMatrixSimulator):
    def initial_density_matrix(self, qubits):
        super().initial_density_matrix(qubits)
        self._density_matrix[0], self._density_matrix[-1] = 0, 1


@pytest.mark.parametrize("n", [5, 14])
def test_state_vector(n):
    print("[case] start override", n, flush=True)
    c = workloads.random_mix_circuit(n, 60, 2)
    v = np.zeros(1 << n, dtype=complex)
    v[-1] = 1
    assert np.array_equal(LastState("GPU").run(c).get(), StateVectorSimulator("GPU").run(c, state_vector=v).get())


def test_density_matrix():
    print("[case] start override dm", flush=True)
    c = workloads.random_mix_circuit(5, 30, 2)
    rho = np.zeros((32, 32), dtype=complex)
    rho[-1, -1] = 1
    assert np.array_equal(LastMatrix("GPU").run(c).get().ravel(),
                          DensityMatrixSimulator("GPU").run(c, density_matrix=rho).get().ravel())
