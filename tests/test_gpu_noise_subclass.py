"""Noise models that override ``transpile`` with its two documented arguments."""
import numpy as np
import pytest

from quict_amd import workloads
from quict_amd.core.noise import NoiseModel

pytestmark = pytest.mark.gpu


class Counting(NoiseModel):
    calls = 0

    def transpile(self, circuit, accumulated_mode=False):
        type(self).calls += 1
        return super().transpile(circuit, accumulated_mode)


@pytest.mark.parametrize("accumulated", [True, False])
def test_an_overridden_transpile_is_called(accumulated):
    print("[case] noise subclass", accumulated, flush=True)
    import random
    from quict_amd.simulation import DensityMatrixSimulator
    c = workloads.random_mix_circuit(4, 30, 2)
    plain = workloads.dm_noise_model()
    model = workloads.dm_noise_model()
    model.__class__ = Counting
    Counting.calls = 0
    out = []
    for nm in (plain, model):
        random.seed(4)
        sim = DensityMatrixSimulator("GPU", accumulated_mode=accumulated)
        rho = sim.run(c, noise_model=nm).get()
        out.append((rho, sim.sample(20)))
    assert Counting.calls > 0
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
