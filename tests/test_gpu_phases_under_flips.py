"""Multi-controlled phases between layers of X (Grover diffusions) on the GPU: planned
passes against the per-gate kernels, 8 roundings of half a unit in the last place of
the state's norm a gate."""
import pytest

from quict_amd import _native as nat
from quict_amd.core import Circuit
from quict_amd.simulation.gate_compiler import compile_gates
from test_gpu_wires import both
from test_wire_plan_sizes import all_ones_phase

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(5, 3), (9, 8), (14, 4), (14, 10), (17, 6)])
def test_diffusions(n, k):
    print("[case] diffusion", n, k, flush=True)
    c = Circuit(n)
    for _ in range(3):
        for g in all_ones_phase(n, k, True).gates:
            c.append(g)
    recs, keep = compile_gates(c.gates, n)
    assert both(recs, n, nat.QS_C128, 2) < 8 * 2.0 ** -53 * len(recs)
    assert both(recs, n, nat.QS_C64, 2) < 8 * 2.0 ** -24 * 2 * len(recs)
