"""Gates that cancel within one program, on the GPU: planned passes against the
per-gate kernels.  Tolerance: a gate rounds an amplitude at most four times, half a
unit in the last place of the state's norm each, on either side; complex64 gates come
rounded to single precision, which adds as much again."""
import pytest

from quict_amd import _native as nat
from quict_amd.simulation.gate_compiler import compile_gates
from test_cancelling_gates import CASES
from test_gpu_wires import both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [nat.QS_C128, nat.QS_C64], ids=["c128", "c64"])
@pytest.mark.parametrize("n", [5, 14, 19])
@pytest.mark.parametrize("name", list(CASES))
def test_gates_that_cancel(name, n, dtype):
    print("[case] cancelling", name, n, dtype, flush=True)
    c = CASES[name](n)
    if dtype == nat.QS_C64:
        c.convert_precision()
    recs, keep = compile_gates(c.gates, n)
    unit = 2.0 ** -53 if dtype == nat.QS_C128 else 2 * 2.0 ** -24
    assert both(recs, n, dtype, 2) < 8 * unit * len(recs)
