"""Diagonal gates and exchanges with entries far from modulus 1 on the GPU: planned
passes against the per-gate kernels, 8 roundings of half a unit in the last place of
the largest amplitude a gate (complex64: the entries are rounded too)."""
import pytest

from quict_amd import _native as nat
from test_gpu_wires import both
from test_wire_nonunit import CASES, records

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [12, 14])
@pytest.mark.parametrize("name", list(CASES))
def test_entries_far_from_one(name, n):
    print("[case] entries", name, n, flush=True)
    one = records(name)
    recs = one[list(range(len(one))) * 7]  # (a small register's list from seven gates on is planned)
    for dtype, unit in ((nat.QS_C128, 2.0 ** -53), (nat.QS_C64, 2 * 2.0 ** -24)):
        assert both(recs, n, dtype, 2) < 8 * unit * len(recs)
