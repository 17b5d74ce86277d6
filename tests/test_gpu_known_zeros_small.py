"""qs_run of programs of several passes on registers below a tile, on the GPU, against
a program over an initialised vector: the same operations on the same numbers."""
import ctypes

import pytest

from quict_amd import _native as nat
from quict_amd.simulation.gate_compiler import compile_gates
from test_known_zeros_small import tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,start", [(3, 0), (5, 0), (8, 0), (11, 0), (3, 1), (5, 1)])
def test_several_passes_from_a_known_start(n, start):
    print("[case] small start", n, start, flush=True)
    import torch
    lib, ctx, s = nat.load_library(), nat.context(0), nat.stream_ptr(0)
    recs, keep = compile_gates(tables(n, 80).gates, n)
    bits = 2 * n if start else n
    gates, passes = nat.gate_array_ptr(recs), ctypes.c_int(0)
    for tdt, code in ((torch.complex128, nat.QS_C128), (torch.complex64, nat.QS_C64)):
        a = torch.full((1 << bits,), float("nan"), dtype=tdt, device="cuda:0")
        b = torch.empty_like(a)
        nat.check(lib.qs_run(ctx, ctypes.c_void_p(a.data_ptr()), bits, code, start, gates, len(recs), 1,
                             ctypes.byref(passes), s))
        assert passes.value > 1
        init = lib.qs_mat_identity if start else lambda c, v, m, d, st: lib.qs_sv_init(c, v, m, d, 0, st)
        nat.check(init(ctx, ctypes.c_void_p(b.data_ptr()), n, code, s))
        nat.check(lib.qs_sv_apply_gates(ctx, ctypes.c_void_p(b.data_ptr()), bits, code, gates, len(recs), 1, None, s))
        torch.cuda.synchronize()
        assert torch.equal(a, b), tdt
