"""Bytes that the fused passes read and write (qs_profile_bytes)."""
import ctypes

import pytest

from quict_amd import _native as nat
from quict_amd import workloads
from quict_amd.core import Circuit, H
from quict_amd.simulation.gate_compiler import compile_gates

pytestmark = pytest.mark.gpu


def moved(lib, ctx):
    b = ctypes.c_double(0)
    nat.check(lib.qs_profile_bytes(ctx, ctypes.byref(b), 1))
    return b.value


@pytest.mark.parametrize("dtype", [nat.QS_C128, nat.QS_C64])
def test_bytes_of_the_passes(dtype):
    import torch
    n, amp = 16, 16 if dtype == nat.QS_C128 else 8
    print("[case] profile bytes", n, dtype, flush=True)
    lib, ctx, s = nat.load_library(), nat.context(0), nat.stream_ptr(0)
    v = torch.zeros(1 << n, dtype=torch.complex128 if amp == 16 else torch.complex64, device="cuda:0")
    ptr, passes = ctypes.c_void_p(v.data_ptr()), ctypes.c_int(0)
    recs, keep = compile_gates(workloads.random_mix_circuit(n, 200, 1).gates, n)
    one = Circuit(n)  # one tile of the first pass holds anything: written, not read
    for q in range(n - 8, n):
        H | one(q)
    first, keep1 = compile_gates(one.gates, n)
    nat.check(lib.qs_profile_enable(ctx, 1))
    try:
        moved(lib, ctx)
        nat.check(lib.qs_sv_apply_gates(ctx, ptr, n, dtype, nat.gate_array_ptr(recs), len(recs), 1,
                                        ctypes.byref(passes), s))
        whole = passes.value * 2 * (1 << n) * amp
        assert moved(lib, ctx) == whole and moved(lib, ctx) == 0
        nat.check(lib.qs_run(ctx, ptr, n, dtype, 0, nat.gate_array_ptr(recs), len(recs), 1, ctypes.byref(passes), s))
        assert 0 < moved(lib, ctx) < passes.value * 2 * (1 << n) * amp
        nat.check(lib.qs_run(ctx, ptr, n, dtype, 0, nat.gate_array_ptr(first), len(first), 1, ctypes.byref(passes), s))
        assert passes.value == 1 and moved(lib, ctx) == 4096 * amp
    finally:
        nat.check(lib.qs_profile_enable(ctx, 0))
        ms, cnt = (ctypes.c_double * 4)(), (ctypes.c_int64 * 4)()
        nat.check(lib.qs_profile_read(ctx, ms, cnt, 1))
