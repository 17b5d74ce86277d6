"""qs_run on the GPU against qs_sv_init / qs_mat_identity followed by
qs_sv_apply_gates: the same operations on the same numbers, so equal results, in
buffers that held NaN before; both planners, tile shapes, the prefetching kernel,
gates that run as their own kernel between passes."""
import ctypes

import numpy as np
import pytest

from quict_amd import _native as nat
from quict_amd import workloads
from quict_amd.core import CX, Circuit, H, QFT, X
from quict_amd.simulation.gate_compiler import compile_gates

pytestmark = pytest.mark.gpu


def few(n):
    c = Circuit(n)
    X | c(n - 1)
    H | c(0)
    CX | c([0, n - 2])
    return c


def own_kernel(n):
    c = workloads.random_mix_circuit(n, 30, 4)
    QFT(5) | c([0, 2, 4, 6, 8])
    CX | c([1, n - 1])
    return c


def empty(n):
    return Circuit(n)


CIRCUITS = {"few": few, "mix": lambda n: workloads.random_mix_circuit(n, 200, 9), "own kernel": own_kernel,
            "empty": empty}


@pytest.mark.parametrize("env", [None, "0"])
@pytest.mark.parametrize("tile,low,prefetch", [(0, 0, 0), (13, 3, 0), (0, 0, 1)])
@pytest.mark.parametrize("name", list(CIRCUITS))
@pytest.mark.parametrize("n,start", [(10, 0), (13, 0), (19, 0), (24, 0), (9, 1), (10, 1)])
def test_run_equals_init_and_apply(n, start, name, tile, low, prefetch, env, monkeypatch):
    print("[case] qs_run", n, start, name, tile, low, prefetch, env, flush=True)
    import torch
    if env is not None:
        monkeypatch.setenv("QS_FUSION_REMAP", env)
    lib, ctx, s = nat.load_library(), nat.context(0), nat.stream_ptr(0)
    recs, keep = compile_gates(CIRCUITS[name](n).gates, n)
    bits = 2 * n if start else n
    nat.check(lib.qs_set_fusion(ctx, tile, low))
    nat.check(lib.qs_set_fusion_launch(ctx, prefetch, 2))
    try:
        for tdt, code in ((torch.complex128, nat.QS_C128), (torch.complex64, nat.QS_C64)):
            a = torch.full((1 << bits,), float("nan"), dtype=tdt, device="cuda:0")
            b = torch.empty_like(a)
            for fuse in (0, 1):
                nat.check(lib.qs_run(ctx, ctypes.c_void_p(a.data_ptr()), bits, code, start, nat.gate_array_ptr(recs),
                                     len(recs), fuse, None, s))
                if start:
                    nat.check(lib.qs_mat_identity(ctx, ctypes.c_void_p(b.data_ptr()), n, code, s))
                else:
                    nat.check(lib.qs_sv_init(ctx, ctypes.c_void_p(b.data_ptr()), n, code, 0, s))
                nat.check(lib.qs_sv_apply_gates(ctx, ctypes.c_void_p(b.data_ptr()), bits, code,
                                                nat.gate_array_ptr(recs), len(recs), fuse, None, s))
                torch.cuda.synchronize()
                assert torch.equal(a, b), (tdt, fuse)
                a.fill_(float("nan"))
    finally:
        nat.check(lib.qs_set_fusion(ctx, 0, 0))
        nat.check(lib.qs_set_fusion_launch(ctx, 0, 2))


def test_refused():
    lib, ctx = nat.load_library(), nat.context(0)
    import torch
    v = torch.zeros(1 << 7, dtype=torch.complex128, device="cuda:0")
    for bits, start in ((7, 1), (7, 2), (7, -1)):
        assert lib.qs_run(ctx, ctypes.c_void_p(v.data_ptr()), bits, nat.QS_C128, start, None, 0, 1, None,
                          None) == nat.QS_ERR_ARG
