"""Tile passes planned in wires on the GPU against the per-gate kernels (fuse=0).

The records cover every op of k_wires: rotations, phases of each kind, general
complex and controlled 2x2, exchanges under register / thread / tile controls,
tables with zero entries, dense gates on 2 to 4 targets, controlled swaps.
Tolerances: 1e-12 max-abs (complex128, the suite's bar for a few hundred gates),
1e-5 for complex64 (two hundred gates of a few 1e-8 each).
"""
import ctypes
import random

import numpy as np
import pytest

from quict_amd import _native as nat
from quict_amd.simulation.gate_compiler import compile_gates
from test_wire_planner import hea, qft, random_types, wide

pytestmark = pytest.mark.gpu


def free_records(n, count, seed):
    """Records with free payloads: non-unitary, zero and non-unit entries included."""
    rng, r = random.Random(seed), np.random.RandomState(seed)
    recs, keep = np.zeros(count, dtype=nat.QS_GATE_DTYPE), []
    kinds = [nat.GATE_XPERM, nat.GATE_PHASE, nat.GATE_DIAG, nat.GATE_XPERM, nat.GATE_SWAP, nat.GATE_DENSE]
    for i in range(count):
        kind = kinds[i % 6]
        nt = {nat.GATE_PHASE: 1, nat.GATE_DIAG: rng.choice([1, 2, 3]), nat.GATE_XPERM: 1, nat.GATE_SWAP: 2,
              nat.GATE_DENSE: rng.choice([1, 1, 2, 3, 4])}[kind]
        nc = 0 if i % 6 == 0 else rng.choice([0, 0, 1, 2, 5])
        recs[i]["kind"], recs[i]["ncontrols"], recs[i]["ntargets"] = kind, nc, nt
        recs[i]["bits"][: nc + nt] = rng.sample(range(n), nc + nt)
        m = r.uniform(0.8, 1.1, 16) * np.exp(1j * r.uniform(0, 6, 16))
        if i % 6 == 0:
            m[:2] = 1
        elif i % 7 == 0:
            m[rng.randrange(2)] = 0
        if kind == nat.GATE_DENSE:
            q, _ = np.linalg.qr(r.randn(1 << nt, 1 << nt) + 1j * r.randn(1 << nt, 1 << nt))
            q = q * (1.05 if i % 4 else 1.0) if nt == 1 else q
            if nt <= 2:
                m[: 1 << (2 * nt)] = q.ravel()
            else:
                keep.append(np.ascontiguousarray(q).view(np.float64).ravel().copy())
                recs[i]["big"] = keep[-1].ctypes.data
        recs[i]["m"][:] = m.view(np.float64)
    return recs, keep


def both(recs, n, dtype, fuse):
    import torch
    lib, ctx, s = nat.load_library(), nat.context(0), nat.stream_ptr(0)
    rng = np.random.RandomState(1)
    x = rng.randn(1 << n) + 1j * rng.randn(1 << n)
    x /= np.linalg.norm(x)
    out = []
    for f in (0, fuse):
        v = torch.as_tensor(x, device="cuda:0").to(torch.complex128 if dtype == nat.QS_C128 else torch.complex64)
        nat.check(lib.qs_sv_apply_gates(ctx, ctypes.c_void_p(v.data_ptr()), n, dtype, nat.gate_array_ptr(recs),
                                        len(recs), f, None, s))
        out.append(v.cpu().numpy())
    return float(np.max(np.abs(out[0] - out[1])) / max(1.0, np.max(np.abs(out[0]))))


@pytest.mark.parametrize("dtype,tol", [(nat.QS_C128, 1e-12), (nat.QS_C64, 1e-5)], ids=["c128", "c64"])
@pytest.mark.parametrize("case", ["free", "types", "wide", "hea", "qft"])
@pytest.mark.parametrize("n", [13, 16])
def test_wires_match_per_gate_kernels(case, n, dtype, tol):
    print("[case] wires", case, n, dtype, flush=True)
    if case == "free":
        recs, keep = free_records(n, 120, 5)
    else:
        c = {"types": lambda: random_types(n, 250, 4), "wide": lambda: wide(n, 3), "hea": lambda: hea(n, 4, 1),
             "qft": lambda: qft(n)}[case]()
        recs, keep = compile_gates(c.gates, n)
    assert both(recs, n, dtype, 2) < tol


@pytest.mark.parametrize("dtype,tol", [(nat.QS_C128, 1e-12), (nat.QS_C64, 1e-5)], ids=["c128", "c64"])
@pytest.mark.parametrize("n", [5, 6, 9, 11, 12])
def test_registers_within_one_tile(n, dtype, tol):
    """Fewer amplitudes than a tile: one launch, nothing outside the register written."""
    import torch
    print("[case] wires small", n, dtype, flush=True)
    recs, keep = compile_gates(random_types(n, 150, n).gates, n)
    assert both(recs, n, dtype, 1) < tol
    if n >= 9:
        recs, keep = free_records(n, 60, n)
        assert both(recs, n, dtype, 1) < tol
    lib, ctx, s = nat.load_library(), nat.context(0), nat.stream_ptr(0)
    v = torch.zeros(1 << 13, dtype=torch.complex128 if dtype == nat.QS_C128 else torch.complex64, device="cuda:0")
    v[1 << n:] = 7
    v[0] = 1
    recs, keep = compile_gates(random_types(n, 40, n).gates, n)
    nat.check(lib.qs_sv_apply_gates(ctx, ctypes.c_void_p(v.data_ptr()), n, dtype, nat.gate_array_ptr(recs), len(recs),
                                    1, None, s))
    assert bool((v[1 << n:] == 7).all()) and abs(float(torch.linalg.vector_norm(v[: 1 << n])) - 1) < 1e-5


@pytest.mark.parametrize("shape,dtype", [((11, 4), nat.QS_C128), ((13, 4), nat.QS_C128), ((13, 5), nat.QS_C64),
                                         ((12, 8), nat.QS_C64), ((12, 2), nat.QS_C128)])
def test_wires_in_other_tile_shapes(shape, dtype):
    print("[case] wires tile", shape, dtype, flush=True)
    lib, ctx = nat.load_library(), nat.context(0)
    n = 15
    recs, keep = free_records(n, 90, 8)
    types, keep2 = compile_gates(random_types(n, 150, 6).gates, n)
    nat.check(lib.qs_set_fusion(ctx, *shape))
    try:
        assert both(recs, n, dtype, 1) < (1e-12 if dtype == nat.QS_C128 else 1e-5)
        assert both(types, n, dtype, 1) < (1e-12 if dtype == nat.QS_C128 else 1e-5)
    finally:
        lib.qs_set_fusion(ctx, 0, 0)
