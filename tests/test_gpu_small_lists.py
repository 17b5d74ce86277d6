"""Which lists on a register of at most a tile run as one launch, and that both ways
give the same state (tolerance: 8 roundings of half a unit in the last place a gate)."""
import ctypes
import random

import numpy as np
import pytest

from quict_amd import _native as nat
from quict_amd.core import CX, Circuit, H, Rz, Unitary
from quict_amd.simulation.gate_compiler import compile_gates

pytestmark = pytest.mark.gpu


def listing(n, simple, wide3, wide4):
    rng, r = random.Random(5), np.random.RandomState(5)
    kinds = [0] * simple + [3] * wide3 + [4] * wide4
    rng.shuffle(kinds)
    c = Circuit(n)
    for i, k in enumerate(kinds):
        if k:
            q, _ = np.linalg.qr(r.randn(1 << k, 1 << k) + 1j * r.randn(1 << k, 1 << k))
            Unitary(q) | c(rng.sample(range(n), k))
        else:
            g = [H, CX, Rz(0.3 + i)][i % 3]
            g | c(rng.sample(range(n), g.controls + g.targets))
    return compile_gates(c.gates, n)


@pytest.mark.parametrize("n", [5, 12])
@pytest.mark.parametrize("simple,wide3,wide4,one", [(6, 0, 0, (False, False)), (7, 0, 0, (True, True)),
                                                    (0, 20, 0, (False, False)), (9, 2, 0, (True, True)),
                                                    (8, 2, 0, (False, False)), (0, 0, 3, (False, True)),
                                                    (8, 0, 2, (False, True))])
def test_kernels_or_one_launch(n, simple, wide3, wide4, one):
    print("[case] small list", n, simple, wide3, wide4, flush=True)
    import torch
    lib, ctx, s = nat.load_library(), nat.context(0), nat.stream_ptr(0)
    recs, keep = listing(n, simple, wide3, wide4)
    gates, passes = nat.gate_array_ptr(recs), ctypes.c_int(0)
    for tdt, code, unit, single in ((torch.complex128, nat.QS_C128, 2.0 ** -53, one[0]),
                                    (torch.complex64, nat.QS_C64, 2.0 ** -24, one[1])):
        out = []
        for fuse in (0, 1):
            v = torch.empty(1 << n, dtype=tdt, device="cuda:0")
            nat.check(lib.qs_run(ctx, ctypes.c_void_p(v.data_ptr()), n, code, 0, gates, len(recs), fuse,
                                 ctypes.byref(passes), s))
            out.append(v)
        assert passes.value == (1 if single else len(recs))
        # (a gate's matrix in complex64 is rounded too)
        assert float((out[0] - out[1]).abs().max()) < 8 * unit * len(recs) * (1 if code == nat.QS_C128 else 2)
