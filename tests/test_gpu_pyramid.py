"""The sampling pyramid where its launches split (eleven levels each): outcomes of
qs_sample_probs and qs_sv_sample against the same pair sums and the same descent in
numpy.  Same sums in 64 bits, same comparisons: the outcomes are equal."""
import ctypes

import numpy as np
import pytest

from quict_amd import _native as nat

pytestmark = pytest.mark.gpu


def descend(p, u):
    levels = [p]
    while len(levels[-1]) > 1:
        levels.append(levels[-1][0::2] + levels[-1][1::2])
    node = np.zeros(len(u), dtype=np.int64)
    for q, level in enumerate(levels[-2::-1]):
        left, right = level[2 * node], level[2 * node + 1]
        tot = left + right
        p0 = np.where(tot > 0, left / np.where(tot > 0, tot, 1.0), 1.0)
        node = 2 * node + (u[:, q] > p0)
    return node


@pytest.mark.parametrize("n", [1, 2, 10, 11, 12, 13, 21, 22, 23])
@pytest.mark.parametrize("shots", [1, 300])
def test_outcomes(n, shots):
    print("[case] pyramid", n, shots, flush=True)
    import torch
    rng = np.random.RandomState(n)
    lib, ctx, s = nat.load_library(), nat.context(0), nat.stream_ptr(0)
    p = rng.rand(1 << n)
    p[rng.rand(1 << n) < 0.3] = 0.0
    p[0] = 0.5
    u = rng.rand(shots, n)
    out = np.zeros(shots, dtype=np.uint64)
    d = torch.as_tensor(p, device="cuda:0")
    nat.check(lib.qs_sample_probs(ctx, ctypes.c_void_p(d.data_ptr()), n, u.ctypes.data, shots, out.ctypes.data, s))
    assert np.array_equal(out.astype(np.int64), descend(p, u))
    # powers of two: |a|^2 is exact in both precisions
    a = 2.0 ** -rng.randint(0, 9, 1 << n)
    for tdt, code in ((torch.complex128, nat.QS_C128), (torch.complex64, nat.QS_C64)):
        v = torch.as_tensor(a * np.exp(0.5j * np.pi * rng.randint(0, 2, 1 << n)).round(), device="cuda:0").to(tdt)
        nat.check(lib.qs_sv_sample(ctx, ctypes.c_void_p(v.data_ptr()), n, code, u.ctypes.data, shots, out.ctypes.data, s))
        assert np.array_equal(out.astype(np.int64), descend(a * a, u))
