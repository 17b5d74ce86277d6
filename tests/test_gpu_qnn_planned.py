"""Batches of variational circuits at the edges of their layouts.  complex128, planned
passes: circuits narrower than a tile (several to a tile, the last tile padded),
exactly one tile, wider ones.  complex64, a workgroup a circuit: the widths where the
state moves from LDS to device memory and the launch shape changes, widths that leave
1, 2 and 3 qubits to the last sweep.  More features than qubits and fewer, one layer
and many, uneven targets.

Reference: the same circuits with their own gate programs (a workgroup a circuit,
one rotation at a time).  Tolerance: both apply at most 2 * 2 * 20 * 8 rotations to
unit vectors in 64 bits, so <Z_0> and the gradients of the mean loss (terms of order
1 for targets of order 1) differ by less than 1e-12.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


CASES = [
    ([2], 1, 1),
    ([2, 3, 2, 3, 2], 5, 2),
    ([12], 12, 3),
    ([11, 12, 13, 11], 16, 4),
    ([13] * 3 + [4] * 70 + [8] * 17, 3, 2),
    ([16, 15, 2, 12, 12, 9], 20, 8),
    ([18, 17], 40, 2),
    ([20], 7, 1),
]


@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("widths,nfeat,layers", CASES + [([14, 13, 12, 11, 10, 5] * 60, 6, 2)])
def test_against_gate_programs(widths, nfeat, layers, precision):
    print("[case] qnn batch", widths[:6], nfeat, layers, precision, flush=True)
    from quict_amd.gradient.qnn import QNNBatch, QNNProgramBatch, circuit_for
    rng = np.random.RandomState(len(widths) + nfeat)
    n, mw = len(widths), max(widths)
    x = rng.randn(n, nfeat)
    t = rng.uniform(-1.5, 1.5, n)
    theta = rng.uniform(-np.pi, np.pi, layers * 2 * mw)
    got = QNNBatch(np.array(widths, dtype=np.int32), x, t, layers=layers, max_width=mw,
                   precision=precision).forward_backward(theta)
    circuits = [circuit_for(w, np.zeros(0), layers, mw) for w in widths]
    encode = [[(j % w, j) for j in range(nfeat)] for w in widths]
    want = QNNProgramBatch(circuits, x, t, nparams=theta.size, encode=encode).forward_backward(theta)
    tol = 1e-12 if precision == "double" else 16 * 2 * mw * layers * 2.0 ** -24
    for g, w in zip(got, want):
        assert np.max(np.abs(np.asarray(g) - np.asarray(w))) < tol
