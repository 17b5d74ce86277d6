"""Gates that cancel within one program, on the CPU model of the planned passes.

One-qubit gates on a wire are multiplied together, so a gate and its inverse become a
matrix that is diagonal up to rounding: the phases of its off-diagonal entries mean
nothing.  Tolerance: a gate rounds an amplitude at most four times, 2^-53 of the
state's norm each, on either side.
"""
import random

import numpy as np
import pytest

from quict_amd.core import CX, Circuit, H, Rx, Ry, Rz, SX, T, T_dagger, U3
from quict_amd.simulation.gate_compiler import compile_gates
from test_wire_planner import check, emu  # noqa: F401  (the fixture)

ANGLES = [0.0, 1e-1, 1e-3, 1e-5, 1e-7, 1e-9, 1e-12, 1e-15]


def on(n, wire, gates):
    c = Circuit(n)
    for g in gates:
        g | c(wire)
    return c


def named(n, name):
    t = {"H T Td H": [H, T, T_dagger, H], "H Td T H": [H, T_dagger, T, H], "H T T SX": [H, T, T, SX],
         "SX T T H": [SX, T, T, H], "H T^8 H": [H] + 8 * [T] + [H], "H Rz Rz H": [H, Rz(0.7), Rz(-0.7), H]}
    return on(n, n // 2, t[name])


def euler(n, seed, count=12):
    """Random U3, then Rx Rz Ry, each followed by its inverse, on random qubits."""
    rng = random.Random(seed)
    c = Circuit(n)
    for i in range(count):
        a = [rng.uniform(-7, 7) for _ in range(3)]
        g = [U3(*a)] if i % 2 else [Rx(a[0]), Rz(a[1]), Ry(a[2])]
        q = rng.randrange(n)
        for k in g + [k.inverse() for k in reversed(g)]:
            k | c(q)
    return c


def residual(n, angle):
    """A gate, a rotation by a small angle and the gate's inverse, on three qubits."""
    c = Circuit(n)
    for q, mid in ((0, Rx), (n // 2, Ry), (n - 1, Rx)):
        for k in (U3(0.4 + q, 0.9, 1.3), mid(angle), U3(0.4 + q, 0.9, 1.3).inverse()):
            k | c(q)
    return c


def echo(n, seed, cx):
    """Random one-qubit gates (with CX among them) and the inverse circuit."""
    rng = random.Random(seed)
    gates = []
    for _ in range(60):
        if cx and rng.random() < 0.3:
            gates.append((CX, rng.sample(range(n), 2)))
            continue
        g = rng.choice([H, T, SX, Rx, Ry, Rz, U3])
        if g in (Rx, Ry, Rz):
            g = g(rng.uniform(-7, 7))
        elif g is U3:
            g = g(*[rng.uniform(-7, 7) for _ in range(3)])
        gates.append((g, [rng.randrange(n)]))
    c = Circuit(n)
    for g, q in gates + [(g.inverse(), q) for g, q in reversed(gates)]:
        g | c(q)
    return c


CASES = {f"named {k}": (lambda n, k=k: named(n, k)) for k in
         ("H T Td H", "H Td T H", "H T T SX", "SX T T H", "H T^8 H", "H Rz Rz H")}
CASES.update({f"euler {s}": (lambda n, s=s: euler(n, s)) for s in range(3)})
CASES.update({f"residual {a:g}": (lambda n, a=a: residual(n, a)) for a in ANGLES})
CASES.update({f"echo {s} {cx}": (lambda n, s=s, cx=cx: echo(n, s, cx)) for s in range(2) for cx in (False, True)})


@pytest.mark.parametrize("shape", ["c128", "c64"])
@pytest.mark.parametrize("n", [5, 14])
@pytest.mark.parametrize("name", list(CASES))
def test_gates_that_cancel(emu, name, n, shape):  # noqa: F811
    recs, keep = compile_gates(CASES[name](n).gates, n)
    check(emu, recs, n, shape, tol=8 * 2.0 ** -53 * len(recs))


def test_products_with_one_zero_off_the_diagonal(emu):  # noqa: F811
    """A matrix whose entry 01 is exactly 0 and 10 is rounding, and the other way round."""
    from quict_amd import _native as nat
    for i in (1, 2):
        for d in ([1, 1j], [0.6 + 0.8j, -1]):
            m = np.zeros(4, dtype=complex)
            m[0], m[3], m[i] = d[0], d[1], 1e-17j
            recs = np.zeros(1, dtype=nat.QS_GATE_DTYPE)
            recs[0]["kind"], recs[0]["ntargets"], recs[0]["bits"][0] = nat.GATE_DENSE, 1, 2
            recs[0]["m"][:8] = m.view(np.float64)
            check(emu, recs, 13, tol=8 * 2.0 ** -53)
