"""The planner in wires (quict_amd/csrc/qsim_wire_plan.hpp) on the CPU.

tests/planner/emu_wires.cpp runs the planner's exact programs: tile predicates,
phases, relayouts and stores that apply pending CX maps, stores that move qubits.
The results must match the C restatement of the reference kernels to 1e-12 from
a random state, over the gate forms and tile shapes the fused calls take.
"""
import ctypes
import os
import random
import subprocess

import numpy as np
import pytest

from quict_amd import _native as nat
from quict_amd import workloads
from quict_amd.core import (CCX, CH, CRz, CSwap, CU1, CX, CY, Circuit, FSim, H, QFT, Rx, Rxx, Ry, Rz, Rzz, S, Swap, T,
                            Unitary, X, Y, Z)
from quict_amd.simulation.gate_compiler import compile_gates
from test_oracle import ALL_TYPES

HERE = os.path.dirname(os.path.abspath(__file__))
SHAPES = {"c128": (4, 8, 16), "c64": (4, 8, 8), "c128-k11": (4, 7, 16), "c128-k13": (4, 9, 16)}


@pytest.fixture(scope="module")
def emu():
    subprocess.run(["make", "-s", "-C", os.path.join(HERE, "planner")], check=True)
    lib = ctypes.CDLL(os.path.join(HERE, "planner", "_build", "libplanner_wires.so"))
    P, I = ctypes.c_void_p, ctypes.c_int
    lib.wires_apply.argtypes = [P, I, P, I, I, I, I, I, P]
    lib.wires_last_error.restype = ctypes.c_char_p
    return lib


def check(lib, recs, n, shape="c128", L=4, seed=0, tol=1e-12):
    """Runs the records both ways from a random state; returns the plan's counts."""
    rng = np.random.RandomState(seed)
    v = rng.randn(1 << n) + 1j * rng.randn(1 << n)
    v /= np.linalg.norm(v)
    ref, st = v.copy(), np.zeros(8, dtype=np.int32)
    lib.cpu_apply_gates(ref.ctypes.data_as(ctypes.c_void_p), n, nat.gate_array_ptr(recs), len(recs), 4)
    RB, TB, S_ = SHAPES[shape]
    rc = lib.wires_apply(v.ctypes.data_as(ctypes.c_void_p), n, nat.gate_array_ptr(recs), len(recs), RB, TB, L, S_,
                         st.ctypes.data_as(ctypes.c_void_p))
    assert rc == 0, lib.wires_last_error()
    assert np.max(np.abs(v - ref)) < tol
    return st


def random_types(n, ngates, seed, types=None):
    c = Circuit(n)
    random.seed(seed)
    np.random.seed(seed)
    c.random_append(ngates, typelist=types or ALL_TYPES, random_params=True)
    return c


def hea(n, layers, seed):
    return workloads.hea_circuit(n, workloads.hea_params(n, layers, seed))


def qft(n):
    c = Circuit(n)
    for q in range(n):
        H | c(q)
        for j in range(q + 1, n):
            CU1(np.pi / (1 << (j - q))) | c([j, q])
    return c


def wide(n, seed):
    """Multi-controlled, wide dense, Toffoli and exchange gates among flips."""
    rng, r = random.Random(seed), np.random.RandomState(seed)
    c = Circuit(n)
    for i in range(60):
        k = rng.choice([1, 2, 3, 3, 4, 5, 6])
        u, _ = np.linalg.qr(r.randn(1 << k, 1 << k) + 1j * r.randn(1 << k, 1 << k))
        if i % 3 == 0:  # controlled on every qubit but the last one or two
            m = np.eye(1 << (k + 2), dtype=complex)
            m[-(1 << min(k, 2)):, -(1 << min(k, 2)):] = u[: 1 << min(k, 2), : 1 << min(k, 2)] if k <= 2 else np.eye(4)[::-1]
            Unitary(m) | c(rng.sample(range(n), k + 2))
        elif i % 3 == 1:
            Unitary(u) | c(rng.sample(range(n), k))
        else:
            (CCX if i % 2 else CSwap) | c(rng.sample(range(n), 3))
        for g in (X, Y, H):
            g | c(rng.randrange(n))
        FSim(0.1 * i, 0.3) | c(rng.sample(range(n), 2))
        CY | c(rng.sample(range(n), 2))
        CH | c(rng.sample(range(n), 2))
    return c


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("n,ngates,seed", [(14, 60, 1), (15, 300, 2), (17, 500, 3)])
def test_all_gate_types(emu, shape, n, ngates, seed):
    recs, keep = compile_gates(random_types(n, ngates, seed).gates, n)
    check(emu, recs, n, shape)


@pytest.mark.parametrize("shape", ["c128", "c64", "c128-k11"])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 8, 11, 12])
def test_registers_within_one_tile(emu, shape, n):
    types = [t for t in ALL_TYPES if n >= 3 or t.name in ("h", "x", "y", "s", "rx", "rz", "u3") or
             (n == 2 and t.name in ("cx", "cz", "swap", "crz"))]
    recs, keep = compile_gates(random_types(n, 120, n, types).gates, n)
    st = check(emu, recs, n, shape)
    assert n > 11 or st[0] == 1 or shape == "c128-k11"
    if n >= 6:
        c = random_types(n, 30, n)
        u, _ = np.linalg.qr(np.random.RandomState(n).randn(32, 32))
        Unitary(u.astype(complex)) | c(random.Random(n).sample(range(n), 5))
        Swap | c([0, n - 1])
        X | c(1)
        for g in random_types(n, 30, n + 1).gates:
            c.append(g)
        recs, keep = compile_gates(c.gates, n)
        check(emu, recs, n, shape)


@pytest.mark.parametrize("L", [2, 3, 5, 8])
def test_low_bit_counts(emu, L):
    recs, keep = compile_gates(random_types(16, 300, 5).gates, 16)
    check(emu, recs, 16, L=L)


@pytest.mark.parametrize("shape", ["c128", "c64"])
@pytest.mark.parametrize("seed", range(3))
def test_clifford_relabelings(emu, shape, seed):
    """CX, CY, X, Y, Swap, CZ and few mixing gates: most of it addresses only."""
    rng = random.Random(seed)
    c = random_types(16, 40, seed)
    from quict_amd.core import CZ, iSwap
    for _ in range(400):
        g = rng.choice([CX, CX, CX, CY, X, Y, Swap, CZ, S, T, Z, iSwap, H])
        g | c(rng.sample(range(16), g.controls + g.targets))
    recs, keep = compile_gates(c.gates, 16)
    check(emu, recs, 16, shape, seed=seed)


@pytest.mark.parametrize("seed", range(2))
def test_wide_gates(emu, seed):
    recs, keep = compile_gates(wide(16, seed).gates, 16)
    check(emu, recs, 16, seed=seed, tol=1e-11)


@pytest.mark.parametrize("shape", ["c128", "c64"])
def test_two_bit_diagonals_and_pauli_rotations(emu, shape):
    rng = random.Random(7)
    c = Circuit(15)
    for i in range(200):
        g = rng.choice([Rxx, Rzz, CRz, CU1, Rx, Ry, Rz, X])
        (g(rng.uniform(0, 6)) if g is not X else g) | c(rng.sample(range(15), g.controls + g.targets))
    recs, keep = compile_gates(c.gates, 15)
    check(emu, recs, 15, shape)


def test_noise_superoperators(emu):
    from quict_amd.simulation.density_matrix import program_records
    n = 8
    c = workloads.random_mix_circuit(n, 80, 12)
    recs, keep = program_records(workloads.dm_noise_model().transpile(c, True).gates, n)
    check(emu, recs, 2 * n)


def test_records_the_front_end_does_not_make(emu):
    """Zero and non-unit diagonal entries, exchanges with zero phases, phases on
    many bits, all under flips: what a caller of the C interface may pass."""
    rng, r = random.Random(3), np.random.RandomState(3)
    n = 15
    recs = np.zeros(160, dtype=nat.QS_GATE_DTYPE)
    for i in range(len(recs)):
        kind = [nat.GATE_XPERM, nat.GATE_PHASE, nat.GATE_DIAG, nat.GATE_XPERM, nat.GATE_SWAP, nat.GATE_DENSE][i % 6]
        nt = {nat.GATE_PHASE: 1, nat.GATE_DIAG: rng.choice([1, 2, 3]), nat.GATE_XPERM: 1, nat.GATE_SWAP: 2,
              nat.GATE_DENSE: rng.choice([1, 2])}[kind]
        nc = 0 if i % 6 == 0 else rng.choice([0, 1, 2, 5])
        recs[i]["kind"], recs[i]["ncontrols"], recs[i]["ntargets"] = kind, nc, nt
        recs[i]["bits"][: nc + nt] = rng.sample(range(n), nc + nt)
        m = r.uniform(0.7, 1.1, 16) * np.exp(1j * r.uniform(0, 6, 16)) / (2 if kind == nat.GATE_DENSE else 1)
        if i % 6 == 0:
            m[:2] = 1
        elif i % 7 == 0:
            m[rng.randrange(2)] = 0
        recs[i]["m"][:] = m.view(np.float64)
    check(emu, recs, n)


def test_fewer_passes_than_whole_gates_in_the_tile(emu):
    """What the planner is for: passes of the 2000-gate workload at 26 qubits and of
    a hardware-efficient ansatz, and phases outside the tile."""
    st = np.zeros(8, dtype=np.int32)

    def plan(c, n):
        recs, keep = compile_gates(c.gates, n)
        assert emu.wires_apply(None, n, nat.gate_array_ptr(recs), len(recs), 4, 8, 4, 16,
                               st.ctypes.data_as(ctypes.c_void_p)) == 0, emu.wires_last_error()
        return int(st[0])

    assert plan(workloads.sv30_circuit(n=26), 26) < 30
    assert plan(hea(25, 8, 1), 25) < 10
    assert plan(qft(24), 24) < 8
    recs, keep = compile_gates(QFT(4).gates if hasattr(QFT(4), "gates") else hea(16, 1, 1).gates, 16)
    check(emu, compile_gates(qft(16).gates, 16)[0], 16)
    check(emu, compile_gates(hea(16, 6, 2).gates, 16)[0], 16)


def variational(n, nops, seed, hea_layers=0):
    """(axis, bit, slot) per gate and the fixed gates: random rotations among CX, X,
    Swap, CZ, H, Toffoli, or the hardware-efficient ansatz."""
    from quict_amd.core import CZ, GateType
    from quict_amd.gradient.adjoint import ParameterizedCircuit
    rng = random.Random(seed)
    if hea_layers:
        return ParameterizedCircuit.hea(n, hea_layers)
    pc = ParameterizedCircuit(n)
    k = 0
    for _ in range(nops):
        t = rng.choice([GateType.rx, GateType.ry, GateType.rz, GateType.rx, GateType.cx, GateType.x, GateType.swap,
                        GateType.cz, GateType.h, GateType.ccx, GateType.s])
        nq = {GateType.cx: 2, GateType.swap: 2, GateType.cz: 2, GateType.ccx: 3}.get(t, 1)
        rot = t in (GateType.rx, GateType.ry, GateType.rz)
        pc.add(t, rng.sample(range(n), nq), param=(k if rng.random() < 0.8 else rng.randrange(k + 1)) if rot else None)
        k += rot
    return pc


@pytest.mark.parametrize("n,nops,seed,layers", [(13, 90, 1, 0), (14, 140, 2, 0), (13, 0, 3, 2), (5, 60, 4, 0),
                                                (8, 0, 5, 3)])
def test_sweep_programs_give_the_shift_gradient(emu, n, nops, seed, layers):
    """Planned forward program, planned inverse with gradient columns: the state, the
    state swept back and d<Z>/d theta by the parameter-shift rule (two terms per gate
    occurrence, so parameters used twice count twice)."""
    from quict_amd.core import GateType
    from quict_amd.gradient.adjoint import _records
    pc = variational(n, nops, seed, layers)
    theta = np.random.RandomState(seed).uniform(-7, 7, pc.nparams)
    fwd, inv, _, slot, keep = _records(pc, theta)
    axes = {GateType.rx: 0, GateType.ry: 1, GateType.rz: 2}
    axis = np.array([axes[t] if p is not None else -1 for t, _, p, _ in pc.ops], dtype=np.int32)
    bit = np.array([n - 1 - q[-1] for _, q, _, _ in pc.ops], dtype=np.int32)
    zbit, N = n - 2, 1 << n
    state, back, grads, st = np.zeros(N, complex), np.zeros(N, complex), np.zeros(pc.nparams), np.zeros(2, np.int32)
    ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    rc = emu.wires_gradient(n, len(pc.ops), ptr(axis), ptr(bit), ptr(slot), nat.gate_array_ptr(fwd),
                            nat.gate_array_ptr(inv), ptr(theta), zbit, 16, ptr(state), ptr(back), ptr(grads), ptr(st))
    assert rc == 0, emu.wires_last_error()

    def run(recs):
        v = np.zeros(N, complex)
        v[0] = 1
        emu.cpu_apply_gates(ptr(v), n, nat.gate_array_ptr(recs), len(recs), 4)
        return v

    sign = 1 - 2.0 * ((np.arange(N) >> zbit) & 1)
    energy = lambda recs: float(np.sum(sign * np.abs(run(recs)) ** 2))
    ref = run(fwd)
    assert abs(abs(np.vdot(ref, state)) - 1) < 1e-12
    assert abs(back[0]) > 1 - 1e-12
    from quict_amd.simulation.gate_compiler import compile_gate
    want = np.zeros(pc.nparams)
    rotations = [j for j in range(len(pc.ops)) if axis[j] >= 0]
    check_ = set(random.Random(0).sample(rotations, min(len(rotations), 12)))
    by_slot = {}
    for j in rotations:
        by_slot.setdefault(int(slot[j]), []).append(j)
    for s, js in by_slot.items():
        if not check_ & set(js):
            continue
        for j in js:
            for sh, w in ((np.pi / 2, 0.5), (-np.pi / 2, -0.5)):
                r = fwd.copy()
                t2 = theta.copy()
                t2[s] += sh
                compile_gate(pc.gate(j, t2), n, r[j], keep)
                want[s] += w * energy(r)
        assert abs(grads[s] - want[s]) < 1e-11
