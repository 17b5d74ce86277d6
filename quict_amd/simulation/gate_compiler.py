"""Translate QuICT-style gates into ``qs_gate`` records for the HIP library.

This replaces the dispatch of StateVectorSimulator.apply_gate
(QuICT/simulation/state_vector/statevector_simulator.py:202-496), which picks a
kernel by (MatrixType, #controls, #targets) and passes reversed qubit indices
(``n-1-q``).  Here the same decision produces a compact record instead:

  MatrixType            record kind   payload
  diagonal / diag_diag  DIAG          last 2^t diagonal entries (the all-controls-one block)
  control               PHASE         matrix[-1, -1]
  swap, 1 target (X)    XPERM         (1, 1)
  swap, 2 targets       SWAP          target block [1, 2], [2, 1]
  reverse               XPERM         matrix[-2, -1], matrix[-1, -2]
  everything else       DENSE         target block (controls folded in as controls)

Gate arguments are ``cargs + targs`` with argument 0 the most significant bit
of the gate-matrix index, mapped to amplitude bit ``n-1-q``.
"""
import ctypes
import os
from typing import List, Tuple

import numpy as np

from ..core import BasicGate, GateType, MatrixType
from .. import _native as nat

_NON_UNITARY = (GateType.measure, GateType.reset, GateType.barrier, GateType.perm)


_OFFDIAG = {}


def _is_diag(m: np.ndarray) -> bool:
    d = m.shape[0]
    mask = _OFFDIAG.get(d)
    if mask is None:
        mask = _OFFDIAG[d] = ~np.eye(d, dtype=bool)
    return not m[mask].any()


def _controlled_split(mat: np.ndarray, nargs: int) -> Tuple[int, np.ndarray]:
    """Largest c such that mat = I on every block except the last 2^(nargs-c) one."""
    d = 1 << nargs
    for c in range(nargs - 1, 0, -1):
        t = nargs - c
        blk = 1 << t
        top = mat[: d - blk, : d - blk]
        if (np.array_equal(top, np.identity(d - blk, dtype=mat.dtype))
                and not np.any(mat[: d - blk, d - blk:]) and not np.any(mat[d - blk:, : d - blk])):
            return c, mat[d - blk:, d - blk:]
    return 0, mat


def _translate(gate: BasicGate, n: int, keep: list, row_offset: int, conj: bool, dagger: bool):
    """(kind, ncontrols, ntargets, bits, payload, big) of one gate, or None for
    gates with no effect.  ``payload`` is a complex128 vector (inline
    coefficients) or None; ``big`` the address of a wider matrix kept in ``keep``."""
    gt = gate.type
    if gt in (GateType.id, GateType.barrier):
        return None
    if gt in _NON_UNITARY:
        raise ValueError(f"{gt.name} is not a unitary gate record")
    args = list(gate.cargs) + list(gate.targs)
    bits = [row_offset + n - 1 - a for a in args]
    mat = np.asarray(gate.matrix, dtype=np.complex128)
    if conj:
        mat = mat.conj()
    if dagger:
        mat = mat.conj().T
    nargs = len(args)
    mt = gate.matrix_type
    c, t = gate.controls, gate.targets

    if gt == GateType.unitary and c == 0:
        # classify by structure (a Unitary carries no controls of its own)
        cc, blk = _controlled_split(mat, nargs)
        c, t = cc, nargs - cc
        mat_t = blk
        mt = MatrixType.diagonal if (_is_diag(mat_t) and t <= 4) else MatrixType.normal
        full_diag = np.diag(mat_t)
    else:
        mat_t = mat[-(1 << t):, -(1 << t):]
        full_diag = None

    if mt in (MatrixType.diagonal, MatrixType.diag_diag) and t <= 4:
        d = np.diag(mat)[-(1 << t):] if full_diag is None else full_diag
        if t == 1 and d[0] == 1:
            return nat.GATE_PHASE, c, t, bits, d[1:2], 0
        return nat.GATE_DIAG, c, t, bits, d, 0
    if mt == MatrixType.control:
        return nat.GATE_PHASE, c, t, bits, mat[-1:, -1], 0
    if mt == MatrixType.swap and t == 1:
        return nat.GATE_XPERM, c, t, bits, np.array([mat_t[0, 1], mat_t[1, 0]]), 0
    if mt == MatrixType.swap and t == 2:
        return nat.GATE_SWAP, c, t, bits, np.array([mat_t[1, 2], mat_t[2, 1]]), 0
    if mt == MatrixType.reverse:
        # reverse-classified gate (also a multi-target unitary): controls are all args but the last
        return nat.GATE_XPERM, nargs - 1, 1, bits, np.array([mat[-2, -1], mat[-1, -2]]), 0
    # dense target block; a diagonal block becomes DIAG / PHASE
    if t <= 4 and _is_diag(mat_t):
        d = np.diag(mat_t)
        if np.all(d[:-1] == 1):
            return nat.GATE_PHASE, c, t, bits, d[-1:], 0
        return nat.GATE_DIAG, c, t, bits, d, 0
    if t <= 2:
        return nat.GATE_DENSE, c, t, bits, mat_t.ravel(), 0
    big = np.ascontiguousarray(mat_t).view(np.float64).ravel().copy()
    keep.append(big)
    return nat.GATE_DENSE, c, t, bits, None, big.ctypes.data


def compile_gate(gate: BasicGate, n: int, rec: np.ndarray, keep: list, row_offset: int = 0,
                 conj: bool = False, dagger: bool = False) -> bool:
    """Fill one QS_GATE_DTYPE record.  Returns False for gates with no effect (id, barrier).

    ``row_offset`` shifts the amplitude bits (used for the row half of a
    density matrix); ``conj`` conjugates the matrix (column half);
    ``dagger`` writes the inverse (conjugate transpose).
    """
    r = _translate(gate, n, keep, row_offset, conj, dagger)
    if r is None:
        return False
    _write(rec, r)
    return True


# Gate types that the native helper turns into records: rotations, in its order, whose
# payloads it computes, and parameter-free types of fixed shape, whose record depends
# only on the type and precision.
_ROTATION_TYPES = (GateType.rx, GateType.ry, GateType.rz, GateType.crz, GateType.u1, GateType.cu1, GateType.u3)
_STATIC_TYPES = (
    GateType.h, GateType.hy, GateType.s, GateType.sdg, GateType.x, GateType.y, GateType.z, GateType.sx,
    GateType.sy, GateType.sw, GateType.t, GateType.tdg, GateType.cx, GateType.cy, GateType.cz, GateType.ch,
    GateType.swap, GateType.iswap, GateType.iswapdg, GateType.sqiswap, GateType.cswap, GateType.ccx,
    GateType.ccz)
_RECORDS_LIB = None  # (function, types, prototypes), set on first use


def _static_prototypes() -> np.ndarray:
    """Records of the fixed types, each in complex128 and complex64, bits unset."""
    protos = np.zeros(2 * len(_STATIC_TYPES), dtype=nat.QS_GATE_DTYPE)
    for i, gt in enumerate(_STATIC_TYPES):
        gate = BasicGate(_type=gt)
        gate._cargs, gate._targs = list(range(gate.controls)), list(range(gate.controls, gate.controls + gate.targets))
        for single in (0, 1):
            compile_gate(gate, gate.controls + gate.targets, protos[2 * i + single], [])
            gate.convert_precision()
    protos["bits"] = 0
    return protos


def _records_lib():
    global _RECORDS_LIB
    if _RECORDS_LIB is None:
        if not os.path.exists(nat.RECORDS_PATH):
            raise nat.qerr.NativeRuntimeError(f"{nat.RECORDS_PATH} is missing: build it with `make -C quict_amd/csrc`")
        fn = ctypes.PyDLL(nat.RECORDS_PATH).gate_records
        fn.restype = ctypes.c_int
        O, P = ctypes.py_object, ctypes.c_void_p
        fn.argtypes = [O, O, O, O, O, P, ctypes.c_int, P, P]
        _RECORDS_LIB = (fn, _ROTATION_TYPES + _STATIC_TYPES, _static_prototypes())
    return _RECORDS_LIB


def _write(rec, r):
    kind, c, t, bits, payload, big = r
    rec["kind"], rec["ncontrols"], rec["ntargets"] = kind, c, t
    rec["bits"][:] = 0
    rec["bits"][: len(bits)] = bits
    rec["m"][:] = 0
    if payload is not None:
        v = np.ascontiguousarray(payload, dtype=np.complex128).view(np.float64)
        rec["m"][: len(v)] = v
    rec["big"] = big


def _write_rows(arr, rows, translate) -> list:
    """Writes the records of the gates numbered ``rows`` and returns the numbers of those
    without one.  Through plain views of the array: a field of a structured record costs
    as much to reach as the record to write (200 two-qubit matrices 4.5 -> 3.6 ms)."""
    G, size = len(arr), arr.dtype.itemsize
    words, doubles = arr.view(np.int32).reshape(G, size // 4), arr.view(np.float64).reshape(G, size // 8)
    m0, big = arr.dtype.fields["m"][1] // 8, arr["big"]
    drop = []
    for k in rows:
        r = translate(k)
        if r is None:
            drop.append(k)
            continue
        kind, c, t, bits, payload, address = r
        doubles[k] = 0
        words[k, : 3 + len(bits)] = [kind, c, t] + bits
        if payload is not None:
            v = np.ascontiguousarray(payload, dtype=np.complex128).view(np.float64)
            doubles[k, m0: m0 + len(v)] = v
        if address:
            big[k] = address
    return drop


def compile_gates(gates: List[BasicGate], n: int, row_offset: int = 0, conj: bool = False,
                  dagger: bool = False) -> Tuple[np.ndarray, list]:
    """Records for a run of unitary gates; ``keep`` holds arrays referenced by pointer.
    The native helper fills the records of fixed gate types and of rotations (plain
    records only: no row offset, conjugation or inverse); the rest goes through
    _translate."""
    keep: list = []
    gates = list(gates)
    G = len(gates)
    arr = np.empty(G, dtype=nat.QS_GATE_DTYPE)
    if row_offset == 0 and not conj and not dagger:
        fn, types, protos = _records_lib()
        left = np.empty(G, dtype=np.int32)
        nleft = fn(gates, BasicGate, types, np.complex128, np.complex64, protos.ctypes.data, n, arr.ctypes.data,
                   left.ctypes.data)
        rest = left[:nleft].tolist()
    else:
        rest = range(G)
    drop = _write_rows(arr, rest, lambda k: _translate(gates[k], n, keep, row_offset, conj, dagger)) if len(rest) else []
    if drop:
        arr = np.delete(arr, drop)
    return arr, keep


def superoperators(K: np.ndarray) -> np.ndarray:
    """sum_k K_k (x) conj(K_k) of channels with Kraus operators K[channel, k]:
    S[(a, c), (b, e)] = sum_k K_k[a, b] conj(K_k[c, e])."""
    d = K.shape[-1]
    return np.einsum("nkab,nkce->nacbe", K, K.conj()).reshape(-1, d * d, d * d)


def superop_write(S: np.ndarray, rec, keep: list):
    """S as a dense record, bits unset."""
    v = np.ascontiguousarray(S).view(np.float64).ravel()
    t = S.shape[0].bit_length() - 1
    rec["kind"], rec["ncontrols"], rec["ntargets"] = nat.GATE_DENSE, 0, t
    rec["bits"][:] = 0
    rec["m"][:] = 0
    rec["big"] = 0
    if t <= 2:
        rec["m"][: len(v)] = v
    else:
        big = v.copy()
        keep.append(big)
        rec["big"] = big.ctypes.data


def superop_record(kraus: List[np.ndarray], args: List[int], n: int, rec, keep: list):
    """Record for a channel sum_k K (.) K^dagger on density-matrix qubits ``args``:
    dense superoperator sum_k K (x) conj(K) on [row bits..., column bits...]."""
    d = 1 << len(args)
    superop_write(superoperators(np.asarray(kraus, dtype=np.complex128).reshape(1, -1, d, d))[0], rec, keep)
    rec["bits"][: 2 * len(args)] = [2 * n - 1 - a for a in args] + [n - 1 - a for a in args]
