"""DensityMatrixSimulator on MI355X.

Drop-in for QuICT's ``DensityMatrixSimulator`` (QuICT/simulation/density_matrix/
density_matrix_simulator.py:14-240): ``run(circuit, density_matrix=None,
noise_model=None, use_previous=False)``, ``sample(shots)``, measure, the
``accumulated_mode`` option and readout errors.

Mechanism: the reference builds a dense 2^n x 2^n unitary per gate group and
multiplies rho <- U rho U^dagger with two cuBLAS GEMMs, and expands every Kraus
operator to 2^n x 2^n on the host (O(4^n) per operator).  Here rho (row-major,
entry (r, c) at index r*2^n + c) is treated as a 2n-bit vector:

  * a gate U on qubit q acts as U on row bit 2n-1-q and conj(U) on column bit
    n-1-q — two gate records that the fusion planner usually puts in the same
    tile pass, so each gate costs at most one read+write of rho;
  * a channel {K_i} on qubits A acts as the dense superoperator
    sum_i K_i (x) conj(K_i) on the 2|A| bits [row bits of A, column bits of A];
  * measurement: P0 from the diagonal, then rho <- P rho P / p.
"""
import ctypes
import random

import numpy as np

from ..core import BasicGate, Circuit, GateType, NoiseGate
from ..core import exception as qerr
from ..core.noise import NoiseModel
from .. import _native as nat
from .device_array import DeviceArray
from .gate_compiler import _translate, _write, superop_record, superop_write, superoperators
from .uniforms import uniforms


_NO_MATRIX = (GateType.id, GateType.barrier, GateType.measure, GateType.reset, GateType.perm)


class _Program:
    """Records of unitary gates and noise channels on the 2n-bit image of rho (row
    bits n..2n-1, column bits 0..n-1): a gate U is U on its row bits and conj(U) on its
    column bits; a channel is its superoperator.  A tensor-product channel applied
    after a gate (accumulated mode) is the gate's two records followed by one
    superoperator per single-qubit factor.

    A record without its bits depends on a matrix (or on a channel and a matrix) only,
    and a circuit repeats few of them: within one program each is made once, the
    superoperators of a channel all together."""

    def __init__(self, n: int):
        self.n = n
        self.keep: list = []
        self._templates = np.zeros(32, dtype=nat.QS_GATE_DTYPE)  # distinct records, bits unset
        self._count = 0
        self._rows: list = []        # template of each record ...
        self._bits: list = []        # ... and its bits
        self._memo: dict = {}
        self._channels: dict = {}    # id(channel) -> (channel, [template], [matrix])
        self._held: list = []        # objects whose ids are keys

    def _new(self) -> int:
        if self._count == len(self._templates):
            grown = np.zeros(2 * self._count, dtype=nat.QS_GATE_DTYPE)
            grown[: self._count] = self._templates
            self._templates = grown
        self._count += 1
        return self._count - 1

    def _put(self, template: int, bits: list):
        self._rows.append(template)
        self._bits.append(bits + [0] * (nat.QS_MAX_GATE_BITS - len(bits)))

    def add(self, g):
        if not isinstance(g, NoiseGate):
            self._unitary(g)
            return
        if g.source is not None:
            noise = g.source[1]
            factors = noise.factors
            if len(factors) > 1 and len(factors) == len(g.targs) and all(f.qubits == 1 for f in factors):
                self._unitary(g.source[0])
                self._held.append(noise)
                for f, q in zip(factors, g.targs):
                    self._superop(("factor", id(f)), f.kraus, [q])
                return
            if g.source_matrix is not None:
                self._after_gate(noise, g.source_matrix, list(g.targs))
                return
        self._superop(None, g.noise_matrix, list(g.targs))

    def _unitary(self, gate):
        n = self.n
        key = None
        if gate.params == 0 and gate.type not in _NO_MATRIX:
            m = np.asarray(gate.matrix)
            key = (id(gate.type), gate.controls, gate.targets, m.dtype.char, m.tobytes())
        pair = self._memo.get(key) if key else None
        if pair is None:
            r = _translate(gate, n, self.keep, n, False, False)
            if r is None:
                return
            kind, c, t, _, payload, big = r
            pair = (self._new(), self._new())
            _write(self._templates[pair[0]], (kind, c, t, (), payload, big))
            if big:
                payload, big = _translate(gate, n, self.keep, 0, True, False)[4:]
            else:
                payload = np.conj(payload)
            _write(self._templates[pair[1]], (kind, c, t, (), payload, big))
            if key:
                self._memo[key] = pair
        args = gate.cargs + gate.targs
        self._put(pair[0], [2 * n - 1 - a for a in args])
        self._put(pair[1], [n - 1 - a for a in args])

    def _channel_bits(self, args):
        return [2 * self.n - 1 - a for a in args] + [self.n - 1 - a for a in args]

    def _superop(self, key, kraus, args):
        t = self._memo.get(key) if key else None
        if t is None:
            t = self._new()
            superop_record(kraus, args, self.n, self._templates[t], self.keep)
            if key:
                self._memo[key] = t
        self._put(t, self._channel_bits(args))

    def _after_gate(self, noise, matrix, args):
        """A channel's Kraus operators times the gate's matrix: left to ``array``."""
        key = (id(noise), matrix.tobytes())
        t = self._memo.get(key)
        if t is None:
            t = self._memo[key] = self._new()
            _, ts, ms = self._channels.setdefault(id(noise), (noise, [], []))
            ts.append(t)
            ms.append(matrix)
        self._put(t, self._channel_bits(args))

    def array(self) -> np.ndarray:
        for noise, ts, ms in self._channels.values():
            K = np.matmul(np.asarray(noise.kraus)[None], np.stack(ms)[:, None])
            for t, S in zip(ts, superoperators(K)):
                superop_write(S, self._templates[t], self.keep)
        arr = self._templates[self._rows]
        arr["bits"] = self._bits
        return arr

    def __len__(self):
        return len(self._rows)


def program_records(ops, n: int):
    """Record array of a measurement-free list of gates and channels (the program
    the density-matrix simulator hands to qs_sv_apply_gates on 2n bits)."""
    prog = _Program(n)
    for g in ops:
        prog.add(g)
    return (prog.array() if len(prog) else np.zeros(0, dtype=nat.QS_GATE_DTYPE)), prog.keep


class DensityMatrixSimulator:
    def __init__(self, device: str = "GPU", precision: str = "double", accumulated_mode: bool = False,
                 gpu_device_id: int = 0, fusion: bool = True):
        if device != "GPU":
            raise qerr.ValueError("DensityMatrixSimulator.device must be 'GPU' (HIP only), got", device)
        if precision not in ("single", "double"):
            raise qerr.ValueError("DensityMatrixSimulator.precision must be single/double, got", precision)
        import torch
        self._torch = torch
        self._device = device
        self._device_id = gpu_device_id
        self._precision = np.complex128 if precision == "double" else np.complex64
        self._tdtype = torch.complex128 if precision == "double" else torch.complex64
        self._dcode = nat.QS_C128 if precision == "double" else nat.QS_C64
        self._accumulated_mode = accumulated_mode
        self._fusion = fusion
        self._density_matrix = None
        self._start = False   # rho stands for |0...0><0...0|, which is not written yet
        self._circuit = None
        self._noise_model = None
        self.last_passes = 0
        self._ctx = nat.context(gpu_device_id)
        self._lib = nat.load_library()

    @property
    def density_matrix(self) -> DeviceArray:
        D = 1 << self._qubits
        return DeviceArray(self._density_matrix, (D, D))

    def _stream(self):
        return nat.stream_ptr(self._device_id)

    def _rptr(self):
        return ctypes.c_void_p(self._density_matrix.data_ptr())

    def initial_circuit(self, circuit: Circuit, noise_model: NoiseModel):
        self._origin_circuit = circuit
        self._circuit = circuit if noise_model is None else self._noisy(noise_model, circuit)
        self._noise_model = noise_model
        self._qubits = int(circuit.width())

    def _noisy(self, noise_model, circuit: Circuit) -> Circuit:
        """The circuit with its channels; Kraus products on demand where ``transpile`` is
        the library's own (others take the two documented arguments)."""
        own = getattr(noise_model.transpile, "__func__", None) is NoiseModel.transpile
        return noise_model.transpile(circuit, self._accumulated_mode, **({"lazy": True} if own else {}))

    def initial_density_matrix(self, qubits: int):
        self._density_matrix = self._torch.empty(1 << (2 * qubits), dtype=self._tdtype,
                                                 device=f"cuda:{self._device_id}")
        self._start = True
        self._write_start(qubits)

    def _write_start(self, qubits: int):
        if self._start:
            self._start = False
            nat.check(self._lib.qs_sv_init(self._ctx, self._rptr(), 2 * qubits, self._dcode, 0, self._stream()),
                      "qs_sv_init")

    def check_matrix(self, matrix) -> bool:
        """density_matrix_simulator.py:70-86: Hermitian, PSD, unit trace."""
        m = np.asarray(matrix.get() if isinstance(matrix, DeviceArray) else matrix)
        if not np.allclose(m.T.conj(), m):
            raise qerr.SimulationMatrixError("density matrix must equal its conjugate transpose")
        ev = np.linalg.eigvalsh(m.astype(np.complex128))
        if np.any((ev < 0) & ~np.isclose(ev, 0, rtol=1e-4)):
            raise qerr.SimulationMatrixError("density matrix eigenvalues must be non-negative")
        if not np.isclose(np.trace(m), 1, rtol=1e-4):
            raise qerr.SimulationMatrixError("density matrix trace must be 1")
        return True

    def run(self, circuit: Circuit, density_matrix=None, noise_model: NoiseModel = None,
            use_previous: bool = False) -> DeviceArray:
        self.initial_circuit(circuit, noise_model)
        if density_matrix is not None:
            self.check_matrix(density_matrix)
            m = np.asarray(density_matrix.get() if isinstance(density_matrix, DeviceArray) else density_matrix)
            self._density_matrix = self._torch.as_tensor(m.astype(self._precision).ravel(),
                                                         device=f"cuda:{self._device_id}")
        elif self._density_matrix is None or not use_previous or \
                self._density_matrix.numel() != (1 << (2 * self._qubits)):
            own = DensityMatrixSimulator.initial_density_matrix
            if getattr(self.initial_density_matrix, "__func__", None) is own:
                self._density_matrix = self._torch.empty(1 << (2 * self._qubits), dtype=self._tdtype,
                                                         device=f"cuda:{self._device_id}")
                self._start = True
            else:  # a subclass's own start
                self.initial_density_matrix(self._qubits)
        self.last_passes = 0
        try:
            self._run(self._circuit)
        finally:
            self._write_start(self._qubits)
        if noise_model is not None:
            noise_model.apply_readout_error(circuit.qubits)
        self._torch.cuda.synchronize(self._device_id)
        return self.density_matrix

    def _run(self, circuit: Circuit):
        n = self._qubits
        prog = _Program(n)

        def flush():
            nonlocal prog
            if not len(prog):
                return
            arr = prog.array()
            passes = ctypes.c_int(0)
            args = (nat.gate_array_ptr(arr), len(arr), 1 if self._fusion else 0, ctypes.byref(passes), self._stream())
            if self._start:
                rc = self._lib.qs_run(self._ctx, self._rptr(), 2 * n, self._dcode, nat.QS_START_ZERO, *args)
                self._start = rc != nat.QS_OK
            else:
                rc = self._lib.qs_sv_apply_gates(self._ctx, self._rptr(), 2 * n, self._dcode, *args)
            nat.check(rc, "qs_sv_apply_gates(density matrix)")
            self.last_passes += passes.value
            prog = _Program(n)

        for g in circuit.gates:
            if isinstance(g, BasicGate) and g.type == GateType.measure:
                flush()
                self._write_start(n)
                self.apply_measure(g.targ)
            elif isinstance(g, BasicGate) and g.type in (GateType.reset, GateType.perm):
                raise qerr.GateTypeNotImplementError(f"{g.type.name} in the density-matrix simulator")
            elif isinstance(g, (BasicGate, NoiseGate)):
                prog.add(g)
            else:
                raise qerr.TypeError("DensityMatrixSimulator takes BasicGate / NoiseGate, got", type(g))
        flush()

    def apply_measure(self, index: int):
        """density_matrix_simulator.py:182-208 (``index`` is the qubit)."""
        n = self._qubits
        bit = n - 1 - index
        p0 = ctypes.c_double(0)
        nat.check(self._lib.qs_dm_prob_zero(self._ctx, self._rptr(), n, self._dcode, bit, ctypes.byref(p0),
                                            self._stream()), "qs_dm_prob_zero")
        prob0 = p0.value
        outcome = int(random.random() > prob0)
        p = (1 - prob0) if outcome else prob0
        nat.check(self._lib.qs_dm_collapse(self._ctx, self._rptr(), n, self._dcode, bit, outcome, 1.0 / p,
                                           self._stream()), "qs_dm_collapse")
        self._circuit.qubits[index].measured = outcome
        return outcome

    def diagonal(self) -> np.ndarray:
        n = self._qubits
        d = self._torch.empty(1 << n, dtype=self._torch.float64, device=f"cuda:{self._device_id}")
        nat.check(self._lib.qs_dm_diagonal(self._ctx, self._rptr(), n, self._dcode, ctypes.c_void_p(d.data_ptr()),
                                           self._stream()), "qs_dm_diagonal")
        return d.cpu().numpy()

    def trace(self) -> complex:
        re, im = ctypes.c_double(0), ctypes.c_double(0)
        nat.check(self._lib.qs_dm_trace(self._ctx, self._rptr(), self._qubits, self._dcode, ctypes.byref(re),
                                        ctypes.byref(im), self._stream()), "qs_dm_trace")
        return complex(re.value, im.value)

    def sample(self, shots: int) -> list:
        """density_matrix_simulator.py:210-240 for the accumulated / noiseless case:
        measure every qubit per shot (CPython ``random``), count, restore rho.
        Trajectory mode (noise without accumulated_mode) re-runs the noisy
        circuit per shot, as the reference does."""
        if self._density_matrix is None:
            raise qerr.SampleBeforeRunError("DensityMatrixSimulator sample without run any circuit.")
        n = self._qubits
        last = self._circuit.get_lastcall_for_each_qubits()
        measured = [i for i in range(n) if last[i] != GateType.measure]
        counts = [0] * (1 << n)
        if self._accumulated_mode or self._noise_model is None:
            if len(measured) == n and self._noise_model is None or (len(measured) == n and
                                                                     not self._noise_model._readout_errors):
                u = uniforms(shots * n)
                d = self._torch.empty(1 << n, dtype=self._torch.float64, device=f"cuda:{self._device_id}")
                nat.check(self._lib.qs_dm_diagonal(self._ctx, self._rptr(), n, self._dcode,
                                                   ctypes.c_void_p(d.data_ptr()), self._stream()), "qs_dm_diagonal")
                out = np.zeros(shots, dtype=np.uint64)
                nat.check(self._lib.qs_sample_probs(self._ctx, ctypes.c_void_p(d.data_ptr()), n,
                                                    u.ctypes.data_as(ctypes.c_void_p), shots,
                                                    out.ctypes.data_as(ctypes.c_void_p), self._stream()),
                          "qs_sample_probs")
                for v in out:
                    counts[int(v)] += 1
                if shots:
                    lastv = int(out[-1])
                    for q in range(n):
                        self._circuit.qubits[q].measured = (lastv >> (n - 1 - q)) & 1
                return counts
            original = self._density_matrix.clone()
            for _ in range(shots):
                for q in measured:
                    self.apply_measure(q)
                if self._noise_model is not None:
                    self._noise_model.apply_readout_error(self._circuit.qubits)
                counts[int(self._circuit.qubits)] += 1
                self._density_matrix.copy_(original)
            return counts
        for _ in range(shots):
            for q in measured:
                self.apply_measure(q)
            self._noise_model.apply_readout_error(self._circuit.qubits)
            counts[int(self._circuit.qubits)] += 1
            self.initial_density_matrix(n)
            noised = self._noisy(self._noise_model, self._origin_circuit)
            self._circuit = noised
            self._run(noised)
        return counts
