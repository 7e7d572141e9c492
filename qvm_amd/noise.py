"""Noisy pure-state evolution: stochastic Kraus maps and classical readout
noise, on the HBM-resident engine.

Mirrors the reference's noisy-qvm (src/noisy-qvm.lisp) for pure states:

    make_pauli_noise_map          src/noisy-qvm.lisp:46-67
    make_pauli_perturbed_1q_gate  src/noisy-qvm.lisp:69-78
    NoisyQVM.set_noisy_gate       src/noisy-qvm.lisp:80-84
    NoisyQVM.set_readout_povm     src/noisy-qvm.lisp:86-89
    evolve_pure_state_stochastically  src/apply-gate.lisp:16-39
    check_kraus_ops / check_povm  src/channel-qvm.lisp:109-135, 197-206
    perturb_measurement           src/channel-qvm.lisp:185-195

The Kraus choice of a 1- or 2-qubit map is one engine call: the running sum of
|K_j psi|^2 is compared with one uniform draw and the chosen operator is
applied in place, renormalised.  Wider maps need a second statevector of the
same size (the trial amplitudes): each candidate K_j is applied to a device
copy of the state, and the chosen trial buffer is swapped in.
"""
from __future__ import annotations

from typing import Dict, List, Sequence, Tuple

import numpy as np

from . import gates as G
from . import quil as Q
from .qvm import PureStateQVM, QVMError, apply_gate_to_state, method_chain
from .state import HipPureState


def check_kraus_ops(kraus_ops: Sequence[np.ndarray]) -> None:
    """Square, equal dimensions, sum_j K_j^H K_j = I within 1e-5."""
    ops = [np.asarray(k, dtype=np.complex128) for k in kraus_ops]
    if not ops:
        raise QVMError("empty Kraus map")
    m, n = ops[0].shape
    if m != n:
        raise QVMError("The Kraus operators be square matrices.")
    acc = np.zeros((m, n), dtype=np.complex128)
    for k in ops:
        if k.shape != (m, m):
            raise QVMError("All Kraus operators must have matching dimensions")
        acc += k.conj().T @ k
    if not np.allclose(acc, np.eye(m), atol=1e-5, rtol=0):
        raise QVMError("The Kraus map must preserve trace")


def check_povm(povm: Sequence[float]) -> None:
    """(p00 p01 p10 p11), each in [0, 1], columns summing to 1."""
    if len(povm) != 4:
        raise QVMError("a readout POVM is the list (p(0|0) p(0|1) p(1|0) p(1|1))")
    p00, p01, p10, p11 = (float(x) for x in povm)
    for p in (p00, p01, p10, p11):
        if not (0.0 <= p <= 1.0):
            raise QVMError("POVM entries must lie in [0, 1]")
    if abs(1.0 - (p00 + p10)) > 1e-10 or abs(1.0 - (p01 + p11)) > 1e-10:
        raise QVMError("POVM columns must sum to 1")


def make_pauli_noise_map(px: float, py: float, pz: float) -> List[np.ndarray]:
    """Kraus ops of rho -> (1-px-py-pz) rho + px X rho X + py Y rho Y + pz Z rho Z:
    sqrt(px) X, sqrt(py) Y, sqrt(pz) Z, then sqrt(1 - sum) I in front when the
    sum is below 1."""
    for p in (px, py, pz):
        if not (0.0 <= p <= 1.0):
            raise QVMError("Pauli probabilities must lie in [0, 1]")
    psum = px + py + pz
    if not (0.0 <= psum <= 1.0):
        raise QVMError("Pauli probabilities must sum to at most 1")
    ops = [np.sqrt(p) * G.gate_matrix(name) for name, p in (("X", px), ("Y", py), ("Z", pz))]
    if psum < 1:
        ops.insert(0, np.sqrt(1.0 - psum) * np.eye(2, dtype=np.complex128))
    return ops


def make_pauli_perturbed_1q_gate(gate_name: str, px: float, py: float, pz: float) -> List[np.ndarray]:
    """The ideal gate U followed by the Pauli noise map: K_j U for each K_j."""
    U = G.gate_matrix(gate_name)
    return [K @ U for K in make_pauli_noise_map(px, py, pz)]


def perturb_measurement(actual: int, p00: float, p01: float, p10: float, p11: float, r: float) -> int:
    """Recorded bit for true outcome ``actual`` and draw r: 0 iff r <= p(0|actual)."""
    if actual == 0:
        return 0 if r <= p00 else 1
    if actual == 1:
        return 0 if r <= p01 else 1
    raise QVMError("outcome must be a bit")


def evolve_pure_state_stochastically(state: HipPureState, trial: HipPureState, kraus_ops, quil_qubits,
                                     r: float) -> int:
    """Apply one Kraus operator of the map, chosen by inverse-transform
    sampling with the draw r: p_j = |K_j psi|^2 is added to a running sum until
    the sum reaches r; K_j psi, renormalised, becomes the state.  Maps on 1 or
    2 qubits read the state once for the p_j and apply the chosen operator in
    place; wider ones set the trial buffer (a state of the same size, or a
    function that gives one) to each K_j psi in turn.  Returns the index j chosen."""
    quil_qubits = list(quil_qubits)
    D = 1 << len(quil_qubits)
    if 2 <= D <= 4:
        kraus_ops = list(kraus_ops)
        ops = [np.asarray(K, dtype=np.complex128) for K in kraus_ops if np.shape(K) == (D, D)]
        # one that does not fit the qubits is refused below, when its turn comes
        if ops and len(ops) == len(kraus_ops):
            return state.apply_kraus_choice(np.stack(ops), G.nat_tuple(*quil_qubits), r)
    if callable(trial):
        trial = trial()
    summed = 0.0
    chosen = -1
    for j, K in enumerate(kraus_ops):
        trial.copy_from(state)
        apply_gate_to_state(trial, np.asarray(K, dtype=np.complex128), quil_qubits)
        summed += trial.total_probability()
        chosen = j
        if summed >= r:
            break
    state.swap_contents(trial)
    state.normalize()
    return chosen


def _unitary_weight(K: np.ndarray) -> float | None:
    """c where K is sqrt(c) times a unitary (2x2, c > 0, to a few roundings), else
    None."""
    (a, b), (c, d) = K.tolist()
    p = a.real * a.real + a.imag * a.imag + c.real * c.real + c.imag * c.imag
    q = b.real * b.real + b.imag * b.imag + d.real * d.real + d.imag * d.imag
    tol = 2.0 ** -49 * p  # 16 roundings
    if p > 0 and abs(p - q) <= tol and abs(a.conjugate() * b + c.conjugate() * d) <= tol:
        return 0.5 * (p + q)
    return None


class NoisyQVM(PureStateQVM):
    """noisy-qvm (src/noisy-qvm.lisp:7-26): a pure-state QVM whose gates may
    have noisy Kraus realisations and whose qubits may have readout POVMs.
    Programs are not compiled (src/noisy-qvm.lisp:145-152)."""

    def __init__(self, num_qubits: int, noisy_gate_definitions: Dict | None = None,
                 readout_povms: Dict | None = None, **kw):
        super().__init__(num_qubits, **kw)
        self.noisy_gate_definitions: Dict[Tuple[str, Tuple[int, ...]], List[np.ndarray]] = {}
        self.readout_povms: Dict[int, Tuple[float, float, float, float]] = {}
        self._trial: HipPureState | None = None
        for (name, qubits), ops in (noisy_gate_definitions or {}).items():
            self.set_noisy_gate(name, qubits, ops)
        for q, povm in (readout_povms or {}).items():
            self.set_readout_povm(q, povm)

    def _trial_state(self) -> HipPureState:
        # check-allocate-computation-space: the trial buffer is made on first need,
        # which maps on 1 and 2 qubits do not have (16 GiB at 30 qubits)
        if self._trial is None:
            self._trial = HipPureState(self.number_of_qubits, dtype=self.state.dtype)
        return self._trial

    def set_noisy_gate(self, gate_name: str, qubits, kraus_ops) -> None:
        ops = [np.asarray(k, dtype=np.complex128) for k in kraus_ops]
        check_kraus_ops(ops)
        self.noisy_gate_definitions[(gate_name.upper(), tuple(int(q) for q in qubits))] = ops

    def set_readout_povm(self, qubit: int, povm) -> None:
        check_povm(povm)
        self.readout_povms[int(qubit)] = tuple(float(x) for x in povm)

    def run(self) -> "NoisyQVM":
        # without noisy gates every step is the pure machine's; code that handles
        # instructions itself sees each of them
        if (self.program is None or self._compiled is not None or not self.noisy_gate_definitions
                or method_chain(self, "transition") != _TRANSITIONS):
            return super().run()
        code = self.program.executable_code
        self.pc = 0
        while self.pc is not None and self.pc < len(code):
            if not self._run_mixtures(code):
                self.pc = self.transition(code[self.pc])
        return self

    def _run_mixtures(self, code) -> bool:
        """Apply the 1-qubit gates from pc on in shared sweeps, as far as they
        are unitary or, where noisy, mixtures of unitaries (every operator
        sqrt(c_j) times a unitary, such as a Pauli channel after a gate), and
        advance pc.  |K_j psi|^2 is then c_j |psi|^2 whatever the state, so the
        choices need one read of the norm instead of one read per gate (24 qubits:
        47 us, and 73 us for the gate chosen).  The draws are taken in the
        program's order, before any of the run's gates is applied.  False, with
        nothing done and no draw taken, when fewer than two follow each other."""
        run = []
        for i in range(self.pc, len(code)):
            ins = code[i]
            if not isinstance(ins, Q.GateApplication) or len(ins.qubits) != 1:
                break
            q = ins.qubits[0]
            ops = self.noisy_gate_definitions.get((ins.name.upper(), (q,)))
            noisy = ops is not None
            if noisy:
                if ins.modifiers or ins.params:
                    break
            else:
                try:
                    ops = [Q.resolve_gate_matrix(ins, self.program.gate_definitions, self.memory)]
                except Exception:
                    break  # its own transition reports it
            if not ops or not 0 <= q < self.number_of_qubits or any(getattr(K, "shape", None) != (2, 2) for K in ops):
                break
            weights = [_unitary_weight(K) for K in ops]
            if None in weights or (not noisy and abs(weights[0] - 1) > 2.0 ** -49):
                break
            run.append((ops, weights if noisy else None, q))
        if len(run) < 2:
            return False
        norm2 = 1.0
        if any(w is not None for _, w, _ in run):
            norm2 = self.state.total_probability()
            if not 0.0 < norm2 < float("inf"):
                return False
        mats = []
        try:
            for ops, weights, q in run:
                if weights is None:
                    mats.append(ops[0])
                    continue
                r, summed = self._draw(), 0.0
                for K, c in zip(ops, weights):
                    summed += c * norm2
                    if summed >= r:
                        break
                mats.append(K / np.sqrt(c))
                norm2 = 1.0  # each noisy gate leaves a normalized state; the factor goes in at the end
        finally:
            # a draw that raises leaves the gates before its own applied
            done = run[:len(mats)]
            if done:
                self.state.apply_1q_run(mats, [q for _, _, q in done], any(w is not None for _, w, _ in done))
                self.pc += len(done)
        return True

    def transition(self, ins):
        if isinstance(ins, Q.GateApplication):
            key = (ins.name.upper(), tuple(ins.qubits))
            ops = self.noisy_gate_definitions.get(key)
            if ops is not None:
                if ins.modifiers:
                    raise QVMError("The noisy QVM doesn't support gate modifiers.")
                if ins.params:
                    raise QVMError("noisy gate definitions apply to static gates only")
                if ops[0].shape[0] != 1 << len(ins.qubits):
                    raise QVMError(f"Kraus operators of {ins.name} do not match its qubit count")
                evolve_pure_state_stochastically(self.state, self._trial_state, ops, ins.qubits, self._draw())
                return self.pc + 1
            return super().transition(ins)
        if isinstance(ins, Q.Measure):
            nxt = super().transition(ins)
            # classical readout noise on the stored bit (src/channel-qvm.lisp:173-183)
            if ins.target is not None and ins.qubit in self.readout_povms:
                name, idx = ins.target
                c = int(self.memory[name][idx])
                self.memory[name][idx] = perturb_measurement(c, *self.readout_povms[ins.qubit], self._draw())
            return nxt
        return super().transition(ins)

    def measure_all(self):
        """measure-all with each bit passed through its POVM
        (perturb-measured-bits, src/measurement.lisp:228-243)."""
        qvm, bits = super().measure_all()
        out = []
        for i, c in enumerate(bits):
            povm = self.readout_povms.get(i)
            out.append(perturb_measurement(c, *povm, self._draw()) if povm else c)
        return qvm, out

    def compile_loaded_program(self, *a, **kw):
        return None

    def close(self) -> None:
        if self._trial is not None:
            self._trial.close()
            self._trial = None
        super().close()


_TRANSITIONS = method_chain(NoisyQVM, "transition")
