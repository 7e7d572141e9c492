"""The interpreters' shared sweeps (several instructions as one engine call)
on a stand-in for the engine state: who still sees each instruction, and what a
failure in the middle leaves behind."""
import numpy as np
import pytest

from qvm_amd import density, gates as G, noise, qvm


class StandIn:
    """Records the engine calls of a machine."""
    made = 0

    def __init__(self, num_qubits, dtype="f64", **kw):
        StandIn.made += 1
        self.num_qubits, self.dtype, self.calls = num_qubits, dtype, []

    def total_probability(self):
        return 1.0

    def apply_1q_run(self, mats, qubits, normalize=False):
        self.calls.append(("run", len(mats)))
        self.normalized = normalize

    def density_apply_kraus_run(self, nq, maps):
        self.calls.append(("run", len(maps)))

    def apply_matrix(self, U, qubits):
        self.calls.append(("gate", 1))

    def apply_kraus_choice(self, kraus_ops, qubits, r):
        self.calls.append(("choice", 1))
        return 0

    def density_apply_kraus(self, nq, kraus_ops, qubits):
        self.calls.append(("map", 1))

    def copy_from(self, other):
        pass

    def swap_contents(self, other):
        self.calls += other.calls

    def normalize(self):
        pass

    def close(self):
        pass


MIX = [np.sqrt(0.75) * G.gate_matrix("X"), 0.5 * G.gate_matrix("Z") @ G.gate_matrix("X")]
TEXT = "X 0\nH 1\nX 0\nCNOT 0 1\nH 0\nX 0\n"


@pytest.fixture
def machine(monkeypatch):
    for module in (qvm, noise, density):
        monkeypatch.setattr(module, "HipPureState", StandIn)

    def make(cls, rng=lambda: 0.1, text=TEXT):
        m = cls(2, noisy_gate_definitions={("X", (0,)): MIX}, rng=rng)
        m.load_program(text)
        return m
    return make


@pytest.mark.parametrize("base", [noise.NoisyQVM, density.DensityQVM])
def test_machines_without_hooks_share_sweeps(machine, base):
    m = machine(base)
    m.run()
    assert [c for c in m.state.calls if c[0] == "run"] == [("run", 3), ("run", 2)] and m.pc == 6


@pytest.mark.parametrize("base", [noise.NoisyQVM, density.DensityQVM])
@pytest.mark.parametrize("way", ["subclass", "instance", "wrapped class", "wrapped base", "mixin"])
def test_every_instruction_reaches_a_hook(machine, monkeypatch, base, way):
    seen = []
    own = qvm.PureStateQVM if base is noise.NoisyQVM and way in ("wrapped base", "mixin") else base
    plain = own.transition

    def hook(self, ins):
        seen.append(ins)
        return plain(self, ins)

    cls = base
    if way == "subclass":
        cls = type("Sub", (base,), {"transition": hook})
    elif way == "mixin":
        if base is density.DensityQVM:
            pytest.skip("no base class to mix in behind")
        cls = type("Mixed", (base, type("Tracer", (qvm.PureStateQVM,), {"transition": hook})), {})
    m = machine(cls)
    if way == "instance":
        m.transition = hook.__get__(m)
    elif way.startswith("wrapped"):
        monkeypatch.setattr(own, "transition", hook)
    m.run()
    # the pure machine's transition sees what the noisy one passes on
    assert len(seen) == (3 if own is qvm.PureStateQVM else 6)
    assert not [c for c in m.state.calls if c[0] == "run"]


@pytest.mark.parametrize("name", ["_kraus_ops", "apply_superoperator"])
def test_every_map_reaches_a_hook(machine, monkeypatch, name):
    seen = []
    plain = getattr(density.DensityQVM, name)
    monkeypatch.setattr(density.DensityQVM, name, lambda self, *a: seen.append(a) or plain(self, *a))
    machine(density.DensityQVM).run()
    assert len(seen) == 6


@pytest.mark.parametrize("good,pc,normalized", [(0, 1, False), (1, 3, True), (2, 5, True)])
def test_a_draw_that_raises_leaves_the_gates_before_it_applied(machine, good, pc, normalized):
    """H 0, X 0 (noisy), H 1, X 0 (noisy), H 1, X 0 (noisy): the draw of the
    gate at pc raises."""
    draws = iter([0.1] * good)
    m = machine(noise.NoisyQVM, rng=lambda: next(draws), text="H 0\nX 0\nH 1\nX 0\nH 1\nX 0\n")
    with pytest.raises(StopIteration):
        m.run()
    assert m.pc == pc and m.draws_used == good + 1
    assert m.state.calls == [("run", pc)] and m.state.normalized == normalized


def test_kraus_evolution_takes_any_iterable():
    """Operators and qubits as generators; an operator of another size behind
    the chosen one is never reached."""
    one, two = MIX, [np.kron(K, np.eye(2)) for K in MIX]
    for ops, qubits, call in ((one, [0], "choice"), (two, [1, 0], "choice"), ([one[0], np.eye(4)], [0], "gate"),
                              ([np.eye(8)], [0, 1, 2], "gate")):
        st = StandIn(3)
        assert noise.evolve_pure_state_stochastically(st, StandIn(3), (K for K in ops), (q for q in qubits), 0.5) == 0
        assert st.calls == [(call, 1)]


def test_the_second_statevector_is_made_for_wide_maps_only(machine):
    """Noisy gates on 1 and 2 qubits, alone and in runs, work in place; the
    first one on 3 qubits makes the trial buffer, the next one finds it."""
    StandIn.made = 0
    m = machine(noise.NoisyQVM)
    m.set_noisy_gate("CNOT", [0, 1], [G.gate_matrix("CNOT")])
    m.run()
    assert ("choice", 1) in m.state.calls and StandIn.made == 1
    wide = noise.NoisyQVM(3, noisy_gate_definitions={("CCNOT", (0, 1, 2)): [G.gate_matrix("CCNOT")]})
    assert StandIn.made == 2
    wide.load_program("CCNOT 0 1 2\nCCNOT 0 1 2\n")
    wide.run()
    assert StandIn.made == 3
    wide.close()
