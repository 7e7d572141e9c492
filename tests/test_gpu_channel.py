"""GPU tests of the noise channels: the density superoperator against dense
numpy Kraus sums."""
import numpy as np
import pytest

from qvm_amd import gates as G

pytestmark = pytest.mark.gpu


def kraus_list(count, k, rng):
    """Random Kraus operators: the blocks of an isometry."""
    D = 1 << k
    A = rng.normal(size=(count * D, D)) + 1j * rng.normal(size=(count * D, D))
    return np.linalg.qr(A)[0].reshape(count, D, D)


def embed(K, qubits, n):
    """K (index bit j <-> qubits[j]) as a 2^n x 2^n matrix."""
    idx = np.arange(1 << n)
    sub = sum(((idx >> q) & 1) << j for j, q in enumerate(qubits))
    rest = idx & ~sum(1 << q for q in qubits)
    return np.where(rest[:, None] == rest[None, :], K[sub[:, None], sub[None, :]], 0)


@pytest.mark.parametrize("dtype,n,k,count", [("f64", 1, 1, 2), ("f64", 2, 1, 1), ("f64", 2, 2, 3), ("f64", 5, 1, 4),
                                             ("f64", 5, 2, 1), ("f64", 5, 2, 16), ("f64", 4, 3, 2),
                                             ("f64", 7, 1, 3), ("f64", 7, 2, 2), ("f32", 5, 1, 4), ("f32", 7, 2, 2)])
def test_density_superoperator_matches_kraus_sum(dtype, n, k, count):
    """Against sum_j K_j rho K_j^H in numpy, entries of order 2^-n.  Bound: each
    output is a sum of 4^k products of rounded superoperator entries,
    (4^k + 2 count + 4) roundings of values below 1."""
    from qvm_amd.state import HipPureState
    rng = np.random.default_rng(100 * n + 10 * k + count)
    d = 1 << n
    u = 2.0 ** (-53 if dtype == "f64" else -24)
    tol = (4 ** k + 2 * count + 4) * u
    with HipPureState(2 * n, dtype) as st:
        for trial in range(4):
            qubits = [int(x) for x in rng.permutation(n)[:k]]
            A = rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d))
            rho = A @ A.conj().T
            rho /= np.trace(rho)
            if dtype == "f32":
                rho = rho.astype(np.complex64).astype(np.complex128)
            K = kraus_list(count, k, rng)
            st.write_amplitudes(rho.reshape(-1))
            st.density_apply_kraus(n, K, qubits)
            want = sum(embed(Kj, qubits, n) @ rho @ embed(Kj, qubits, n).conj().T for Kj in K)
            assert np.max(np.abs(st.amplitudes().reshape(d, d) - want)) < tol, qubits


def test_density_permutation_and_diagonal_gates_are_exact():
    """CNOT and CZ as superoperators move and negate entries: bit-exact."""
    from qvm_amd.state import HipPureState
    rng = np.random.default_rng(3)
    n, d = 5, 32
    rho = rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d))
    with HipPureState(2 * n, "f64") as st:
        for name in ("CNOT", "CZ", "SWAP"):
            for q in ([0, 1], [4, 2], [1, 3]):
                U = G.gate_matrix(name)
                F = embed(U, q, n).real
                st.write_amplitudes(rho.reshape(-1))
                st.density_apply_kraus(n, U[None], q)
                assert np.array_equal(st.amplitudes().reshape(d, d), F @ rho @ F.T), (name, q)


def test_density_apply_kraus_refuses():
    from qvm_amd import _native as N
    from qvm_amd.state import HipPureState
    with HipPureState(6, "f64") as st:
        I2 = np.eye(2)[None]
        for nq, K, q in ((2, I2, [0]), (3, I2, [3]), (3, np.eye(4)[None], [1, 1]), (3, I2 * np.nan, [0])):
            with pytest.raises(N.QVMHipError):
                st.density_apply_kraus(nq, K, q)


@pytest.mark.parametrize("dtype,big,small", [("f64", 1e200, 1e-300), ("f32", 1e25, 1e-30)])
def test_density_products_past_the_range(dtype, big, small):
    """A finite operator whose products of two entries overflow, on a state
    that stays finite under one operator after another: a single gate, a list, a
    run of gates, and a run whose product overflows though no map does.  Bound:
    the gates' products are single ones, rounded four times on the way."""
    from qvm_amd._native import ERANGE, QVMHipError
    from qvm_amd.density import DensityQVM
    u = 2.0 ** (-53 if dtype == "f64" else -24)
    rho = np.arange(1, 257).reshape(16, 16) * (1 + 0.5j) * small
    A, mid = np.diag([big, -big]), np.diag([big ** 0.5, 1])
    S = embed(A, [1], 4)
    qvm = DensityQVM(4, dtype=dtype)
    text = (f"DEFGATE A:\n    {big!r}, 0\n    0, {-big!r}\n\nDEFGATE B:\n    {big ** 0.5!r}, 0\n    0, 1\n\n"
            f"DEFGATE C:\n    {big ** -0.6!r}, 0\n    0, 1\n\n")
    for way in ("gate", "list", "A 1\nZ 0\n", "B 1\nB 1\nC 1\nZ 0\n"):
        want = S @ rho @ S
        qvm.state.write_amplitudes(rho.reshape(-1))
        if way == "gate":
            with pytest.raises(QVMHipError) as e:
                qvm.state.density_apply_kraus(4, A[None], [1])
            assert e.value.code == ERANGE
            qvm.apply_superoperator([A], [1])
        elif way == "list":
            qvm.apply_superoperator([A, 0 * A], [1])
        else:
            want = rho
            for ins in way.split("\n")[:-1]:
                M = {"A": A, "B": mid, "C": np.diag([big ** -0.6, 1]), "Z": np.diag([1, -1])}[ins[0]]
                F = embed(M, [int(ins[2])], 4)
                want = F @ want @ F
            qvm.load_program(text + way)
            qvm.run()
        assert np.max(np.abs(qvm.density_matrix() - want)) <= 16 * u * np.max(np.abs(want)), way
    qvm.close()


def test_density_calls_refuse_a_qubit_count_that_wraps():
    """Twice 2^31 + 3 is 6 in 32 bits: the row bits of that many qubits lie
    outside a 6-qubit state."""
    from qvm_amd import _native as N
    from qvm_amd.state import HipPureState
    nq, eye = 2 ** 31 + 3, np.eye(2)
    out = np.zeros(8)
    with HipPureState(6, "f64") as st:
        for call in (lambda: st.density_apply_kraus(nq, eye[None], [0]),
                     lambda: st.density_apply_kraus_run(nq, [([eye], 0), ([eye], 1)]),
                     lambda: N.check(N.lib().qvmhip_density_diagonal(st.handle, nq, N.dptr(out)))):
            with pytest.raises(N.QVMHipError):
                call()
        assert st.amplitudes()[0] == 1


@pytest.mark.parametrize("dtype,n,k,count", [("f64", 1, 1, 2), ("f64", 2, 2, 3), ("f64", 3, 1, 9), ("f64", 9, 1, 4),
                                             ("f64", 9, 2, 5), ("f64", 13, 1, 5), ("f32", 9, 1, 4), ("f32", 9, 2, 3)])
def test_kraus_choice(dtype, n, k, count):
    """Every operator of the map chosen in turn (a draw inside its interval),
    maps longer than one read included; a draw past the total takes the last
    one.  Bound: 2^k + 2 roundings per product sum, the norm's sum over the
    state and its division, on amplitudes below 1."""
    from qvm_amd.state import HipPureState
    rng = np.random.default_rng(1000 * n + 10 * k + count)
    tol = (4 * 2 ** k + n + 24) * 2.0 ** (-53 if dtype == "f64" else -24)
    idx = np.arange(1 << n)
    with HipPureState(n, dtype) as st:
        qubits = [int(x) for x in rng.permutation(n)[:k]]
        psi = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
        psi /= np.linalg.norm(psi)
        if dtype == "f32":
            psi = psi.astype(np.complex64).astype(np.complex128)
        K = kraus_list(count, k, rng)
        D = 1 << k
        rest = idx & ~sum(1 << q for q in qubits)
        sub = sum(((idx >> q) & 1) << j for j, q in enumerate(qubits))
        member = [rest | sum(((c >> j) & 1) << q for j, q in enumerate(qubits)) for c in range(D)]
        out = [sum(Kj[sub, c] * psi[member[c]] for c in range(D)) for Kj in K]
        p = np.array([np.sum(np.abs(o) ** 2) for o in out])
        cum = np.cumsum(p)
        for j in range(count + 1):
            want = min(j, count - 1)
            r = cum[want] - 0.5 * p[want] if j < count else 2.0
            st.write_amplitudes(psi)
            assert st.apply_kraus_choice(K, qubits, r) == want
            assert np.max(np.abs(st.amplitudes() - out[want] / np.sqrt(p[want]))) < tol, j


def test_kraus_choice_refuses_an_annihilated_state():
    from qvm_amd import _native as N
    from qvm_amd.state import HipPureState
    lower = np.array([[[0, 1], [0, 0]]], dtype=np.complex128)
    with HipPureState(4, "f64") as st:
        with pytest.raises(N.QVMHipError):
            st.apply_kraus_choice(lower, [1], 0.5)  # |0> has nothing to lower
        assert st.amplitudes()[0] == 1
        with pytest.raises(N.QVMHipError):
            st.apply_kraus_choice(np.eye(8)[None], [0, 1, 2], 0.5)
        with pytest.raises(N.QVMHipError):
            st.apply_kraus_choice(np.full((1, 2, 2), np.inf), [0], 0.5)
        # an operator past the chosen one is never looked at
        assert st.apply_kraus_choice(np.stack([np.eye(2), np.eye(2) * np.nan]), [0], 0.5) == 0


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 6, 7])
def test_density_run_of_maps_matches_kraus_sums(dtype, n):
    """A run of 1-qubit maps (dense, diagonal, several on one qubit; below the
    smallest tile, one pass, several passes) against numpy, entry by entry.
    Bound: (4 + 2 count + 4) roundings per map as for a single one, of entries of
    order 2^-n, the maps contracting."""
    from qvm_amd.state import HipPureState
    rng = np.random.default_rng(40 + n)
    d = 1 << n
    u = 2.0 ** (-53 if dtype == "f64" else -24)
    maps = []
    for i in range(2 * n + 3):
        q = int(rng.integers(n)) if i < n + 3 else i - n - 3
        if i % 3 == 2:
            p = rng.uniform(0.1, 0.4)
            maps.append(([np.sqrt(1 - p) * np.eye(2), np.sqrt(p) * G.gate_matrix("Z") @ G.gate_matrix("S")], q))
        else:
            maps.append((list(kraus_list(1 + i % 4, 1, rng)), q))
    tol = sum(8 + 2 * len(ops) for ops, _ in maps) * u
    A = rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d))
    rho = A @ A.conj().T
    rho /= np.trace(rho)
    with HipPureState(2 * n, dtype) as st:
        st.write_amplitudes(rho.reshape(-1))
        st.density_apply_kraus_run(n, maps)
        got = st.amplitudes().reshape(d, d)
    for ops, q in maps:
        rho = sum(embed(K, [q], n) @ rho @ embed(K, [q], n).conj().T for K in ops)
    assert np.max(np.abs(got - rho)) <= tol


def test_density_run_refuses_and_keeps_the_maps_before():
    from qvm_amd._native import QVMHipError
    from qvm_amd.state import HipPureState
    X, bad = G.gate_matrix("X"), np.full((2, 2), np.nan)
    for maps in ([([X], 1), ([bad], 0)], [([X], 1), ([X], 4)]):
        with HipPureState(8) as st:
            with pytest.raises(QVMHipError):
                st.density_apply_kraus_run(4, maps)
            assert st.density_diagonal(4)[2] == 1.0
    with HipPureState(8) as st, pytest.raises(QVMHipError):
        st.density_apply_kraus_run(3, [([X], 1), ([X], 2)])


def test_density_program_fuses_runs_only_between_other_instructions():
    """The interpreter's shared sweeps against one instruction at a time:
    runs broken by 2-qubit gates, a label and a measurement, a noisy definition,
    an unresolvable gate after a run."""
    from qvm_amd.density import DensityQVM
    from qvm_amd.qvm import QVMError
    g = 0.3
    noise = {("I", (1,)): [np.diag([1, np.sqrt(1 - g)]), np.array([[0, np.sqrt(g)], [0, 0]])]}
    text = ("DECLARE ro BIT[5]\n" + "".join(f"RX(0.{q + 1}) {q}\nH {q}\n" for q in range(5))
            + "I 1\nCNOT 0 1\nRZ(0.4) 2\nLABEL @a\nRY(1.0) 2\nI 1\nX 3\nMEASURE 3 ro[3]\nH 3\nT 3\n")
    got = []
    for cls in (DensityQVM, type("OneByOne", (DensityQVM,), {"transition": lambda s, i: DensityQVM.transition(s, i)})):
        qvm = cls(5, noisy_gate_definitions=noise, rng=lambda: 0.25)
        qvm.load_program(text)
        qvm.run()
        got.append((qvm.amplitudes(), list(qvm.memory["ro"]), qvm.pc))
        qvm.reset_quantum_state()
        qvm.load_program("X 0\nX 1\nDAGGER S 2\n")
        with pytest.raises(QVMError):
            qvm.run()
        assert qvm.pc == 2 and qvm.measurement_probabilities()[3] == 1.0
        qvm.close()
    assert got[0][1:] == got[1][1:]
    assert np.max(np.abs(got[0][0] - got[1][0])) <= 25 * 12 * 2.0 ** -53


def _noisy_pair(n, dtype, defs, text, draws, amps=None):
    """(amplitudes, memory, draws used) of a program run with shared sweeps
    and one instruction at a time."""
    from qvm_amd.noise import NoisyQVM
    out = []
    for cls in (NoisyQVM, type("OneByOne", (NoisyQVM,), {"transition": lambda s, i: NoisyQVM.transition(s, i)})):
        qvm = cls(n, noisy_gate_definitions=defs, dtype=dtype, rng=iter(draws).__next__)
        if amps is not None:
            qvm.set_amplitudes(amps)
        qvm.load_program(text)
        qvm.run()
        out.append((qvm.amplitudes(), list(qvm.memory.get("ro", [])), qvm.draws_used))
        qvm.close()
    return out


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("n", [2, 7, 8, 12, 13])
def test_noisy_runs_match_one_by_one(dtype, n):
    """Runs of unitary and unitary-mixture gates (below the smallest tile, one
    pass, several) around gates that end a run: amplitude damping, a noisy CNOT, a
    measurement.  The state starts with norm 1.5.  Bound: eight roundings of values
    up to 1.5 per gate on either side."""
    rng = np.random.default_rng(n)
    m = G.gate_matrix
    defs = {}
    for q in range(n):
        p = rng.uniform(0.1, 0.3, 3)
        defs["H", (q,)] = [np.sqrt(1 - p.sum()) * m("H")] + [np.sqrt(x) * m(P) @ m("H") for x, P in zip(p, "XYZ")]
    g = 0.4
    defs["I", (0,)] = [np.diag([1, np.sqrt(1 - g)]), np.array([[0, np.sqrt(g)], [0, 0]])]
    defs["CNOT", (0, 1)] = [np.sqrt(0.7) * m("CNOT"), np.sqrt(0.3) * np.kron(m("Z"), m("Z")) @ m("CNOT")]
    layer = "".join(f"RX({rng.uniform(0, 6):.6f}) {q}\n" for q in range(n)) + "".join(f"H {q}\n" for q in range(n))
    text = ("DECLARE ro BIT[2]\n" + layer + "I 0\nCNOT 0 1\n" + layer + "T 1\nMEASURE 0 ro[0]\nH 1\nS 0\nH 0\n"
            + "I 0\nX 1\n")
    amps = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    amps *= 1.5 / np.linalg.norm(amps)
    for trial in range(4):
        draws = rng.random(6 * n + 20)
        (a, ra, da), (b, rb, db) = _noisy_pair(n, dtype, defs, text, draws, amps)
        assert ra == rb and da == db
        u = 2.0 ** (-53 if dtype == "f64" else -24)
        assert np.max(np.abs(a - b)) <= 2 * 8 * 1.5 * (4 * n + 10) * u
        assert abs(np.linalg.norm(a) - 1) <= (4 * n + 10) * 8 * u


@pytest.mark.parametrize("n", [1, 5, 9, 13])
def test_1q_run_whose_norm_is_not_finite_is_applied_whole(n):
    """Amplitudes of 1e200 have no finite norm: the run reports it, after one
    gate, in sweeps, in one pass and in two, with every gate applied.  Bound: two
    roundings of the entry and one of the sum per gate."""
    from qvm_amd import _native as N
    from qvm_amd.state import HipPureState
    H = G.gate_matrix("H")
    with HipPureState(n) as st:
        psi = np.zeros(1 << n, dtype=np.complex128)
        psi[0] = 1e200
        st.write_amplitudes(psi)
        with pytest.raises(N.QVMHipError) as e:
            st.apply_1q_run([H] * n, list(range(n)), normalize=True)
        assert e.value.code == N.ERANGE
        want = 1e200 * 2.0 ** (-n / 2)
        assert np.max(np.abs(st.amplitudes() - want)) <= 3 * n * 2.0 ** -53 * want


@pytest.mark.parametrize("dtype,big,small", [("f64", 1e200, 1e-300), ("f32", 1e25, 1e-30)])
@pytest.mark.parametrize("n", [3, 9])
def test_1q_run_whose_product_overflows(dtype, big, small, n):
    """Two gates on one qubit whose product is past the range go gate by
    gate: the same bits as apply_matrix."""
    from qvm_amd.state import HipPureState
    mats = [np.diag([big, 1]), G.gate_matrix("H"), np.diag([big, 1j]), np.diag([1 / big, 1])]
    qubits = [n - 1, 0, n - 1, n - 1]
    psi = np.arange(1, (1 << n) + 1) * (1 - 2j) * small
    with HipPureState(n, dtype) as st, HipPureState(n, dtype) as ref:
        st.write_amplitudes(psi)
        ref.write_amplitudes(psi)
        st.apply_1q_run(mats, qubits)
        for U, q in zip(mats, qubits):
            ref.apply_matrix(U, [q])
        assert np.all(np.isfinite(ref.amplitudes())) and np.array_equal(st.amplitudes(), ref.amplitudes())


def test_noisy_run_takes_no_draw_for_a_gate_it_does_not_cover():
    """Damping only, a plain matrix that is not unitary, a modifier on a noisy gate."""
    from qvm_amd.noise import NoisyQVM
    from qvm_amd.qvm import QVMError
    g = 0.5
    damp = [np.diag([1, np.sqrt(1 - g)]), np.array([[0, np.sqrt(g)], [0, 0]])]
    mix = [np.sqrt(0.5) * G.gate_matrix("X"), np.sqrt(0.5) * G.gate_matrix("Z") @ G.gate_matrix("X")]
    text = "DEFGATE A:\n    1.0, 0\n    0, 0.5\n\nX 0\nX 0\nA 0\nH 0\nI 0\nI 0\n"
    (a, _, da), (b, _, db) = _noisy_pair(2, "f64", {("I", (0,)): damp, ("X", (0,)): mix}, text, [0.3, 0.9, 0.2, 0.6])
    assert da == db == 4 and np.max(np.abs(a - b)) <= 1e-15 * 8
    qvm = NoisyQVM(2, noisy_gate_definitions={("X", (0,)): mix}, rng=lambda: 0.1)
    qvm.load_program("X 0\nX 0\nDAGGER X 0\n")
    with pytest.raises(QVMError):
        qvm.run()
    assert qvm.draws_used == 2 and qvm.pc == 2
    qvm.close()
