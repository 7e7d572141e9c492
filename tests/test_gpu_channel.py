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
