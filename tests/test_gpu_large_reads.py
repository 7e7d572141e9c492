"""Read, collapse and Kraus-choice kernels at the sizes where a workgroup takes
several steps, where the partial sums are added on the device and where the
accesses become non-temporal (states above 256 MiB)."""
import numpy as np
import pytest

from qvm_amd import gates as G

pytestmark = pytest.mark.gpu

WINDOW = 1 << 18


def kraus_list(count, k, rng):
    """Random Kraus operators: the blocks of an isometry."""
    D = 1 << k
    A = rng.normal(size=(count * D, D)) + 1j * rng.normal(size=(count * D, D))
    return np.linalg.qr(A)[0].reshape(count, D, D)


@pytest.mark.parametrize("dtype,n,k,count", [("f64", 22, 1, 2), ("f64", 22, 1, 4), ("f64", 22, 2, 3), ("f64", 21, 2, 2),
                                             ("f32", 22, 1, 4), ("f32", 22, 2, 3)])
def test_kraus_choice_of_many_steps(dtype, n, k, count):
    """1024 workgroups, up to eight groups per thread, the last groups of the
    state among them; every operator chosen once.  Bound, relative to the largest
    sum of moduli an amplitude is made of: 2^k products and sums of three roundings
    and the rounded factor; the weight's relative error is twice that of an
    amplitude, and the factor's half of it."""
    from qvm_amd.state import HipPureState
    rng = np.random.default_rng(1000 * n + 10 * k + count)
    u = 2.0 ** (-53 if dtype == "f64" else -24)
    psi = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    psi /= np.linalg.norm(psi)
    if dtype == "f32":
        psi = psi.astype(np.complex64).astype(np.complex128)
    K = kraus_list(count, k, rng)
    D = 1 << k
    for qubits in ([n - 1, 0][:k], [3, n - 2][:k]):
        # axes of the qubits in front, matrix bit j <-> qubits[j]
        order = [n - 1 - q for q in reversed(qubits)]
        rest = [a for a in range(n) if a not in order]
        v = psi.reshape((2,) * n).transpose(order + rest).reshape(D, -1)
        out = [Kj @ v for Kj in K]
        p = np.array([np.sum(np.abs(o) ** 2) for o in out])
        cum = np.cumsum(p)
        with HipPureState(n, dtype) as st:
            for j in range(count):
                st.write_amplitudes(psi)
                assert st.apply_kraus_choice(K, qubits, cum[j] - 0.5 * p[j]) == j
                got = st.amplitudes().reshape((2,) * n).transpose(order + rest).reshape(D, -1)
                scale = np.max(np.abs(K[j])) * D * np.max(np.abs(psi)) / np.sqrt(p[j])
                assert np.max(np.abs(got - out[j] / np.sqrt(p[j]))) <= (6 * D + 8) * u * scale, (qubits, j)


@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_reads_and_collapses_of_cached_and_streamed_states(dtype):
    """A product state of 256 MiB (cached accesses) and the same with one more
    qubit in |0> (512 MiB, non-temporal): probabilities and ZZ sums against their
    closed form, collapses and Kraus choices against each other, and the upper
    half of the larger state zero throughout.  Bound of the sums: two roundings per
    gate and amplitude, three gates' worth of entries, and the additions of
    tests/test_gpu_reductions.py."""
    from qvm_amd.state import HipPureState
    n = 24 if dtype == "f64" else 25
    u = 2.0 ** (-53 if dtype == "f64" else -24)
    sums = ((1 << (n + 1)) / 256 + 40) * 2.0 ** -53 + 12 * n * u
    rng = np.random.default_rng(n)
    angles = rng.uniform(0.3, 2.8, n)
    z = np.cos(angles)
    edges = rng.integers(0, n, size=(120, 2))
    zz = sum(1.0 if a == b else z[a] * z[b] for a, b in edges)
    K1, K2 = kraus_list(3, 1, rng), kraus_list(3, 2, rng)

    def same_lower_half(a, b, rel):
        for start in (0, (1 << (n - 1)) - WINDOW // 2, (1 << n) - WINDOW):
            x, y = a.read_amplitudes(start, WINDOW), b.read_amplitudes(start, WINDOW)
            assert np.max(np.abs(x - y)) <= rel * np.max(np.abs(x)), start
            assert not np.any(b.read_amplitudes((1 << n) + start, WINDOW)), start

    with HipPureState(n, dtype) as a, HipPureState(n + 1, dtype) as b:
        for st in (a, b):
            for q in range(n):
                st.apply_matrix(G.gate_matrix("RY", [angles[q]]), [q])
            assert abs(st.total_probability() - 1) <= sums
            for q in (0, 1, 5, 11, 17, n - 1):
                assert abs(st.prob_excited(q) - (1 - z[q]) / 2) <= sums, q
                assert abs(st.prob_ground(q) - (1 + z[q]) / 2) <= sums, q
            assert abs(st.expectation_zz(edges) - zz) <= 2 * len(edges) * sums
        assert b.prob_excited(n) == 0.0
        same_lower_half(a, b, 0)
        for q, bit in ((0, 1), (9, 0), (n - 1, 1)):
            p1 = a.prob_excited(q)
            a.force_measure(q, bit, p1)
            b.force_measure(q, bit, p1)
            same_lower_half(a, b, 0)
            assert (b.prob_excited(q) if bit == 0 else b.prob_ground(q)) == 0.0
            for st in (a, b):
                st.apply_matrix(G.gate_matrix("RY", [angles[q]]), [q])
        for K, qubits in ((K1, [6]), (K2, [n - 1, 2]), (K1, [n - 1]), (K2, [10, 9])):
            r = float(rng.uniform(0.2, 0.8))
            assert a.apply_kraus_choice(K, qubits, r) == b.apply_kraus_choice(K, qubits, r)
            same_lower_half(a, b, 8 * u)  # the weights are added in another order
        assert abs(b.norm() - 1) <= sums


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("count", [2, 5])
def test_three_qubit_map_on_a_three_qubit_density_state(dtype, count):
    """One column group of the 64 x 64 block: the whole state."""
    from tests.test_gpu_channel import test_density_superoperator_matches_kraus_sum as check
    check(dtype, 3, 3, count)
