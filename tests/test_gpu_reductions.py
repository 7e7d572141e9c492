"""GPU tests of the read sweeps (probabilities, norm, ZZ expectation) and of
the collapse kernel around their segment sizes: one element, below, at and
above one workgroup's 2048 elements, and several workgroups."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def random_state(n, dtype, rng):
    v = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    v /= np.linalg.norm(v)
    return v if dtype == "f64" else v.astype(np.complex64).astype(np.complex128)


def bound(n):
    """A thread adds at most 2^n / 256 + 8 terms one after another, then 30
    levels of waves, workgroups and partials; every term is below 1 in sum."""
    return ((1 << n) / 256 + 40) * 2.0 ** -53


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("n", [1, 2, 5, 10, 11, 12, 13, 17, 19])
def test_probabilities(dtype, n):
    from qvm_amd.state import HipPureState
    rng = np.random.default_rng(n)
    psi = random_state(n, dtype, rng)
    p = np.abs(psi) ** 2
    idx = np.arange(1 << n)
    with HipPureState(n, dtype) as st:
        st.write_amplitudes(psi)
        assert abs(st.total_probability() - p.sum()) < bound(n)
        for q in range(n):
            one = (idx >> q) & 1 == 1
            assert abs(st.prob_excited(q) - p[one].sum()) < bound(n), q
            assert abs(st.prob_ground(q) - p[~one].sum()) < bound(n), q
        st.reset_zero()
        assert st.prob_excited(0) == 0.0 and st.prob_ground(n - 1) == 1.0


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("n,nedges", [(1, 1), (2, 3), (8, 12), (11, 20), (12, 30), (13, 256), (18, 40), (18, 200)])
def test_expectation_zz(dtype, n, nedges):
    """Edge lists with up to 32 and with more cross edges, repeated edges and
    edges from a qubit to itself (<Z_a Z_a> = 1)."""
    from qvm_amd.state import HipPureState
    rng = np.random.default_rng(100 + n + nedges)
    psi = random_state(n, dtype, rng)
    p = np.abs(psi) ** 2
    idx = np.arange(1 << n)
    edges = rng.integers(0, n, size=(nedges, 2))
    want = sum(np.sum(p * (1 - 2 * (((idx >> a) ^ (idx >> b)) & 1))) for a, b in edges)
    with HipPureState(n, dtype) as st:
        st.write_amplitudes(psi)
        assert abs(st.expectation_zz(edges) - want) < 2 * nedges * bound(n)
        assert st.expectation_zz(np.zeros((0, 2))) == 0.0


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("n", [11, 12, 14, 22, 24])
def test_expectation_zz_of_basis_states(dtype, n):
    """Every edge is +1 or -1 on a basis state, so the sum is exact: dense edge
    lists across bit 11, one edge up to 256 times, states of several chunks per
    workgroup."""
    from qvm_amd import gates as G
    from qvm_amd.state import HipPureState
    rng = np.random.default_rng(n)
    lists = [rng.integers(0, n, size=(256, 2)), np.array([(i % min(n, 11), n - 1 - i % (n - 10)) for i in range(200)])]
    lists += [np.repeat([[3, n - 1]], m, axis=0) for m in (2, 7, 255, 256)]
    lists.append(np.repeat([[0, n - 1], [n - 1, 2], [n - 2, n - 1]], [5, 130, 64], axis=0))
    with HipPureState(n, dtype) as st:
        for _ in range(12):
            bits = rng.integers(0, 2, size=n)
            st.reset_zero()
            for q in np.flatnonzero(bits):
                st.apply_matrix(G.gate_matrix("X"), [int(q)])
            z = 1 - 2 * bits
            for edges in lists:
                assert st.expectation_zz(edges) == np.sum(z[edges[:, 0]] * z[edges[:, 1]])


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("n", [1, 2, 7, 9, 12])
def test_collapse_bit_exact(dtype, n):
    """Both forms, every qubit: the kept half times the rounded factor, zeros
    elsewhere; a NaN in the annihilated half vanishes in the interpreted form."""
    from qvm_amd.state import HipPureState
    rng = np.random.default_rng(7 * n)
    real = np.float64 if dtype == "f64" else np.float32
    psi = random_state(n, dtype, rng)
    idx = np.arange(1 << n)
    with HipPureState(n, dtype) as st:
        for q in range(n):
            for bit in (0, 1):
                kept = ((idx >> q) & 1) == bit
                v = psi.copy()
                v[~kept] = np.nan
                st.write_amplitudes(v)
                st.force_measure(q, bit, 0.37)
                f = real(1.0 / np.sqrt(0.37 if bit else 1.0 - 0.37))
                want = np.zeros(1 << n, dtype=np.complex128)
                want.real[kept] = f * psi.real[kept].astype(real)
                want.imag[kept] = f * psi.imag[kept].astype(real)
                assert np.array_equal(st.amplitudes(), want), (q, bit)
        st.write_amplitudes(psi)
        p0 = st.prob_ground(0)
        bit, _ = st.measure(0, 0.5, compiled=True)
        f = real(1.0 / np.sqrt(p0 if bit == 0 else 1.0 - p0))
        kept = (idx & 1) == bit
        want = np.zeros(1 << n, dtype=np.complex128)
        want.real[kept] = f * psi.real[kept].astype(real)
        want.imag[kept] = f * psi.imag[kept].astype(real)
        assert np.array_equal(st.amplitudes(), want)
