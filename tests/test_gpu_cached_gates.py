"""Plain gates on both sides of the size above which the sweeps use
non-temporal accesses (256 MiB): the cached and the streamed forms of every
kernel give the same bits."""
import numpy as np
import pytest

from qvm_amd import gates as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_cached_and_streamed_forms_agree(dtype):
    """A state of n qubits (256 MiB, cached) against one with a spectator
    qubit more (512 MiB, streamed) in |0>: its lower half goes through the same
    gates and must end with the same bits, its upper half at zero."""
    from qvm_amd.state import HipPureState
    n = 24 if dtype == "f64" else 25
    rng = np.random.default_rng(8)
    U2 = np.linalg.qr(rng.normal(size=(4, 4)) + 1j * rng.normal(size=(4, 4)))[0]
    m = G.gate_matrix
    gates = [(m("H"), [q]) for q in (0, 3, 5, 6, 7, 13, n - 1)]
    gates += [(m("RX", [0.3 + q]), [q]) for q in (0, 2, 5, 6, 9, n - 1)]
    gates += [(m("RZ", [0.7]), [4]), (m("CPHASE", [1.1]), [n - 1, 13]), (m("CPHASE", [0.4]), [13, 2]),
              (m("CPHASE", [0.9]), [9, 0]), (m("PHASE", [0.2]), [7]), (m("RZZ", [0.5]), [3, 13])]
    gates += [(m("CNOT"), q) for q in ([0, 1], [1, 0], [3, 4], [4, 2], [2, 9], [9, 2], [9, 13], [n - 1, 6])]
    gates += [(m("SWAP"), q) for q in ([0, n - 1], [8, 13], [1, 2])] + [(m("ISWAP"), [5, 12])]
    gates += [(U2, [0, 8]), (U2, [7, 12]), (m("CCNOT"), [5, 2, 9])]
    with HipPureState(n, dtype) as a, HipPureState(n + 1, dtype) as b:
        for U, q in gates:
            nat = G.nat_tuple(*q)
            a.apply_matrix(U, nat)
            b.apply_matrix(U, nat)
        for start in (0, (1 << n) - (1 << 18), (1 << (n - 1)) - (1 << 17)):
            x, y = a.read_amplitudes(start, 1 << 18), b.read_amplitudes(start, 1 << 18)
            assert np.array_equal(x, y), start
        assert abs(a.norm() - 1) < (1e-12 if dtype == "f64" else 1e-5)
        u = (np.arange(2000) + 0.5) / 2000
        assert np.array_equal(a.sample(u), b.sample(u))
