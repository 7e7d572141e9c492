"""Compiled programs at the qubit counts where the default tile width changes:
in-order passes give the bits of the gate-by-gate path at every width."""
import numpy as np
import pytest

from qvm_amd import circuits as C
from qvm_amd import gates as G
from qvm_amd import planner as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("n", [8, 11, 12, 17, 18, 19])
def test_default_width_matches_plain(n, dtype):
    from qvm_amd.state import HipPureState
    rng = np.random.default_rng(n)
    gates = list(C.layered(n, 3, seed=n))
    for _ in range(2 * n):
        a, b = (int(x) for x in rng.choice(n, 2, replace=False))
        U = np.linalg.qr(rng.normal(size=(2, 2)) + 1j * rng.normal(size=(2, 2)))[0]
        gates += [(U, [a]), (G.gate_matrix("CPHASE", [float(rng.uniform(0, 6))]), [a, b]), (G.gate_matrix("CNOT"), [b, a])]
    with HipPureState(n, dtype) as ref, HipPureState(n, dtype) as st:
        for U, q in gates:
            ref.apply_matrix(U, G.nat_tuple(*q))
        prog = P.compile_gates(st, gates, mode="tiled", reorder=False)
        assert all(len(it.qubits) <= P.default_tile_m(dtype, n) for it in prog.plan)
        for _ in range(2):  # replays of one program
            st.reset_zero()
            prog.run()
            assert np.array_equal(st.amplitudes(), ref.amplitudes())
        prog.close()


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("nops", [1, 25, 60, 300, 1500])
def test_op_lists_of_every_length_reach_the_device(dtype, nops):
    """One exact pass of nops gates, twice in a row with other angles: lists
    that travel in one and two launches, by copy and in a buffer of their own.  The
    same bits as gate by gate."""
    from qvm_amd.state import HipPureState
    rng = np.random.default_rng(nops)
    m, n = 11, 12
    with HipPureState(n, dtype) as st, HipPureState(n, dtype) as ref:
        for _ in range(2):
            gates = []
            for i in range(nops):
                a, b = (int(x) for x in rng.permutation(m)[:2])
                gates.append([(G.gate_matrix("H"), [a]), (G.gate_matrix("RX", [rng.uniform(0, 6)]), [a]),
                              (G.gate_matrix("CNOT"), [a, b]), (G.gate_matrix("CPHASE", [rng.uniform(0, 6)]), [a, b])][i % 4])
            st.apply_tile_pass(list(range(m)), [P.tile_op(U, q, {x: x for x in range(m)}) for U, q in gates])
            for U, q in gates:
                ref.apply_matrix(U, G.nat_tuple(*q))
        assert np.array_equal(st.amplitudes(), ref.amplitudes())
