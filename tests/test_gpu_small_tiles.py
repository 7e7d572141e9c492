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
