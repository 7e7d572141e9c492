"""GPU tests of the diagonal ops of a tile pass: every place of the two
qubits (lane, wave, register, outside the tile) with the entry patterns that
the kernel treats apart (1 outside the condition, -1 on it, neither, no use
of the tile)."""
import numpy as np
import pytest

from qvm_amd import gates as G, planner as P

pytestmark = pytest.mark.gpu


def apply_diagonal(psi, d, nat):
    idx = np.arange(psi.size)
    j = sum(((idx >> q) & 1) << b for b, q in enumerate(nat))
    return psi * d[j]


@pytest.mark.parametrize("fma", [False, True])
@pytest.mark.parametrize("dtype,m", [("f64", 8), ("f64", 11), ("f32", 9), ("f32", 12)])
def test_diagonals_of_a_tile_pass(dtype, m, fma):
    from qvm_amd.state import HipPureState, Program
    n = m + 2
    rng = np.random.default_rng(m)
    psi = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    psi /= np.linalg.norm(psi)
    if dtype == "f32":
        psi = psi.astype(np.complex64).astype(np.complex128)
    # low bits, bits 5 to 7 around the wave's six, the top bits, outside qubits
    qubits = sorted({0, 3, 5, 6, 7, m - 4, m - 3, m - 2, m - 1, m, m + 1} & set(range(n)))
    local = {q: q for q in range(m)}
    ops, ref = [], psi.copy()
    for a in qubits:
        for b in qubits:
            if a == b:
                continue
            e = np.exp(1j * rng.uniform(0, 2 * np.pi, 4))
            for d in ([1, 1, 1, -1], [1, 1, 1, e[0]], [1, 1, e[1], e[2]], [e[0], e[1], e[1], e[0]], list(e)):
                d = np.array(d, dtype=np.complex128)
                if rng.random() > 0.4:
                    continue
                nat = G.nat_tuple(a, b)
                ops.append(P.tile_op(np.diag(d), (a, b), local))
                ref = apply_diagonal(ref, d, nat)
        # a dense gate between them moves tile qubits to other places
        if a < m:
            U = G.gate_matrix("H")
            ops.append(P.tile_op(U, (a,), local))
            v = ref.reshape(-1, 2, 1 << a)
            ref = np.stack([U[0, 0] * v[:, 0] + U[0, 1] * v[:, 1], U[1, 0] * v[:, 0] + U[1, 1] * v[:, 1]],
                           axis=1).reshape(-1)
    with HipPureState(n, dtype, fma_tiles=fma) as st:
        st.write_amplitudes(psi)
        p = Program(st)
        p.add_tile_pass(list(range(m)), ops)
        p.finalize(True)
        p.run()
        out = st.read_amplitudes()
        p.close()
    # an amplitude is below 1; an op rounds four products and two sums of it
    eps = 2.0 ** (-53 if dtype == "f64" else -24)
    assert np.abs(out - ref).max() < 6 * len(ops) * eps
