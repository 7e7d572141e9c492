// channel.hip -- noise channels (Kraus maps): the superoperator of a
// density-matrix gate in one sweep.
//
// A density matrix rho is held as vec(rho), row-major, in a 2*nq-qubit state:
// column bits 0..nq-1, row bits nq..2*nq-1 (src/density-qvm.lisp).  A Kraus map
// rho -> sum_j K_j rho K_j^H on k qubits is then one linear map on the 2k index
// bits (q_i, q_i + nq), with the 4^k x 4^k matrix
//     S[(r', c'), (r, c)] = sum_j K_j[r'][r] conj(K_j[c'][c]).
// The reference applies each K_j to a pristine copy and adds the results up
// (src/apply-gate.lisp:66-99).  Swept that way a map of m operators moves
// 2 m gate sweeps, m - 1 restored copies, m - 1 accumulations and two more
// copies; as one superoperator it is one read and one write of the state
// whatever m is.  A 12-qubit noisy circuit (2^24 amplitudes, 94 gates with 1,
// 2 or 4 operators) went from 80.2 to 8.05 ms, 85 us or 6.3 TB/s per gate.
#include <cmath>
#include <complex>
#include <vector>

#include "qvmhip_internal.h"

namespace qvmhip {

using cd = std::complex<double>;

// The superoperator on (q_0 .. q_{k-1}, q_0 + nq .. q_{k-1} + nq): index
// bits 0..k-1 are the column bits, k..2k-1 the row bits.
static std::vector<cd> superoperator(const cd *K, uint32_t count, uint32_t k) {
    const size_t D = size_t(1) << k, DD = D * D;
    std::vector<cd> S(DD * DD, cd(0, 0));
    for (uint32_t j = 0; j < count; ++j) {
        const cd *A = K + (size_t)j * DD;
        for (size_t rp = 0; rp < D; ++rp)
            for (size_t r = 0; r < D; ++r) {
                const cd a = A[rp * D + r];
                if (a == cd(0, 0)) continue;  // structural zeros stay exact zeros
                for (size_t cp = 0; cp < D; ++cp)
                    for (size_t c = 0; c < D; ++c) {
                        const cd b = std::conj(A[cp * D + c]);
                        if (b == cd(0, 0)) continue;
                        S[(rp * D + cp) * DD + r * D + c] += a * b;
                    }
            }
    }
    return S;
}

int launch_kraus(qvmhip_state *s, uint32_t nq, const double *K, uint32_t count, uint32_t k, const uint32_t *qubits) {
    const std::vector<cd> S = superoperator(reinterpret_cast<const cd *>(K), count, k);
    uint32_t q[6];
    for (uint32_t i = 0; i < k; ++i) {
        q[i] = qubits[i];
        q[k + i] = qubits[i] + nq;
    }
    const double *m = reinterpret_cast<const double *>(S.data());
    // one qubit: a 4x4 by value.  Wider maps that are diagonal or permute
    // (CZ, CNOT, SWAP) keep the structured kernels; dense ones (16x16, 64x64)
    // go to the matrix cores.
    if (k == 1 || !gate_is_dense(m, 2 * k, q)) return launch_gate(s, m, 2 * k, q, 0);
    void *dst = (char *)s->mat + kFusedMatOffset;
    QH_CHECK(hipMemcpyAsync(dst, m, S.size() * sizeof(cd), hipMemcpyHostToDevice, s->stream));
    return launch_fused_dense(s, dst, 2 * k, q);
}

}  // namespace qvmhip
