// channel.hip -- noise channels (Kraus maps): the superoperator of a
// density-matrix gate in one sweep, and the stochastic choice of one Kraus
// operator on a pure state in one read and one gate sweep.
//
// Density matrices.
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
// 2 or 4 operators) went from 80.2 to 8.05 ms, 85 us or 6.3 TB/s per gate (73 us with
// cached accesses).
//
// Pure states.  One operator of the map is chosen by inverse-transform
// sampling over p_j = |K_j psi|^2 (src/apply-gate.lisp:16-39).  Trying the operators
// one after another on a copy moves, per operator tried, a copied state (32
// bytes per amplitude), a gate sweep (32) and a norm (16), then a norm and a
// scale sweep (48).  k_kraus_norms reads the state once for up to four
// operators: every group's products K_j x are formed in registers and only
// their squares are kept.  The chosen operator, divided by sqrt(p_j), is then
// one ordinary gate in place: 48 bytes per amplitude in all.
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <limits>
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

// Whether the state's type holds every entry.  Finite Kraus entries can have
// products past the range (1e25 twice in FP32), where the operators applied one
// after another still give finite amplitudes.
static bool in_range(const qvmhip_state *s, const std::vector<cd> &A) {
    const double top = s->dtype == QVMHIP_F64 ? std::numeric_limits<double>::max() : std::numeric_limits<float>::max();
    return std::all_of(A.begin(), A.end(),
                       [&](const cd &z) { return std::abs(z.real()) <= top && std::abs(z.imag()) <= top; });
}

static int past_range() { return fail(QVMHIP_ERANGE, "the map's superoperator is past the range of the state's type"); }

int launch_kraus(qvmhip_state *s, uint32_t nq, const double *K, uint32_t count, uint32_t k, const uint32_t *qubits) {
    const std::vector<cd> S = superoperator(reinterpret_cast<const cd *>(K), count, k);
    if (!in_range(s, S)) return past_range();
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
    const std::vector<char> A = fused_operand(s->dtype, m, 2 * k, q);
    void *dst = (char *)s->mat + kFusedMatOffset;
    if (const int rc = upload_operand(s, dst, A.data(), A.size())) return rc;
    return launch_fused_dense(s, dst, 2 * k, q);
}

// The tile of the next pass over the qubits on[i], on[i + 1], ...: as many as
// fit 11 (FP64) or 12 (FP32) index bits beside the low bits that keep accesses
// whole lines; a qubit brings bit q and, on a density state, bit q + nq.  i
// moves past them.
namespace {
struct TileGroup {
    uint32_t m, tq[16], local[64];
    std::vector<uint32_t> members;
    TileGroup(const qvmhip_state *s, const std::vector<uint32_t> &on, size_t &i, uint32_t nq) {
        const bool f64 = s->dtype == QVMHIP_F64;
        const uint32_t low = f64 ? 3 : 4;
        m = std::min<uint32_t>(s->n, f64 ? 11 : 12);
        uint64_t tile = (uint64_t(1) << low) - 1;
        for (; i < on.size(); ++i) {
            const uint64_t with = tile | uint64_t(1) << on[i] | uint64_t(1) << (on[i] + nq);
            if ((uint32_t)__builtin_popcountll(with) > m) break;  // never at the first: low + 2 <= 8 <= m
            tile = with;
            members.push_back(on[i]);
        }
        for (uint32_t q = 0; (uint32_t)__builtin_popcountll(tile) < m; ++q) tile |= uint64_t(1) << q;
        uint32_t nb = 0;
        for (uint32_t q = 0; q < s->n; ++q)
            if ((tile >> q) & 1u) {
                local[q] = nb;
                tq[nb++] = q;
            }
    }
};
}  // namespace

// A run of 1-qubit maps.  Each would be a sweep of its own (73 us at 2^24 FP64
// amplitudes, bound by memory), but maps on one qubit multiply to one 4x4 and
// maps on different qubits commute, so the run is at most one 4x4 per qubit,
// and these share tile passes, five or four qubits each.  24 gates on 12 qubits: three
// passes of 124 us instead of 24 sweeps, and the noisy circuit above 6.3 ->
// 2.1 ms (its 11 two-qubit maps are 0.9 of that).  Less than two qubits, or a
// state below the smallest tile (2^8), stay sweeps.
int launch_kraus_run(qvmhip_state *s, uint32_t nq, uint32_t nmaps, const uint32_t *qubits, const uint32_t *counts,
                     const double *K) {
    std::vector<std::vector<cd>> S(nq);
    bool fits = true;
    const cd *k = reinterpret_cast<const cd *>(K);
    for (uint32_t i = 0; i < nmaps; k += 4 * (size_t)counts[i], ++i) {
        const std::vector<cd> A = superoperator(k, counts[i], 1);
        if (!in_range(s, A)) return past_range();
        std::vector<cd> &B = S[qubits[i]];
        if (B.empty()) {
            B = A;
            continue;
        }
        std::vector<cd> P(16, cd(0, 0));
        for (int r = 0; r < 4; ++r)
            for (int c = 0; c < 4; ++c)
                for (int j = 0; j < 4; ++j) {
                    const cd a = A[4 * r + j], b = B[4 * j + c];
                    if (a != cd(0, 0) && b != cd(0, 0)) P[4 * r + c] += a * b;
                }
        fits = fits && in_range(s, P);
        B.swap(P);
    }
    if (!fits) {  // a product past the range: map by map, as given
        k = reinterpret_cast<const cd *>(K);
        for (uint32_t i = 0; i < nmaps; k += 4 * (size_t)counts[i], ++i)
            if (const int rc = launch_kraus(s, nq, reinterpret_cast<const double *>(k), counts[i], 1, qubits + i))
                return rc;
        return QVMHIP_OK;
    }
    std::vector<uint32_t> on;
    for (uint32_t q = 0; q < nq; ++q)
        if (!S[q].empty()) on.push_back(q);
    if (on.size() < 2 || s->n < 8) {
        for (uint32_t q : on) {
            const uint32_t bits[2] = {q, q + nq};
            if (const int rc = launch_gate(s, reinterpret_cast<const double *>(S[q].data()), 2, bits, 0)) return rc;
        }
        return QVMHIP_OK;
    }
    for (size_t i = 0; i < on.size();) {
        TileGroup g(s, on, i, nq);
        std::vector<qvmhip_tile_op> ops;
        for (uint32_t q : g.members) {
            qvmhip_tile_op op;
            std::memset(&op, 0, sizeof(op));
            op.kind = QVMHIP_TILE_DIAG2;
            for (int r = 0; r < 16; ++r)
                if (r % 5 && S[q][r] != cd(0, 0)) op.kind = QVMHIP_TILE_DENSE2;
            op.q0 = g.local[q];
            op.q1 = g.local[q + nq];
            for (int r = 0, j = 0; r < 16; r += op.kind == QVMHIP_TILE_DIAG2 ? 5 : 1, ++j) {
                op.m[2 * j] = S[q][r].real();
                op.m[2 * j + 1] = S[q][r].imag();
            }
            ops.push_back(op);
        }
        if (const int rc = launch_tile_pass(s, g.m, g.tq, (uint32_t)ops.size(), ops.data())) return rc;
    }
    return QVMHIP_OK;
}

// A run of 1-qubit gates on a pure state (a sweep of 73 us each at 2^24 FP64
// amplitudes), multiplied together per qubit and applied up to eleven qubits a
// pass.  normalize, for unitary gates: the state ends with norm 1; its norm is
// read before the last pass, whose first matrix takes the factor.  A norm that
// cannot be divided by is found there too: the run is finished without the factor
// and reported, as by gate after gate and a normalization that is refused.
int launch_1q_run(qvmhip_state *s, uint32_t count, const uint32_t *qubits, const double *U, bool normalize) {
    std::vector<std::vector<cd>> S(s->n);
    const cd *u = reinterpret_cast<const cd *>(U);
    bool fits = true;
    for (uint32_t i = 0; i < count; ++i, u += 4) {
        std::vector<cd> &B = S[qubits[i]];
        if (B.empty()) {
            B.assign(u, u + 4);
            continue;
        }
        const cd P[4] = {u[0] * B[0] + u[1] * B[2], u[0] * B[1] + u[1] * B[3], u[2] * B[0] + u[3] * B[2],
                         u[2] * B[1] + u[3] * B[3]};
        B.assign(P, P + 4);
        fits = fits && in_range(s, B);
    }
    std::vector<uint32_t> on;
    for (uint32_t q = 0; q < s->n; ++q)
        if (!S[q].empty()) on.push_back(q);
    bool normalized = true;
    auto scale = [&](std::vector<cd> &A) -> int {
        double n2 = 0;
        if (const int rc = reduce_norm2(s, &n2)) return rc;
        const double len = std::sqrt(n2);
        normalized = len > 0 && std::isfinite(len);
        for (cd &x : A) x *= normalized ? 1.0 / len : 1.0;
        return QVMHIP_OK;
    };
    auto done = [&] {
        return normalized ? QVMHIP_OK : fail(QVMHIP_ERANGE, "cannot normalize a zero/non-finite state");
    };
    if (!fits) {  // a product past the range: gate by gate, as given
        u = reinterpret_cast<const cd *>(U);
        for (uint32_t i = 0; i < count; ++i, u += 4) {
            std::vector<cd> A(u, u + 4);
            if (normalize && i + 1 == count)
                if (const int rc = scale(A)) return rc;
            if (const int rc = launch_gate(s, reinterpret_cast<const double *>(A.data()), 1, qubits + i, 0)) return rc;
        }
        return done();
    }
    if (on.size() < 2 || s->n < 8) {
        for (uint32_t q : on) {
            if (normalize && q == on.back())
                if (const int rc = scale(S[q])) return rc;
            if (const int rc = launch_gate(s, reinterpret_cast<const double *>(S[q].data()), 1, &q, 0)) return rc;
        }
        return done();
    }
    for (size_t i = 0; i < on.size();) {
        TileGroup g(s, on, i, 0);
        if (normalize && i == on.size())
            if (const int rc = scale(S[g.members[0]])) return rc;
        std::vector<qvmhip_tile_op> ops;
        for (uint32_t q : g.members) {
            const std::vector<cd> &A = S[q];
            qvmhip_tile_op op;
            std::memset(&op, 0, sizeof(op));
            const bool diag = A[1] == cd(0, 0) && A[2] == cd(0, 0);
            op.kind = diag ? QVMHIP_TILE_DIAG1 : QVMHIP_TILE_DENSE1;
            op.q0 = g.local[q];
            for (int r = 0, j = 0; r < 4; r += diag ? 3 : 1, ++j) {
                op.m[2 * j] = A[r].real();
                op.m[2 * j + 1] = A[r].imag();
            }
            ops.push_back(op);
        }
        if (const int rc = launch_tile_pass(s, g.m, g.tq, (uint32_t)ops.size(), ops.data())) return rc;
    }
    return done();
}

// Operators per read: every one adds 2^k complex products per amplitude.  Four
// 1-qubit operators stay under the time of the read (2^24 FP64 amplitudes: 4 x 18
// FP64 operations per amplitude, about 30 us of issue against 45 us).  Two 2-qubit
// ones do not: their 64 FP64 coefficients do not fit the scalar registers (115
// spills, 106 VGPRs, four waves per SIMD), and the read takes 57 us where the
// 1-qubit form takes 40.
constexpr int kraus_per_read(int k) { return k == 1 ? 4 : 2; }
constexpr int kNormBlocks = 1024;  // partials of kNormBlocks * 4 sums fit the state's reduction scratch
static_assert(kNormBlocks * 4 <= kRedBlocks * 2, "reduction scratch");

template <typename T, int K, int C>
struct KrausArgs {
    static constexpr int D = 1 << K;
    GroupSpec g;
    uint64_t off[D];
    T ur[C * D * D];
    T ui[C * D * D];
};

// partial[C * block + j] = the block's share of sum |K_j x|^2, in FP64; the
// products are rounded in T and summed left to right, as the gate kernels do.
// Bound by the read; UN groups per thread are in flight.  For one qubit a
// workgroup takes a contiguous segment of the groups, and maps of one or two
// operators form two products, not four: 2^24 FP64 amplitudes 47.4 -> 40.3 us
// (6.7 TB/s).  For two qubits segments gained nothing (58.9 us against 57.7), and the
// grid strides over the groups.
template <typename T, int K, int C, bool NTM>
__global__ __launch_bounds__(kBlock) void k_kraus_norms(const vec2_t<T> *__restrict__ psi, const KrausArgs<T, K, C> a,
                                                        double *__restrict__ partial) {
    constexpr int D = 1 << K, UN = K == 1 ? 4 : 2, NW = kBlock / 64;
    using V = vec2_t<T>;
    __shared__ double sm[C][NW];
    double acc[C];
#pragma unroll
    for (int j = 0; j < C; ++j) acc[j] = 0.0;
    // 1 qubit: a segment per workgroup (both counts are powers of two)
    const uint64_t step = K == 1 ? kBlock : (uint64_t)gridDim.x * kBlock;
    const uint64_t seg = K == 1 ? a.g.ngroups / gridDim.x : a.g.ngroups;
    const uint64_t first = K == 1 ? seg * xcd_block(blockIdx.x, gridDim.x) : 0;
    for (uint64_t i0 = (K == 1 ? 0 : (uint64_t)blockIdx.x * kBlock) + threadIdx.x; i0 < seg; i0 += UN * step) {
        V x[UN][D];
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const uint64_t i = i0 + u * step;
            const uint64_t base = group_base(a.g, first + (i < seg ? i : i0));
#pragma unroll
            for (int d = 0; d < D; ++d) x[u][d] = ldg<NTM>(&psi[base + a.off[d]]);
        }
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            if (i0 + u * step >= seg) break;
#pragma unroll
            for (int j = 0; j < C; ++j)
#pragma unroll
                for (int r = 0; r < D; ++r) {
                    T yr = T(0), yi = T(0);
#pragma unroll
                    for (int c = 0; c < D; ++c) {
                        const T mr = a.ur[(j * D + r) * D + c], mi = a.ui[(j * D + r) * D + c];
                        const T pr = x[u][c].x * mr - x[u][c].y * mi;
                        const T pi = x[u][c].x * mi + x[u][c].y * mr;
                        yr = c ? yr + pr : pr;
                        yi = c ? yi + pi : pi;
                    }
                    acc[j] += (double)yr * (double)yr + (double)yi * (double)yi;
                }
        }
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int j = 0; j < C; ++j) {
        double v = acc[j];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        if (lane == 0) sm[j][wid] = v;
    }
    __syncthreads();
    if (threadIdx.x < C) {
        double t = 0.0;
        for (int w = 0; w < NW; ++w) t += sm[threadIdx.x][w];
        partial[C * blockIdx.x + threadIdx.x] = t;
    }
}

// out[j] = |K_j psi|^2 for the first `count` (at most C) operators.
template <typename T, int K, int C>
static int kraus_norms_c(qvmhip_state *s, const cd *ops, uint32_t count, const uint32_t *qubits, double *out) {
    constexpr int D = 1 << K;
    KrausArgs<T, K, C> a;
    std::memset(&a, 0, sizeof(a));
    a.g.nsorted = K;
    for (int b = 0; b < K; ++b) a.g.sorted[b] = qubits[b];
    std::sort(a.g.sorted, a.g.sorted + K);
    a.g.ngroups = uint64_t(1) << (s->n - K);
    for (int d = 0; d < D; ++d)
        for (int b = 0; b < K; ++b)
            if ((d >> b) & 1) a.off[d] |= uint64_t(1) << qubits[b];
    for (uint32_t e = 0; e < count * D * D; ++e) {
        a.ur[e] = (T)ops[e].real();
        a.ui[e] = (T)ops[e].imag();
    }
    const uint32_t grid = (uint32_t)std::min<uint64_t>((a.g.ngroups + kBlock - 1) / kBlock, kNormBlocks);
    double *partial = partials_of(s, (int)grid, C);
    if (stream_accesses(s))
        hipLaunchKernelGGL((k_kraus_norms<T, K, C, true>), dim3(grid), dim3(kBlock), 0, s->stream,
                           (const vec2_t<T> *)s->amps, a, partial);
    else
        hipLaunchKernelGGL((k_kraus_norms<T, K, C, false>), dim3(grid), dim3(kBlock), 0, s->stream,
                           (const vec2_t<T> *)s->amps, a, partial);
    QH_LAUNCH_CHECK();
    return sums_to_host(s, (int)grid, C, out, (int)count);
}

template <typename T, int K>
static int kraus_norms(qvmhip_state *s, const cd *ops, uint32_t count, const uint32_t *qubits, double *out) {
    return count <= 2 ? kraus_norms_c<T, K, 2>(s, ops, count, qubits, out)
                      : kraus_norms_c<T, K, kraus_per_read(K)>(s, ops, count, qubits, out);
}

int launch_kraus_choice(qvmhip_state *s, const double *K, uint32_t count, uint32_t k, const uint32_t *qubits, double r,
                        uint32_t *index) {
    const size_t DD = size_t(1) << (2 * k);
    const cd *ops = reinterpret_cast<const cd *>(K);
    const uint32_t per = (uint32_t)kraus_per_read((int)k);
    double sum = 0.0, p = 0.0;
    uint32_t chosen = count - 1;
    bool found = false;
    for (uint32_t j0 = 0; j0 < count && !found; j0 += per) {
        const uint32_t c = std::min(per, count - j0);
        double pj[4];
        int rc;
        if (s->dtype == QVMHIP_F64)
            rc = k == 1 ? kraus_norms<double, 1>(s, ops + j0 * DD, c, qubits, pj)
                        : kraus_norms<double, 2>(s, ops + j0 * DD, c, qubits, pj);
        else
            rc = k == 1 ? kraus_norms<float, 1>(s, ops + j0 * DD, c, qubits, pj)
                        : kraus_norms<float, 2>(s, ops + j0 * DD, c, qubits, pj);
        if (rc) return rc;
        for (uint32_t j = 0; j < c && !found; ++j) {
            // operators past the chosen one are never looked at
            const double *m = K + 2 * (j0 + j) * DD;
            if (!std::all_of(m, m + 2 * DD, [](double v) { return std::isfinite(v); }))
                return fail(QVMHIP_EINVAL, "matrix is not finite");
            p = pj[j];
            sum += p;
            chosen = j0 + j;
            found = sum >= r;
        }
    }
    const double len = std::sqrt(p);
    if (!(len > 0) || !std::isfinite(len)) return fail(QVMHIP_ERANGE, "cannot normalize a zero/non-finite state");
    std::vector<cd> U(ops + chosen * DD, ops + (chosen + 1) * DD);
    for (cd &z : U) z *= 1.0 / len;
    *index = chosen;
    return launch_gate(s, reinterpret_cast<const double *>(U.data()), k, qubits, 0);
}

}  // namespace qvmhip
