// tile.hip -- gate sequences applied to register-resident blocks of the state.
//
// A tile pass names m "tile qubits".  For every assignment of the other n-m
// qubits one workgroup loads the 2^m amplitudes spanned by the tile qubits,
// applies the pass's gates one after another and writes the block back: the
// whole gate sequence costs one HBM read and one write of the state.  Tile
// qubit sets that include qubits 0..L-1 give contiguous runs of 2^L
// amplitudes, so loads and stores stay coalesced; high-order gate targets are
// brought in by naming them as tile qubits (the load is a strided gather of
// those runs), which is the qubit permutation into an on-chip block.
//
// Inside the workgroup the block lives in registers.  Slot s = t + NT*r of
// the block is register r of thread t, so the low TB = m - RB slot bits are
// thread bits and the high RB bits are register bits (R = 2^RB amplitudes per
// thread).  A gate whose non-diagonal targets sit on register bits runs in
// registers with no data exchange; diagonal gates and control tests run on any
// bit.  When a gate needs a target that sits on a thread bit, the block is
// re-laid out through LDS (REMAP: every thread stores its registers, and loads
// back the slots of a new bit permutation).  Uncontrolled SWAPs are pure
// relabelings of that permutation and move no data.  The host scheduler
// (schedule_tile_ops) turns a pass's op list, written against tile-local bit
// positions, into this slot-space program: it picks which local bits become
// register bits at each REMAP by next use (farthest next use is evicted), and
// ends the pass with the identity layout so the store is coalesced.
//
// Arithmetic per gate is the same as the plain kernels (gates.hip): separate
// complex products summed left to right, built with -ffp-contract=off, so an
// in-order pass is bit-identical to gate-by-gate application.
#include <algorithm>
#include <array>
#include <complex>
#include <cstring>
#include <vector>

#include "qvmhip_internal.h"

namespace qvmhip {

// Slot-space op kinds that only the scheduler emits (after the public ones).
constexpr uint32_t kTileXReg = 16;   // X on register bit (q0 - TB) where ctrl_mask holds
constexpr uint32_t kTileRSwap = 17;  // exchange register bits q0 and q1 (both < RB)
constexpr uint32_t kTileRemap = 18;  // relayout through LDS; new slot bit j <- old bit src[j]
constexpr uint32_t kTileRDiag = 19;  // multiply register r by entry r (m holds R complex entries)
// Uncontrolled 1-qubit ops on register bit (q0 - TB) whose entries have zero
// parts, with those parts left out: every entry real (m[0..3] = u00, u01,
// u10, u11: H, RY), or real diagonal and imaginary off-diagonal (m[0..3] =
// Re u00, Im u01, Im u10, Re u11: RX).
constexpr uint32_t kTileD1Real = 20;
constexpr uint32_t kTileD1RX = 21;
// FMA passes: a run of ZZ phases with one angle (diag(a, b, b, a) on qubit
// pairs, the MaxCut cost layer of QAOA) multiplies amplitude x by
// T[cut(x)], cut(x) = the number of the run's pairs whose bits differ in x,
// T[c] = a^(E - c) b^c.  CUT_PHASE holds the pairs by where their ends sit
// (byte layout in cut_phase_op); the ceil((E + 1) / 16) ops after it are
// DATA ops holding T, which the kernel reads and skips.
constexpr uint32_t kTileCutPhase = 22;
constexpr uint32_t kTileData = 23;
constexpr int kCutMaxEdges = 32;
constexpr int kCutHeader = 192;  // bytes of CUT_PHASE before its table in a packed program

// Register bits per thread (measured on MI355X): 3 (8 amplitudes) for FP64
// and for exact FP32, 4 (16) for FP32 with FMA contraction; fewer for small
// tiles so a workgroup keeps at least 64 threads.
__host__ __device__ constexpr int tile_reg_bits(int m, bool f64, bool fma) {
    return (m - 6) < ((!f64 && fma) ? 4 : 3) ? (m - 6) : ((!f64 && fma) ? 4 : 3);
}

struct TileArgs {
    GroupSpec g;        // tile base: inject zeros at the m tile positions
    uint32_t tq[16];    // global positions of the tile qubits (ascending)
    uint64_t roff[32];  // global offset of register r (slot bits >= TB)
};

template <int TB>
__device__ inline uint64_t thread_offset(const TileArgs &a, uint32_t t) {
    uint64_t o = 0;
#pragma unroll
    for (int b = 0; b < TB; ++b)
        if ((t >> b) & 1u) o |= uint64_t(1) << a.tq[b];
    return o;
}

__device__ __forceinline__ double qfma(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float qfma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// a * b + c and a * b - c as instructions whose result the register allocator
// may place freely.  For __builtin_fma the compiler picks the two-address
// form, whose result takes the register of c: right for accumulating into c,
// a copy of the block where the result replaces another component.  SC: b is
// in scalar registers at FP64.  FP32 operands are always vector registers (see
// operand()).
template <bool SC = true>
__device__ __forceinline__ double fma_to(double a, double b, double c) {
    double r;
    if constexpr (SC)
        asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
    else
        asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
template <bool SC = true>
__device__ __forceinline__ float fma_to(float a, float b, float c) {
    float r;
    asm("v_fma_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
template <bool SC = true>
__device__ __forceinline__ double fms_to(double a, double b, double c) {
    double r;
    if constexpr (SC)
        asm("v_fma_f64 %0, %1, %2, -%3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
    else
        asm("v_fma_f64 %0, %1, %2, -%3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
template <bool SC = true>
__device__ __forceinline__ float fms_to(float a, float b, float c) {
    float r;
    asm("v_fma_f32 %0, %1, %2, -%3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// An op's coefficient as the arithmetic wants it: FP64 stays in scalar
// registers, FP32 is moved to a vector register.  FP32 vector instructions
// with a scalar operand issue at the FP64 rate, without one nearly twice as
// fast (per op over 2^30 amplitudes: RX 113 -> 68 us, general 1q 224 -> 130).
__device__ __forceinline__ double operand(double s) { return s; }
__device__ __forceinline__ float operand(float s) {
    float r;
    asm("v_mov_b32 %0, %1" : "=v"(r) : "s"(s));
    return r;
}

// A move the compiler cannot see through: keeps the block's components out of
// the register tuples of the 16-byte loads and stores.
__device__ __forceinline__ double vmov(double a) {
    double r;
    asm("v_mov_b64 %0, %1" : "=v"(r) : "v"(a));
    return r;
}

// The arithmetic below is written as in-place updates in an order that needs
// no copy of the block: a component is overwritten only by an instruction
// after which its old value has no reader.  The compiler follows that order;
// written as y = f(x) it kept old and new values side by side and moved one
// of them back after every op.

// x *= f (complex).  FMA = false: four separately rounded products, as the
// plain kernels; FMA = true: one product and one fused multiply-add per part.
// SC: f is in scalar registers.
template <typename T, bool FMA, bool SC = false>
__device__ __forceinline__ void cmul(vec2_t<T> &x, T fr, T fi) {
    if constexpr (FMA) {
        const T t = x.y * fi;
        x.y = x.y * fr;
        x.y = qfma(x.x, fi, x.y);
        x.x = fms_to<SC>(x.x, fr, t);
    } else {
        const T t = x.y * fi, u = x.x * fi;
        x.y = x.y * fr;
        x.y = u + x.y;
        x.x = x.x * fr;
        x.x = x.x - t;
    }
}

// (p, q) = (a p + s b q, c p + d q) for real a..d, s = +1 or -1 (NEG); each
// output is its p term plus its q term, as the general complex form rounds it.
template <typename T, bool FMA, bool NEG>
__device__ __forceinline__ void rot2(T &p, T &q, T a, T b, T c, T d) {
    if constexpr (FMA) {
        const T t = q * b;
        q = q * d;
        q = qfma(p, c, q);
        if constexpr (NEG)
            p = fms_to(p, a, t);
        else
            p = fma_to(p, a, t);
    } else {
        const T t = q * b, u = p * c;
        q = q * d;
        q = u + q;
        p = p * a;
        p = NEG ? p - t : p + t;
    }
}

// What the kernels run: the scheduled op list packed into 80-byte slots
// (pack_tile_ops).  `f` says what to do with one bit per case, tested in turn
// as nested one-armed ifs.  A switch over op kinds looks simpler and costs
// far more: the block (32 VGPRs at FP64) is then a value merged from many
// arms, of which the compiler keeps old and new copies -- it moved the whole
// block twice per op and needed 95 VGPRs.  Operands are in the pass's type;
// an op with more than 64 bytes of them runs on into the following slots
// (`f` >> 28 of them).
struct TileDevOp {
    uint32_t f;
    uint32_t a, b, c;  // lane mask, wanted lane bits, register mask (bit r: register r takes part)
    double m[8];
};
static_assert(sizeof(TileDevOp) == 80, "slot size");

enum : uint32_t {
    kF_Bit0 = 1u << 0,   // the target is register bit 0 (.. 3)
    kF_Gen = 1u << 4,    // 1q: general
    kF_GenC = 1u << 5,   // 1q: general, where lane and register controls hold
    kF_Real = 1u << 6,   // 1q: real entries
    kF_RX = 1u << 7,     // 1q: real diagonal, imaginary off-diagonal
    kF_1q = 0xF0u,
    kF_X = 1u << 8,      // exchange register pairs where the lane condition holds
    kF_DL = 1u << 9,     // diagonal: one of two entries per lane, on all registers, those with the
                         // target bit set, or (Mask) those of c
    kF_DL4 = 1u << 10,   // diagonal: one of four entries per lane (bits a & 0xff, a >> 8)
    kF_DR = 1u << 11,    // diagonal: entry by lane condition and target register bit
    kF_RDiag = 1u << 12, // diagonal: entry r on register r
    kF_Out = 1u << 13,   // with DL / DR: qubits outside the tile select the entry pair
    kF_Diag = kF_DL | kF_DL4 | kF_DR | kF_RDiag,
    kF_Remap = 1u << 14,
    kF_Dense2 = 1u << 15,
    kF_Dense2C = 1u << 16,
    kF_SwapC = 1u << 17,
    kF_RSwap = 1u << 18,
    kF_Cut = 1u << 19,
    kF_Rare = kF_Dense2 | kF_Dense2C | kF_SwapC | kF_RSwap | kF_Cut,
    kF_End = 1u << 20,
    kF_Mask = 1u << 21,  // DL on the registers of c
    kF_Id0 = 1u << 22,   // DL: lanes outside the condition keep their amplitudes (entry 0 is 1)
    kF_Neg = 1u << 23,   // DL with Id0: entry 1 is -1
};

// The 80 bytes of a slot, loaded as scalars one op ahead (as 64-bit words:
// half the scalar moves when the next op becomes the current one).
struct TileHead {
    uint64_t w[10];
    __device__ __forceinline__ uint32_t f() const { return (uint32_t)w[0]; }
    __device__ __forceinline__ uint32_t a() const { return (uint32_t)(w[0] >> 32); }
    __device__ __forceinline__ uint32_t b() const { return (uint32_t)w[1]; }
    __device__ __forceinline__ uint32_t c() const { return (uint32_t)(w[1] >> 32); }
    template <typename T>
    __device__ __forceinline__ T m(int i) const {
        if constexpr (sizeof(T) == 8)
            return __longlong_as_double((long long)w[2 + i]);
        else
            return operand(__uint_as_float((uint32_t)(w[2 + i / 2] >> (32 * (i & 1)))));
    }
};

// Operands of an op that is not only its own slot long.
template <typename T>
__device__ __forceinline__ const T *operands(const TileDevOp *op) {
    return reinterpret_cast<const T *>(op->m);
}

// register index with a zero inserted at bit I
template <int I>
__device__ constexpr int rins0(int p) {
    return ((p >> I) << (I + 1)) | (p & ((1 << I) - 1));
}

template <typename T>
__device__ __forceinline__ vec2_t<T> vsel(bool c, vec2_t<T> a, vec2_t<T> b) {
    vec2_t<T> r;
    r.x = c ? a.x : b.x;
    r.y = c ? a.y : b.y;
    return r;
}

// The register ops compute every pair unconditionally and, for controlled
// ops (CTRL), keep the old values by selection where the control bits are not
// all 1 (lane part lane_ok, register part in the op's register mask):
// straight-line code, so the pairs of all registers interleave.

// (xa, xb) = U (xa, xb), each output the sum of its rounded products in
// column order or (FMA) one product and three fused multiply-adds.
template <typename T, int R, int I, bool CTRL, bool FMA>
__device__ __forceinline__ void reg_dense1(vec2_t<T> (&x)[R], const TileHead &h, bool lane_ok) {
    using V = vec2_t<T>;
    const T u00r = h.m<T>(0), u00i = h.m<T>(1), u01r = h.m<T>(2), u01i = h.m<T>(3);
    const T u10r = h.m<T>(4), u10i = h.m<T>(5), u11r = h.m<T>(6), u11i = h.m<T>(7);
#pragma unroll
    for (int p = 0; p < R / 2; ++p) {
        V &a = x[rins0<I>(p)], &b = x[rins0<I>(p) | (1 << I)];
        const V a0 = a, b0 = b;
        if constexpr (FMA) {
            T tr = qfma(b.x, u01r, -(b.y * u01i));
            T ti = qfma(b.x, u01i, b.y * u01r);
            cmul<T, true, true>(b, u11r, u11i);
            b.x = qfma(-a.y, u10i, b.x);
            b.y = qfma(a.y, u10r, b.y);
            b.x = qfma(a.x, u10r, b.x);
            b.y = qfma(a.x, u10i, b.y);
            tr = qfma(-a.y, u00i, tr);
            ti = qfma(a.y, u00r, ti);
            a.y = fma_to(a.x, u00i, ti);
            a.x = fma_to(a.x, u00r, tr);
        } else {
            V s = b, t = a;
            cmul<T, false>(s, u01r, u01i);
            cmul<T, false>(b, u11r, u11i);
            cmul<T, false>(t, u10r, u10i);
            b.x = t.x + b.x;
            b.y = t.y + b.y;
            cmul<T, false>(a, u00r, u00i);
            a.x = a.x + s.x;
            a.y = a.y + s.y;
        }
        if constexpr (CTRL) {
            const bool ok = lane_ok && ((h.c() >> rins0<I>(p)) & 1u);
            a = vsel<T>(ok, a, a0);
            b = vsel<T>(ok, b, b0);
        }
    }
}

// 4x4 on register bits 0 (matrix bit 0) and 1 (matrix bit 1)
template <typename T, int R, bool CTRL, bool FMA>
__device__ __forceinline__ void reg_dense2(vec2_t<T> (&x)[R], const T *__restrict__ u, bool lane_ok, uint32_t regs) {
    using V = vec2_t<T>;
#pragma unroll
    for (int p = 0; p < R / 4; ++p) {
        const int r0 = p << 2;
        V in[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) in[j] = x[r0 | j];
        const bool ok = !CTRL || (lane_ok && ((regs >> r0) & 1u));
#pragma unroll
        for (int row = 0; row < 4; ++row) {
            V y = in[0];
            cmul<T, FMA>(y, u[8 * row], u[8 * row + 1]);
#pragma unroll
            for (int c = 1; c < 4; ++c) {
                const T ur = u[8 * row + 2 * c], ui = u[8 * row + 2 * c + 1];
                if constexpr (FMA) {
                    y.x = qfma(in[c].x, ur, qfma(-in[c].y, ui, y.x));
                    y.y = qfma(in[c].x, ui, qfma(in[c].y, ur, y.y));
                } else {
                    V p = in[c];
                    cmul<T, false>(p, ur, ui);
                    y.x = y.x + p.x;
                    y.y = y.y + p.y;
                }
            }
            x[r0 | row] = CTRL ? vsel<T>(ok, y, in[row]) : y;
        }
    }
}

// The 1-qubit product of reg_dense1 with the terms whose matrix factor is 0
// left out.  x*0 is an exact zero and adding an exact zero leaves a nonzero
// value as it is, so every output is the same rounded value as the general
// form's, in both the separately rounded and the FMA form (an exact-zero
// result may differ in its sign only).  Half the multiplies of reg_dense1.
template <typename T, int R, int I, bool FMA>
__device__ __forceinline__ void reg_dense1_real(vec2_t<T> (&x)[R], T u00, T u01, T u10, T u11) {
#pragma unroll
    for (int p = 0; p < R / 2; ++p) {
        vec2_t<T> &a = x[rins0<I>(p)], &b = x[rins0<I>(p) | (1 << I)];
        rot2<T, FMA, false>(a.x, b.x, u00, u01, u10, u11);
        rot2<T, FMA, false>(a.y, b.y, u00, u01, u10, u11);
    }
}

// u00 = a, u01 = i b, u10 = i c, u11 = d (a, b, c, d real):
// ya = (a xa.re - b xb.im, a xa.im + b xb.re), yb = (d xb.re - c xa.im,
// d xb.im + c xa.re), each sum in the general form's order.
template <typename T, int R, int I, bool FMA>
__device__ __forceinline__ void reg_dense1_rx(vec2_t<T> (&x)[R], T u00, T u01, T u10, T u11) {
#pragma unroll
    for (int p = 0; p < R / 2; ++p) {
        vec2_t<T> &a = x[rins0<I>(p)], &b = x[rins0<I>(p) | (1 << I)];
        rot2<T, FMA, true>(a.x, b.y, u00, u01, u10, u11);
        if constexpr (FMA) {
            const T t = b.x * u01;
            b.x = b.x * u11;
            b.x = qfma(-a.y, u10, b.x);
            a.y = fma_to(a.y, u00, t);
        } else {
            const T t = b.x * u01, s = a.y * u10;
            b.x = b.x * u11;
            b.x = b.x - s;
            a.y = a.y * u00;
            a.y = a.y + t;
        }
    }
}

template <typename T, int R, int I>
__device__ __forceinline__ void reg_x(vec2_t<T> (&x)[R], bool lane_ok, uint32_t regs) {
    using V = vec2_t<T>;
#pragma unroll
    for (int p = 0; p < R / 2; ++p) {
        const int ra = rins0<I>(p), rb = ra | (1 << I);
        const bool ok = lane_ok && ((regs >> ra) & 1u);
        const V xa = x[ra], xb = x[rb];
        x[ra] = vsel<T>(ok, xb, xa);
        x[rb] = vsel<T>(ok, xa, xb);
    }
}

// controlled SWAP of register bits 0 and 1
template <typename T, int R>
__device__ __forceinline__ void reg_swap01(vec2_t<T> (&x)[R], bool lane_ok, uint32_t regs) {
    using V = vec2_t<T>;
#pragma unroll
    for (int p = 0; p < R / 4; ++p) {
        const int r0 = p << 2;
        const bool ok = lane_ok && ((regs >> r0) & 1u);
        const V a = x[r0 | 1], b = x[r0 | 2];
        x[r0 | 1] = vsel<T>(ok, b, a);
        x[r0 | 2] = vsel<T>(ok, a, b);
    }
}

// relabel register bits A < B (no arithmetic)
template <int A, int B>
__device__ constexpr int bit_swapped(int r) {
    return (((r >> A) & 1) == ((r >> B) & 1)) ? r : (r ^ (1 << A) ^ (1 << B));
}

template <typename T, int R, int A, int B>
__device__ __forceinline__ void reg_rswap(vec2_t<T> (&x)[R]) {
    using V = vec2_t<T>;
    V y[R];
#pragma unroll
    for (int r = 0; r < R; ++r) y[r] = x[bit_swapped<A, B>(r)];
#pragma unroll
    for (int r = 0; r < R; ++r) x[r] = y[r];
}

template <typename T, int R>
__device__ __forceinline__ void reg_rswap_any(vec2_t<T> (&x)[R], uint32_t pair) {
#define QH_RS(BIT, A, B)                                        \
    if constexpr ((1 << B) < R) {                               \
        if ((pair >> BIT) & 1u) reg_rswap<T, R, A, B>(x);       \
    }
    QH_RS(0, 0, 1) QH_RS(1, 0, 2) QH_RS(2, 0, 3) QH_RS(3, 1, 2) QH_RS(4, 1, 3) QH_RS(5, 2, 3)
#undef QH_RS
}

// Diagonals.  A diagonal's index has a lane part (the same for all registers)
// and a register part.  No case needs a per-register vector select: the lane
// part picks one entry (or two) per lane once per op, and the register part
// is a scalar choice or a compile-time one.  A lane whose condition fails
// multiplies by exactly 1, which leaves its amplitude's value unchanged; a
// wave without a lane that meets it skips the op.

// apply(x[r]) on the registers an op names: all, those with target bit I set,
// or those of its mask.  The first two are compile-time sets: tested one by
// one, eight registers cost sixteen scalar instructions and branches.
template <typename T, int R, int I, typename F>
__device__ __forceinline__ void on_bit(vec2_t<T> (&x)[R], const F &apply) {
#pragma unroll
    for (int u = 0; u < R / 2; ++u) apply(x[((u >> I) << (I + 1)) | (1 << I) | (u & ((1 << I) - 1))]);
}

template <typename T, int R, typename F>
__device__ __forceinline__ void on_registers(vec2_t<T> (&x)[R], uint32_t f, uint32_t mask, const F &apply) {
    if (f & kF_Mask) {
#pragma unroll
        for (int r = 0; r < R; ++r)
            if ((mask >> r) & 1u) apply(x[r]);
    } else if (f & (kF_Bit0 << 0)) {
        on_bit<T, R, 0>(x, apply);
    } else if (f & (kF_Bit0 << 1)) {
        on_bit<T, R, 1>(x, apply);
    } else if (R > 4 && (f & (kF_Bit0 << 2))) {
        if constexpr (R > 4) on_bit<T, R, 2>(x, apply);
    } else if (R > 8 && (f & (kF_Bit0 << 3))) {
        if constexpr (R > 8) on_bit<T, R, 3>(x, apply);
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r) apply(x[r]);
    }
}

// Flips the sign of v where `bit` is 0x80000000 (0 elsewhere).
__device__ __forceinline__ double flip_sign(double v, uint32_t bit) {
    return __hiloint2double((int)((uint32_t)__double2hiint(v) ^ bit), __double2loint(v));
}
__device__ __forceinline__ float flip_sign(float v, uint32_t bit) { return __uint_as_float(__float_as_uint(v) ^ bit); }

// Register r takes entry c1 when its bit RS is set, c0 otherwise.
template <typename T, int R, int RS, bool FMA>
__device__ __forceinline__ void diag_rbit(vec2_t<T> (&x)[R], T c0r, T c0i, T c1r, T c1i) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const bool one = ((r >> RS) & 1) != 0;
        cmul<T, FMA>(x[r], one ? c1r : c0r, one ? c1i : c0i);
    }
}

// Register r times entry r: a diagonal whose index bits (and controls) are
// all register bits, with its per-register entries worked out by the
// scheduler.
template <typename T, int R, bool FMA>
__device__ __forceinline__ void reg_rdiag(vec2_t<T> (&x)[R], const T *__restrict__ d) {
#pragma unroll
    for (int r = 0; r < R; ++r) cmul<T, FMA, true>(x[r], operand(d[2 * r]), operand(d[2 * r + 1]));
}

// DL, DL4, DR and RDIAG (see the flags).  Out: the bits of the block's base
// index named by b (g0 | g1 << 8 | count << 16) select one of the op's entry
// pairs; bit 20 + sel of b is set where that pair is (1, 1), which is skipped.
template <typename T, int R, bool FMA>
__device__ __forceinline__ void reg_diag(vec2_t<T> (&x)[R], const TileHead &h, const TileDevOp *__restrict__ op,
                                         uint32_t t, uint64_t gb) {
    const uint32_t f = h.f();
    if (f & kF_RDiag) {
        reg_rdiag<T, R, FMA>(x, operands<T>(op));
    } else if (f & kF_DL4) {
        const bool b0 = ((t >> (h.a() & 0xFFu)) & 1u) != 0, b1 = ((t >> (h.a() >> 8)) & 1u) != 0;
        const T ra = b0 ? h.m<T>(2) : h.m<T>(0), ia = b0 ? h.m<T>(3) : h.m<T>(1);
        const T rb = b0 ? h.m<T>(6) : h.m<T>(4), ib = b0 ? h.m<T>(7) : h.m<T>(5);
        const T dr = b1 ? rb : ra, di = b1 ? ib : ia;
#pragma unroll
        for (int r = 0; r < R; ++r) cmul<T, FMA>(x[r], dr, di);
    } else {
        // the pair of entries: by default the first, with qubits outside the
        // tile the one they select (two pairs fit the slot)
        T e0r = h.m<T>(0), e0i = h.m<T>(1), e1r = h.m<T>(2), e1i = h.m<T>(3);
        uint32_t want = h.b();
        bool go = true;
        if (f & kF_Out) {
            const uint32_t d = h.b();
            uint32_t sel = (uint32_t)(gb >> (d & 63u)) & 1u;
            want = h.a();
            if (((d >> 16) & 3u) == 2u) {
                sel |= ((uint32_t)(gb >> ((d >> 8) & 63u)) & 1u) << 1;
                const T *m = operands<T>(op) + 4 * sel;
                e0r = operand(m[0]), e0i = operand(m[1]), e1r = operand(m[2]), e1i = operand(m[3]);
            } else {
                e0r = sel ? h.m<T>(4) : e0r;
                e0i = sel ? h.m<T>(5) : e0i;
                e1r = sel ? h.m<T>(6) : e1r;
                e1i = sel ? h.m<T>(7) : e1i;
            }
            go = ((d >> (20 + sel)) & 1u) == 0;
        }
        if (go) {
            const bool hit = (t & h.a()) == want;
            if (f & kF_DR) {
                // entries (lane, register): the pair without the lane condition, m[4..7] with it
                T c0r = e0r, c0i = e0i, c1r = e1r, c1i = e1i;
                if (!(f & kF_Out)) {
                    c0r = hit ? h.m<T>(4) : c0r;
                    c0i = hit ? h.m<T>(5) : c0i;
                    c1r = hit ? h.m<T>(6) : c1r;
                    c1i = hit ? h.m<T>(7) : c1i;
                }
                if (f & (kF_Bit0 << 0)) {
                    diag_rbit<T, R, 0, FMA>(x, c0r, c0i, c1r, c1i);
                } else if (f & (kF_Bit0 << 1)) {
                    diag_rbit<T, R, 1, FMA>(x, c0r, c0i, c1r, c1i);
                } else if (f & (kF_Bit0 << 2)) {
                    if constexpr (R > 4) diag_rbit<T, R, 2, FMA>(x, c0r, c0i, c1r, c1i);
                } else {
                    if constexpr (R > 8) diag_rbit<T, R, 3, FMA>(x, c0r, c0i, c1r, c1i);
                }
            } else if (!(f & kF_Id0) || __ballot(hit) != 0) {
                if (f & kF_Neg) {
                    const uint32_t bit = hit ? 0x80000000u : 0u;
                    on_registers<T, R>(x, f, h.c(), [&](vec2_t<T> &v) {
                        v.x = flip_sign(v.x, bit);
                        v.y = flip_sign(v.y, bit);
                    });
                } else if (h.a() == 0) {  // the same entry on every lane
                    on_registers<T, R>(x, f, h.c(), [&](vec2_t<T> &v) { cmul<T, FMA, true>(v, e1r, e1i); });
                } else {
                    const T dr = hit ? e1r : e0r, di = hit ? e1i : e0i;
                    on_registers<T, R>(x, f, h.c(), [&](vec2_t<T> &v) { cmul<T, FMA>(v, dr, di); });
                }
            }
        }
    }
}

// CUT_PHASE (the layout of its bytes is described at cut_phase_op; the phase
// table T follows them): T goes to LDS, each thread counts the
// cut pairs of its amplitudes and multiplies register r by T[cut].
template <typename T, int R, int TB, bool FMA>
__device__ __forceinline__ void reg_cut_phase(vec2_t<T> (&x)[R], const TileDevOp *__restrict__ op,
                                              vec2_t<T> *sa, uint32_t t, uint64_t gb) {
    const uint8_t *b = (const uint8_t *)op->m;
    const uint32_t E = b[0];
    // values derived from t stay inside this op (hoisted out of the op loop
    // they would hold registers through every other op)
    asm volatile("" : "+v"(t));
    __syncthreads();  // earlier readers of sa are done
    if (t <= E) sa[t] = reinterpret_cast<const vec2_t<T> *>(b + kCutHeader)[t];
    uint32_t c = 0, A = 0;
#pragma unroll 4  // by four: one scalar load per four pairs (a full unroll computed the pair terms ahead and spilled)
    for (uint32_t i = 0; i < E; ++i) {
        {
            const uint32_t cls = b[72 + i], e0 = b[8 + 2 * i], e1 = b[9 + 2 * i];
            if (cls == 0u) c += ((t >> e0) ^ (t >> e1)) & 1u;                          // LL
            else if (cls == 1u) c += ((t >> e0) ^ (uint32_t)(gb >> e1)) & 1u;          // LO
            else if (cls == 2u) A |= ((t >> e0) & 1u) << i;                            // LR
            else if (cls == 3u) A |= ((uint32_t)(gb >> e1) & 1u) << i;                 // RO
            else if (cls == 5u) c += (uint32_t)((gb >> e0) ^ (gb >> e1)) & 1u;         // OO
        }
    }
    const uint32_t *B = (const uint32_t *)(b + 128);
    __syncthreads();  // the table is in LDS
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const vec2_t<T> f = sa[c + (uint32_t)__popc(A ^ B[r])];
        cmul<T, FMA>(x[r], f.x, f.y);
        __builtin_amdgcn_sched_barrier(0);  // one table read at a time: R reads ahead hold 2R registers
    }
}

// LDS address of slot s: register row r = s >> TB of NT slots is padded by
// one element, so a thread's store of register r is t + r*(NT+1) (a fixed
// offset from t), and a lane bit that a REMAP takes from register bit b of the
// old layout steps by (NT+1)*2^b, i.e. 2^b modulo the bank count: with the
// scheduler pairing vacated lane bit p with evicted register bit p, the lanes
// of one LDS access hit distinct banks.
template <int TB>
__device__ __forceinline__ uint32_t lds_addr(uint32_t s) {
    return s + (s >> TB);
}

// src4: the op's first 16 operand bytes as four words; byte j is the old
// slot bit of new slot bit j.  Blocks go through LDS one component at a time
// (real parts, then imaginary parts): the exchange buffer is half a block, and
// more workgroups fit on a CU.
template <typename T, int R, int TB>
__device__ __forceinline__ void reg_remap(vec2_t<T> (&x)[R], T *sa, const uint32_t (&src4)[4], uint32_t t) {
    constexpr uint32_t NT = 1u << TB;
    auto src = [&](int j) -> uint32_t { return (src4[j >> 2] >> (8 * (j & 3))) & 0xFFu; };
    uint32_t base = 0;
#pragma unroll
    for (int j = 0; j < TB; ++j)
        if ((t >> j) & 1u) base |= 1u << src(j);
    uint32_t pw[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) pw[b] = (1 << b) < R ? (1u << src(TB + b)) : 0u;
    auto addr = [&](int r) -> uint32_t {
        uint32_t off = 0;
#pragma unroll
        for (int b = 0; (1 << b) < R; ++b)
            if ((r >> b) & 1) off |= pw[b];
        return lds_addr<TB>(base | off);
    };
    __syncthreads();  // readers of the previous layout are done with sa
#pragma unroll
    for (int r = 0; r < R; ++r) sa[t + (uint32_t)r * (NT + 1)] = x[r].x;
    __syncthreads();
    T re[R];
#pragma unroll
    for (int r = 0; r < R; ++r) re[r] = sa[addr(r)];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) sa[t + (uint32_t)r * (NT + 1)] = x[r].y;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
        x[r].x = re[r];
        x[r].y = sa[addr(r)];
    }
}

// One tile: load the 2^M amplitudes of tile `tile` into registers, run the
// scheduled op list, store.  Shared by the single-state and batched kernels.
template <typename T, int M, int RB>
__device__ __forceinline__ void tile_load(const vec2_t<T> *__restrict__ psi, const TileArgs &a, uint64_t gb,
                                          uint64_t toff, vec2_t<T> (&x)[1 << RB]) {
    const vec2_t<T> *p = psi + gb + toff;
#pragma unroll
    for (int r = 0; r < (1 << RB); ++r) x[r] = ldg<true>(&p[a.roff[r]]);
    if constexpr (sizeof(T) == 8) {
#pragma unroll
        for (int r = 0; r < (1 << RB); ++r) {
            x[r].x = vmov(x[r].x);
            x[r].y = vmov(x[r].y);
        }
    }
}

template <typename T, int M, int RB>
__device__ __forceinline__ void tile_store(vec2_t<T> *__restrict__ psi, const TileArgs &a, uint64_t gb,
                                           uint64_t toff, const vec2_t<T> (&x)[1 << RB]) {
    // recompute the store addresses instead of keeping them live across
    // the op loop (the barrier is on the offset: on the pointer itself it
    // would hide the global address space, and flat stores count against
    // the LDS and scalar-load waits of the next tile)
    uint64_t o = gb + toff;
    asm volatile("" : "+v"(o));
    vec2_t<T> *p = psi + o;
#pragma unroll
    for (int r = 0; r < (1 << RB); ++r) {
        vec2_t<T> v = x[r];
        if constexpr (sizeof(T) == 8) {
            v.x = vmov(v.x);
            v.y = vmov(v.y);
        }
        stg<true>(&p[a.roff[r]], v);
    }
}

// Run a packed op list (ended by kF_End) on the block held in x.  Each op's
// slot is loaded as scalars while the op before it runs: read on demand, the
// load was a wait of some 500 cycles in every op.
// CUT: the op list holds CUT_PHASE ops (FMA passes only).  Kernels without
// them are built without that code: its registers and code size slow every
// other op down.
template <typename T, int M, int RB, bool FMA, bool CUT>
__device__ __forceinline__ void tile_ops(vec2_t<T> (&x)[1 << RB], const TileDevOp *__restrict__ op, T *sa, uint64_t gb) {
    constexpr int R = 1 << RB, TB = M - RB;
    const uint32_t t = threadIdx.x;
    TileHead h = *reinterpret_cast<const TileHead *>(op);
    while (!(h.f() & kF_End)) {
        const TileDevOp *next = op + 1 + (h.f() >> 28);
        const TileHead hn = *reinterpret_cast<const TileHead *>(next);
        const uint32_t f = h.f();
// CALL(I) for the op's target register bit I
#define QH_BITS(CALL)                          \
    if (f & (kF_Bit0 << 0)) {                  \
        CALL(0);                               \
    } else if (f & (kF_Bit0 << 1)) {           \
        if constexpr (RB > 1) CALL(1);         \
    } else if (f & (kF_Bit0 << 2)) {           \
        if constexpr (RB > 2) CALL(2);         \
    } else {                                   \
        if constexpr (RB > 3) CALL(3);         \
    }
        if (f & kF_1q) {
            if (f & kF_RX) {
#define QH_C(I) reg_dense1_rx<T, R, I, FMA>(x, h.m<T>(0), h.m<T>(1), h.m<T>(2), h.m<T>(3))
                QH_BITS(QH_C)
#undef QH_C
            } else if (f & kF_Gen) {
#define QH_C(I) reg_dense1<T, R, I, false, FMA>(x, h, true)
                QH_BITS(QH_C)
#undef QH_C
            } else if (f & kF_Real) {
#define QH_C(I) reg_dense1_real<T, R, I, FMA>(x, h.m<T>(0), h.m<T>(1), h.m<T>(2), h.m<T>(3))
                QH_BITS(QH_C)
#undef QH_C
            } else {
                const bool lane_ok = (t & h.a()) == h.b();
#define QH_C(I) reg_dense1<T, R, I, true, FMA>(x, h, lane_ok)
                QH_BITS(QH_C)
#undef QH_C
            }
        } else if (f & kF_Diag) {
            reg_diag<T, R, FMA>(x, h, op, t, gb);
        } else if (f & kF_X) {
            const bool lane_ok = (t & h.a()) == h.b();
#define QH_C(I) reg_x<T, R, I>(x, lane_ok, h.c())
            QH_BITS(QH_C)
#undef QH_C
        } else if (f & kF_Remap) {
            const uint32_t src4[4] = {(uint32_t)h.w[2], (uint32_t)(h.w[2] >> 32), (uint32_t)h.w[3],
                                      (uint32_t)(h.w[3] >> 32)};
            reg_remap<T, R, TB>(x, sa, src4, t);
        } else {
            const bool lane_ok = (t & h.a()) == h.b();
            if (f & kF_Dense2) {
                reg_dense2<T, R, false, FMA>(x, operands<T>(op), true, 0u);
            } else if (f & kF_Dense2C) {
                reg_dense2<T, R, true, FMA>(x, operands<T>(op), lane_ok, h.c());
            } else if (f & kF_SwapC) {
                reg_swap01<T, R>(x, lane_ok, h.c());
            } else if (f & kF_RSwap) {
                reg_rswap_any<T, R>(x, h.c());
            } else {
                if constexpr (FMA && CUT)
                    reg_cut_phase<T, R, TB, FMA>(x, op, reinterpret_cast<vec2_t<T> *>(sa), t, gb);
            }
        }
#undef QH_BITS
        h = hn;
        op = next;
    }
}

// FP32 FMA forms are held to eight waves per SIMD, which limits their scalar
// registers to 96 (layered circuit, 28 qubits: 1791 -> 1742 us per pass); the
// FP64 forms lose by it (exact 3502 -> 4366 us, FMA unchanged).
template <typename T, int M, int RB, bool FMA, bool CUT>
__global__ __launch_bounds__(1 << (M - RB))
__attribute__((amdgpu_waves_per_eu(FMA && sizeof(T) == 4 ? 8 : 1))) void k_tile(vec2_t<T> *__restrict__ psi, const TileArgs a,
                                                       const TileDevOp *__restrict__ ops) {
    using V = vec2_t<T>;
    // the remap buffer: one component of the block (2^M reals, padded rows)
    __shared__ __align__(16) T sa[(1 << M) + (1 << RB)];
    const uint64_t toff = thread_offset<M - RB>(a, threadIdx.x);
    // One tile per workgroup (grid-striding only past the dispatch limit):
    // many resident workgroups overlap each other's loads, ops and stores.
    for (uint64_t tile = xcd_block(blockIdx.x, gridDim.x); tile < a.g.ngroups; tile += gridDim.x) {
        V x[1 << RB];
        const uint64_t gb = group_base(a.g, tile);
        tile_load<T, M, RB>(psi, a, gb, toff, x);
        tile_ops<T, M, RB, FMA, CUT>(x, ops, sa, gb);
        tile_store<T, M, RB>(psi, a, gb, toff, x);
    }
}

// Batched form: many states of one buffer, one entry per state.  Work block
// b of a launch belongs to entry blk_ent[b] (a host-built map, one load
// instead of a search) and covers tiles [(b - block_start) * CH, ... + CH) of
// that entry's state.
// The op lists of all entries live in one device buffer passed to the kernel
// as a restrict argument; an entry holds its byte offset there.  (A pointer
// read from memory would not be known to be unaliased with the state, and
// the op loads would become per-lane vector loads with every op field in
// vector registers instead of scalar loads into SGPRs.)
struct TileEntry {
    TileArgs args;
    uint64_t amp_offset;   // first amplitude of the state in the batch buffer
    uint64_t block_start;  // first work block of the launch that works on this entry
    uint64_t op_off;       // byte offset of the entry's scheduled ops in the op buffer
    // state qubits that no earlier pass or gate of the run has touched: the
    // run starts from |0...0>, so a block whose base index has one of them set
    // is all zeros before this pass, and every tile op keeps it zero
    uint64_t zero_mask;
    uint32_t from_zero;    // 1: the state is |0...0>, built in registers instead of loaded
};

// ZERO: some entry of the launch starts from |0...0> or has all-zero
// blocks; launches without (every level after the first few) are built
// without that code.
template <typename T, int M, int RB, bool FMA, bool CUT, bool ZERO>
__global__ __launch_bounds__(1 << (M - RB))
__attribute__((amdgpu_waves_per_eu(FMA && sizeof(T) == 4 ? 8 : 1))) void k_tile_batch(
    vec2_t<T> *__restrict__ base, const TileEntry *__restrict__ ent, const uint32_t *__restrict__ blk_ent,
    uint64_t total_blocks, uint32_t tiles_per_block, const char *__restrict__ op_buf) {
    using V = vec2_t<T>;
    // the remap buffer: one component of the block (2^M reals, padded rows)
    __shared__ __align__(16) T sa[(1 << M) + (1 << RB)];
    // round robin over the XCDs (no xcd_block): work blocks of different
    // entries differ in cost, and contiguous shares per XCD measured 5-6 %
    // slower on the 512-instance QAOA batch
    for (uint64_t b = blockIdx.x; b < total_blocks; b += gridDim.x) {
        const TileEntry &e = ent[blk_ent[b]];
        const uint64_t toff = thread_offset<M - RB>(e.args, threadIdx.x);
        const uint64_t first = (b - e.block_start) * tiles_per_block;
        const uint64_t last = first + tiles_per_block < e.args.g.ngroups ? first + tiles_per_block : e.args.g.ngroups;
        V *psi = base + e.amp_offset;
        for (uint64_t tile = first; tile < last; ++tile) {
            V x[1 << RB];
            const uint64_t gb = group_base(e.args.g, tile);
            if (!ZERO) {
                tile_load<T, M, RB>(psi, e.args, gb, toff, x);
                tile_ops<T, M, RB, FMA, CUT>(x, (const TileDevOp *)(op_buf + e.op_off), sa, gb);
                tile_store<T, M, RB>(psi, e.args, gb, toff, x);
                continue;
            }
            if (gb & e.zero_mask) {
                // an all-zero block stays zero: the first pass of a run stores
                // it (the buffer holds the previous run), later passes leave
                // the zeros in place
                if (e.from_zero) {
#pragma unroll
                    for (int r = 0; r < (1 << RB); ++r) x[r].x = x[r].y = T(0);
                    tile_store<T, M, RB>(psi, e.args, gb, toff, x);
                }
                continue;
            }
            if (e.from_zero) {
                // the first pass of a batch run: |0...0> needs no read
#pragma unroll
                for (int r = 0; r < (1 << RB); ++r) {
                    x[r].x = (gb + toff + e.args.roff[r] == 0) ? T(1) : T(0);
                    x[r].y = T(0);
                }
            } else {
                tile_load<T, M, RB>(psi, e.args, gb, toff, x);
            }
            tile_ops<T, M, RB, FMA, CUT>(x, (const TileDevOp *)(op_buf + e.op_off), sa, gb);
            tile_store<T, M, RB>(psi, e.args, gb, toff, x);
        }
    }
}

// ---------------------------------------------------------------------------
// Host side.

int check_tile_ops(int dtype, uint32_t m, uint32_t nops, const qvmhip_tile_op *ops) {
    if (m < 8 || m > 13 || (m == 13 && dtype == QVMHIP_F64))
        return fail(QVMHIP_EINVAL, "tile size m must be 8..12 (F64) or 8..13 (F32)");
    for (uint32_t o = 0; o < nops; ++o) {
        const qvmhip_tile_op &op = ops[o];
        if (op.kind < QVMHIP_TILE_DENSE1 || op.kind > QVMHIP_TILE_GDIAG)
            return fail(QVMHIP_EINVAL, "unknown tile op kind");
        if (op.kind == QVMHIP_TILE_GDIAG) {
            const uint32_t ng = op.q1 >> 16;
            if (op.q0 >= m) return fail(QVMHIP_EINVAL, "tile op qubit out of range");
            if (ng < 1 || ng > 2) return fail(QVMHIP_EINVAL, "GDIAG reads one or two outside qubits");
            if (op.ctrl_mask) return fail(QVMHIP_EINVAL, "GDIAG takes no controls");
            continue;
        }
        const bool two = op.kind != QVMHIP_TILE_DENSE1 && op.kind != QVMHIP_TILE_DIAG1;
        if (op.q0 >= m || (two && (op.q1 >= m || op.q1 == op.q0)))
            return fail(QVMHIP_EINVAL, "tile op qubit out of range");
        if (m < 32 && (op.ctrl_mask >> m)) return fail(QVMHIP_EINVAL, "tile op control outside the tile");
        if ((op.ctrl_mask >> op.q0) & 1u || (two && ((op.ctrl_mask >> op.q1) & 1u)))
            return fail(QVMHIP_EINVAL, "tile op control overlaps its targets");
    }
    return QVMHIP_OK;
}

int check_tile_globals(uint32_t n, uint32_t m, const uint32_t *tq, uint32_t nops, const qvmhip_tile_op *ops) {
    for (uint32_t o = 0; o < nops; ++o) {
        const qvmhip_tile_op &op = ops[o];
        if (op.kind != QVMHIP_TILE_GDIAG) continue;
        const uint32_t ng = op.q1 >> 16;
        const uint32_t g[2] = {op.q1 & 0xffu, (op.q1 >> 8) & 0xffu};
        for (uint32_t k = 0; k < ng; ++k) {
            if (g[k] >= n) return fail(QVMHIP_EINVAL, "GDIAG qubit out of range");
            for (uint32_t i = 0; i < m; ++i)
                if (tq[i] == g[k]) return fail(QVMHIP_EINVAL, "GDIAG outside qubit is a tile qubit");
        }
        if (ng == 2 && g[0] == g[1]) return fail(QVMHIP_EINVAL, "GDIAG outside qubits repeat");
    }
    return QVMHIP_OK;
}

namespace {

// A scheduled DIAG1 / DIAG2 / CPHASE whose index bits and controls are all
// register bits becomes a register diagonal: entry r is the factor register
// r takes (1 where the controls are not met).
bool to_register_diagonal(qvmhip_tile_op &o, int tb, int rb) {
    if (o.kind != QVMHIP_TILE_DIAG1 && o.kind != QVMHIP_TILE_DIAG2 && o.kind != QVMHIP_TILE_CPHASE) return false;
    const bool two = o.kind != QVMHIP_TILE_DIAG1;
    const uint32_t lanes = (1u << tb) - 1u;
    if ((int)o.q0 < tb || (two && (int)o.q1 < tb) || (o.ctrl_mask & lanes)) return false;
    const uint32_t rcm = o.ctrl_mask >> tb, b0 = o.q0 - tb, b1 = two ? o.q1 - tb : 0u;
    double f[32];
    for (int r = 0; r < (1 << rb); ++r) {
        double re = 1.0, im = 0.0;
        const uint32_t ur = (uint32_t)r;
        if ((ur & rcm) == rcm) {
            const uint32_t j0 = (ur >> b0) & 1u, j1 = two ? (ur >> b1) & 1u : 0u;
            if (o.kind == QVMHIP_TILE_CPHASE) {
                if (j0 && j1) {
                    re = o.m[0];
                    im = o.m[1];
                }
            } else {
                const uint32_t j = j0 | (j1 << 1);
                re = o.m[2 * j];
                im = o.m[2 * j + 1];
            }
        }
        f[2 * r] = re;
        f[2 * r + 1] = im;
    }
    o.kind = kTileRDiag;
    o.q0 = o.q1 = o.ctrl_mask = 0;
    std::memset(o.m, 0, sizeof(o.m));
    std::memcpy(o.m, f, sizeof(double) * 2 * (1 << rb));
    return true;
}

// An uncontrolled 1-qubit op whose entries are all real, or whose diagonal is
// real and off-diagonal imaginary, becomes the matching reduced kind.
void to_split_dense1(qvmhip_tile_op &o) {
    const double *u = o.m;  // u00 = (u[0], u[1]), u01 = (u[2], u[3]), u10 = (u[4], u[5]), u11 = (u[6], u[7])
    double v[4];
    if (u[1] == 0.0 && u[3] == 0.0 && u[5] == 0.0 && u[7] == 0.0) {
        o.kind = kTileD1Real;
        v[0] = u[0], v[1] = u[2], v[2] = u[4], v[3] = u[6];
    } else if (u[1] == 0.0 && u[2] == 0.0 && u[4] == 0.0 && u[7] == 0.0) {
        o.kind = kTileD1RX;
        v[0] = u[0], v[1] = u[3], v[2] = u[5], v[3] = u[6];
    } else {
        return;
    }
    std::memset(o.m, 0, sizeof(o.m));
    std::memcpy(o.m, v, sizeof(v));
}

// A public op that is a ZZ phase diag(a, b, b, a) between two qubits, each
// a tile bit (local position) or a state qubit outside the tile.
struct ZZEdge {
    std::complex<double> a, b;
    int end[2];  // local position, or 64 + outside state qubit
};

bool zz_edge(const qvmhip_tile_op &op, ZZEdge &e) {
    auto c = [&](int i) { return std::complex<double>(op.m[2 * i], op.m[2 * i + 1]); };
    if (op.kind == QVMHIP_TILE_DIAG2 && op.ctrl_mask == 0) {
        if (!(c(0) == c(3) && c(1) == c(2))) return false;
        e.a = c(0), e.b = c(1);
        e.end[0] = (int)op.q0, e.end[1] = (int)op.q1;
        return true;
    }
    if (op.kind != QVMHIP_TILE_GDIAG) return false;
    const uint32_t ng = op.q1 >> 16, g0 = op.q1 & 0xFFu, g1 = (op.q1 >> 8) & 0xFFu;
    if (ng == 1) {  // entry index: local bit | outside bit << 1
        if (!(c(0) == c(3) && c(1) == c(2))) return false;
        e.a = c(0), e.b = c(1);
        e.end[0] = (int)op.q0, e.end[1] = 64 + (int)g0;
        return true;
    }
    // both ends outside: entries must not depend on the local bit
    for (int i = 0; i < 8; i += 2)
        if (!(c(i) == c(i + 1))) return false;
    if (!(c(0) == c(6) && c(2) == c(4))) return false;
    e.a = c(0), e.b = c(2);
    e.end[0] = 64 + (int)g0, e.end[1] = 64 + (int)g1;
    return true;
}

// Local positions an op reads or changes (a ZZ phase with both ends outside
// the tile touches none).
uint32_t touched_bits(const qvmhip_tile_op &op) {
    ZZEdge e;
    if (zz_edge(op, e)) {
        uint32_t msk = 0;
        for (int k = 0; k < 2; ++k)
            if (e.end[k] < 64) msk |= 1u << e.end[k];
        return msk;
    }
    uint32_t msk = (1u << op.q0) | op.ctrl_mask;
    if (op.kind == QVMHIP_TILE_DENSE2 || op.kind == QVMHIP_TILE_DIAG2 || op.kind == QVMHIP_TILE_CPERM ||
        op.kind == QVMHIP_TILE_SWAP || op.kind == QVMHIP_TILE_CPHASE)
        msk |= 1u << op.q1;
    return msk;
}

bool diagonal_public(uint32_t kind) {
    return kind == QVMHIP_TILE_DIAG1 || kind == QVMHIP_TILE_DIAG2 || kind == QVMHIP_TILE_CPHASE ||
           kind == QVMHIP_TILE_GDIAG;
}

// Ops in layers: op i goes one layer after the latest earlier op it does
// not commute with (a shared bit, unless both are diagonal); within a layer
// the ZZ phases come first, grouped by angle, in their original order.
std::vector<qvmhip_tile_op> layer_order(const qvmhip_tile_op *in, uint32_t nin) {
    std::vector<uint32_t> level(nin, 0), bits(nin);
    std::vector<bool> diag(nin), zz(nin);
    std::vector<ZZEdge> edge(nin);
    for (uint32_t i = 0; i < nin; ++i) {
        bits[i] = touched_bits(in[i]);
        diag[i] = diagonal_public(in[i].kind);
        zz[i] = zz_edge(in[i], edge[i]);
        for (uint32_t j = 0; j < i; ++j)
            if ((bits[i] & bits[j]) && !(diag[i] && diag[j])) level[i] = std::max(level[i], level[j] + 1);
    }
    // angle group of each ZZ phase: index of the first ZZ phase of its level with the same entries
    std::vector<uint32_t> group(nin, UINT32_MAX);
    for (uint32_t i = 0; i < nin; ++i) {
        if (!zz[i]) continue;
        group[i] = i;
        for (uint32_t j = 0; j < i; ++j) {
            if (zz[j] && level[j] == level[i] && edge[j].a == edge[i].a && edge[j].b == edge[i].b) {
                group[i] = group[j];
                break;
            }
        }
    }
    std::vector<uint32_t> order(nin);
    for (uint32_t i = 0; i < nin; ++i) order[i] = i;
    std::stable_sort(order.begin(), order.end(), [&](uint32_t x, uint32_t y) {
        if (level[x] != level[y]) return level[x] < level[y];
        if (zz[x] != zz[y]) return (bool)zz[x];
        if (zz[x]) return group[x] < group[y];
        return false;
    });
    std::vector<qvmhip_tile_op> out(nin);
    for (uint32_t i = 0; i < nin; ++i) out[i] = in[order[i]];
    return out;
}

// Local bits an op needs on register bits (its non-diagonal targets).
uint32_t reg_need(const qvmhip_tile_op &op) {
    switch (op.kind) {
        case QVMHIP_TILE_DENSE1: return 1u << op.q0;
        case QVMHIP_TILE_DENSE2: return (1u << op.q0) | (1u << op.q1);
        case QVMHIP_TILE_CPERM: return 1u << op.q0;
        case QVMHIP_TILE_SWAP: return op.ctrl_mask ? ((1u << op.q0) | (1u << op.q1)) : 0u;
        default: return 0u;
    }
}

struct Layout {
    int m, tb, rb;
    int l2s[16], s2l[16];  // local bit <-> slot bit
    void swap_slots(int a, int b) {
        const int la = s2l[a], lb = s2l[b];
        s2l[a] = lb;
        s2l[b] = la;
        l2s[la] = b;
        l2s[lb] = a;
    }
    bool identity() const {
        for (int i = 0; i < m; ++i)
            if (l2s[i] != i) return false;
        return true;
    }
    uint32_t slot_mask(uint32_t local_mask) const {
        uint32_t o = 0;
        for (int i = 0; i < m; ++i)
            if ((local_mask >> i) & 1u) o |= 1u << l2s[i];
        return o;
    }
};

qvmhip_tile_op remap_op(const Layout &from, const int *new_s2l) {
    qvmhip_tile_op o;
    std::memset(&o, 0, sizeof(o));
    o.kind = kTileRemap;
    uint8_t src[16] = {0};
    for (int j = 0; j < from.m; ++j) src[j] = (uint8_t)from.l2s[new_s2l[j]];
    std::memcpy(o.m, src, sizeof(src));
    return o;
}

// Whether two consecutive ops are ZZ phases of one angle.
bool has_cut_run(const std::vector<qvmhip_tile_op> &ops) {
    ZZEdge prev, e;
    bool have = false;
    for (const qvmhip_tile_op &o : ops) {
        const bool z = zz_edge(o, e);
        if (z && have && e.a == prev.a && e.b == prev.b) return true;
        have = z;
        prev = e;
    }
    return false;
}

// CUT_PHASE for a run of ZZ phases of one angle under layout L, followed by
// its DATA ops.  Bytes of m: [0] E (pairs, <= 32), [1] number of DATA ops;
// pair i: ends at bytes 8 + 2i and 9 + 2i, class at byte 72 + i; bytes
// 128..191: B[r] (uint32, r < 16).  Classes by where the ends sit: LL (two
// thread bits), LO (thread bit, outside qubit), LR (thread bit, register
// bit), RO (register bit, outside qubit), RR (two register bits), OO (two
// outside qubits).  For thread t, register r and block base gb:
//   cut = sum over LL, LO, OO pairs of (bit ^ bit) + popc(A ^ B[r])
// where bit i of A is t's thread bit (LR) or gb's outside bit (RO) of pair
// i, and bit i of B[r] is r's register bit (LR, RO) or the xor of r's two
// register bits (RR).
enum : uint8_t { kCutLL = 0, kCutLO = 1, kCutLR = 2, kCutRO = 3, kCutRR = 4, kCutOO = 5 };

void cut_phase_op(const Layout &L, const std::vector<ZZEdge> &run, std::vector<qvmhip_tile_op> &out) {
    struct End {
        int kind;  // 0 thread bit, 1 register bit, 2 outside qubit
        int pos;
    };
    auto where = [&](int end) -> End {
        if (end >= 64) return {2, end - 64};
        const int sbit = L.l2s[end];
        return sbit < L.tb ? End{0, sbit} : End{1, sbit - L.tb};
    };
    qvmhip_tile_op o;
    std::memset(&o, 0, sizeof(o));
    o.kind = kTileCutPhase;
    uint8_t *b = (uint8_t *)o.m;
    const int E = (int)run.size(), ndata = (E + 1 + 15) / 16;
    b[0] = (uint8_t)E;
    b[1] = (uint8_t)ndata;
    uint32_t B[16] = {0};
    for (int i = 0; i < E; ++i) {
        End x = where(run[i].end[0]), y = where(run[i].end[1]);
        if (x.kind > y.kind) std::swap(x, y);
        uint8_t cls;
        if (x.kind == 0) cls = y.kind == 0 ? kCutLL : (y.kind == 1 ? kCutLR : kCutLO);
        else if (x.kind == 1) cls = y.kind == 1 ? kCutRR : kCutRO;
        else cls = kCutOO;
        b[72 + i] = cls;
        b[8 + 2 * i] = (uint8_t)x.pos;
        b[9 + 2 * i] = (uint8_t)y.pos;
        for (int r = 0; r < (1 << L.rb); ++r) {
            uint32_t v = 0;
            if (cls == kCutLR) v = (uint32_t)(r >> y.pos) & 1u;
            else if (cls == kCutRO) v = (uint32_t)(r >> x.pos) & 1u;
            else if (cls == kCutRR) v = (uint32_t)((r >> x.pos) ^ (r >> y.pos)) & 1u;
            B[r] |= v << i;
        }
    }
    std::memcpy(b + 128, B, sizeof(B));
    out.push_back(o);
    // T[c] = a^(E - c) b^c
    for (int d = 0; d < ndata; ++d) {
        qvmhip_tile_op t;
        std::memset(&t, 0, sizeof(t));
        t.kind = kTileData;
        for (int k = 0; k < 16 && 16 * d + k <= E; ++k) {
            const int c = 16 * d + k;
            std::complex<double> v(1.0, 0.0);
            for (int j = 0; j < E - c; ++j) v *= run[0].a;
            for (int j = 0; j < c; ++j) v *= run[0].b;
            t.m[2 * k] = v.real();
            t.m[2 * k + 1] = v.imag();
        }
        out.push_back(t);
    }
}

}  // namespace

// Turn a pass's op list (tile-local bit positions) into the slot-space
// program the kernel runs.  `pin` places the targets of 2-qubit dense ops and
// controlled SWAPs on register bits 0 and 1.
void schedule_tile_ops(int dtype, bool fma, uint32_t m, const qvmhip_tile_op *in_ops, uint32_t nin,
                       std::vector<qvmhip_tile_op> &out) {
    Layout L;
    L.m = (int)m;
    L.rb = tile_reg_bits((int)m, dtype == QVMHIP_F64, fma);
    L.tb = L.m - L.rb;
    for (int i = 0; i < L.m; ++i) L.l2s[i] = L.s2l[i] = i;
    // FMA passes do not keep gate-by-gate rounding: commuting ops are
    // regrouped into layers so that ZZ phases of one angle become one op
    std::vector<qvmhip_tile_op> layered;
    if (fma) {
        // the layering compares every pair of ops: passes longer than 4096
        // ops keep their order (and still merge the runs they hold)
        if (nin <= 4096) layered = layer_order(in_ops, nin);
        if (nin > 4096 || !has_cut_run(layered)) layered.assign(in_ops, in_ops + nin);  // nothing to merge
    }
    const qvmhip_tile_op *in = fma ? layered.data() : in_ops;
    out.clear();
    out.reserve(nin + nin / 2 + 2);
    std::vector<uint32_t> need(nin);
    for (uint32_t i = 0; i < nin; ++i) need[i] = reg_need(in[i]);
    // next_use[i][l]: first op index >= i that needs local bit l on a register
    std::vector<std::array<uint32_t, 16>> next_use(nin + 1);
    next_use[nin].fill(UINT32_MAX);
    for (int i = (int)nin - 1; i >= 0; --i) {
        next_use[i] = next_use[i + 1];
        for (int l = 0; l < L.m; ++l)
            if ((need[i] >> l) & 1u) next_use[i][l] = (uint32_t)i;
    }
    auto reg_local_mask = [&]() {
        uint32_t msk = 0;
        for (int b = 0; b < L.rb; ++b) msk |= 1u << L.s2l[L.tb + b];
        return msk;
    };
    for (uint32_t i = 0; i < nin; ++i) {
        const qvmhip_tile_op &op = in[i];
        if (fma) {
            ZZEdge e0;
            if (zz_edge(op, e0)) {
                // the run of ZZ phases of this angle that starts here
                std::vector<ZZEdge> run{e0};
                uint32_t k = i + 1;
                ZZEdge e;
                while (k < nin && (int)run.size() < kCutMaxEdges && zz_edge(in[k], e) && e.a == e0.a &&
                       e.b == e0.b) {
                    run.push_back(e);
                    ++k;
                }
                if (run.size() >= 2) {
                    cut_phase_op(L, run, out);
                    i = k - 1;
                    continue;
                }
            }
        }
        if (op.kind == QVMHIP_TILE_SWAP && op.ctrl_mask == 0) {
            L.swap_slots(L.l2s[op.q0], L.l2s[op.q1]);  // relabel only
            continue;
        }
        const bool pin2 = op.kind == QVMHIP_TILE_DENSE2 || op.kind == QVMHIP_TILE_SWAP;
        if (need[i] & ~reg_local_mask()) {
            // New register set: this op's targets, then the local bits with the
            // nearest next use (ties keep bits that are already registers).
            std::vector<int> order(L.m);
            for (int l = 0; l < L.m; ++l) order[l] = l;
            const uint32_t cur = reg_local_mask();
            std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
                const uint64_t ka = ((uint64_t)next_use[i][a] << 1) | (((cur >> a) & 1u) ? 0u : 1u);
                const uint64_t kb = ((uint64_t)next_use[i][b] << 1) | (((cur >> b) & 1u) ? 0u : 1u);
                return ka < kb;
            });
            uint32_t nset = 0;
            for (int k = 0; k < L.rb; ++k) nset |= 1u << order[k];
            int ns2l[16];
            for (int j = 0; j < L.m; ++j) ns2l[j] = L.s2l[j];
            // register bits: keep residents in place, then fill freed positions
            bool taken[16] = {false};
            int placed_l[16];
            for (int l = 0; l < 16; ++l) placed_l[l] = -1;
            if (pin2) {
                ns2l[L.tb + 0] = (int)op.q0;
                ns2l[L.tb + 1] = (int)op.q1;
                taken[0] = taken[1] = true;
                placed_l[op.q0] = L.tb + 0;
                placed_l[op.q1] = L.tb + 1;
            }
            for (int b = 0; b < L.rb; ++b) {
                const int l = L.s2l[L.tb + b];
                if (((nset >> l) & 1u) && placed_l[l] < 0 && !taken[b]) {
                    ns2l[L.tb + b] = l;
                    taken[b] = true;
                    placed_l[l] = L.tb + b;
                }
            }
            std::vector<int> entering;
            for (int l = 0; l < L.m; ++l)
                if (((nset >> l) & 1u) && placed_l[l] < 0) entering.push_back(l);
            for (int b = 0, e = 0; b < L.rb; ++b)
                if (!taken[b]) {
                    ns2l[L.tb + b] = entering[e];
                    placed_l[entering[e]] = L.tb + b;
                    taken[b] = true;
                    ++e;
                }
            // thread bits: the slots vacated by entering bits take the evicted
            // bits; pair vacated thread bit p with an evicted bit whose old
            // register position is p when there is one (distinct LDS banks)
            std::vector<int> vacated, evicted;
            for (int p = 0; p < L.tb; ++p)
                if ((nset >> L.s2l[p]) & 1u) vacated.push_back(p);
            for (int b = 0; b < L.rb; ++b) {
                const int l = L.s2l[L.tb + b];
                if (!((nset >> l) & 1u)) evicted.push_back(l);
            }
            std::vector<bool> used(evicted.size(), false);
            for (int p : vacated) {
                int pick = -1;
                for (size_t e = 0; e < evicted.size(); ++e)
                    if (!used[e] && L.l2s[evicted[e]] - L.tb == p) pick = (int)e;
                if (pick < 0)
                    for (size_t e = 0; e < evicted.size() && pick < 0; ++e)
                        if (!used[e]) pick = (int)e;
                used[pick] = true;
                ns2l[p] = evicted[pick];
            }
            out.push_back(remap_op(L, ns2l));
            for (int j = 0; j < L.m; ++j) {
                L.s2l[j] = ns2l[j];
                L.l2s[ns2l[j]] = j;
            }
        } else if (pin2) {
            // both targets are registers; move them to register bits 0 and 1
            for (int want = 0; want < 2; ++want) {
                const int l = want == 0 ? (int)op.q0 : (int)op.q1;
                const int b = L.l2s[l] - L.tb;
                if (b != want) {
                    qvmhip_tile_op r;
                    std::memset(&r, 0, sizeof(r));
                    r.kind = kTileRSwap;
                    r.q0 = (uint32_t)std::min(b, want);
                    r.q1 = (uint32_t)std::max(b, want);
                    out.push_back(r);
                    L.swap_slots(L.tb + b, L.tb + want);
                }
            }
        }
        qvmhip_tile_op o = op;
        o.ctrl_mask = L.slot_mask(op.ctrl_mask);
        o.q0 = (uint32_t)L.l2s[op.q0];
        const bool two = op.kind != QVMHIP_TILE_DENSE1 && op.kind != QVMHIP_TILE_DIAG1 &&
                         op.kind != QVMHIP_TILE_GDIAG;
        if (op.kind != QVMHIP_TILE_GDIAG) o.q1 = two ? (uint32_t)L.l2s[op.q1] : 0u;  // GDIAG: outside qubits
        if (op.kind == QVMHIP_TILE_CPERM) {  // X on the target where the control is 1
            o.kind = kTileXReg;
            o.ctrl_mask |= 1u << L.l2s[op.q1];
            o.q1 = 0;
        }
        if (o.kind == QVMHIP_TILE_DENSE1 && o.ctrl_mask == 0) to_split_dense1(o);
        if (to_register_diagonal(o, L.tb, L.rb)) {
            // consecutive register diagonals multiply into one when the
            // pass contracts with FMAs (no promise of gate-by-gate rounding)
            if (fma && !out.empty() && out.back().kind == kTileRDiag) {
                qvmhip_tile_op &prev = out.back();
                for (int r = 0; r < (1 << L.rb); ++r) {
                    const double ar = prev.m[2 * r], ai = prev.m[2 * r + 1];
                    const double br = o.m[2 * r], bi = o.m[2 * r + 1];
                    prev.m[2 * r] = ar * br - ai * bi;
                    prev.m[2 * r + 1] = ar * bi + ai * br;
                }
                continue;
            }
        }
        out.push_back(o);
    }
    if (!L.identity()) {
        int ns2l[16];
        for (int j = 0; j < L.m; ++j) ns2l[j] = j;
        out.push_back(remap_op(L, ns2l));
    }
    if (dtype == QVMHIP_F32) {
        for (qvmhip_tile_op &o : out) {
            if (o.kind == kTileRemap || o.kind == kTileRSwap || o.kind == kTileXReg || o.kind == kTileCutPhase)
                continue;
            float f[32];
            for (int i = 0; i < 32; ++i) f[i] = (float)o.m[i];
            std::memset(o.m, 0, sizeof(o.m));
            std::memcpy(o.m, f, sizeof(f));
        }
    }
}

// Packs a scheduled program into the slots the kernels run.
static void pack_tile_ops(int dtype, bool fma, uint32_t m, const std::vector<qvmhip_tile_op> &sched,
                          std::vector<TileDevOp> &out) {
    const bool f64 = dtype == QVMHIP_F64;
    const size_t ts = f64 ? 8 : 4;
    const uint32_t rb = (uint32_t)tile_reg_bits((int)m, f64, fma), tb = m - rb, R = 1u << rb;
    const uint32_t lanes = (1u << tb) - 1u, all = (1u << R) - 1u;
    // registers whose bits under rmask equal rwant
    auto regs_with = [&](uint32_t rmask, uint32_t rwant) {
        uint32_t o = 0;
        for (uint32_t r = 0; r < R; ++r)
            if ((r & rmask) == rwant) o |= 1u << r;
        return o;
    };
    // operand i of a scheduled op (already floats for FP32 passes)
    auto val = [&](const qvmhip_tile_op &o, int i) -> double {
        return f64 ? o.m[i] : (double)reinterpret_cast<const float *>(o.m)[i];
    };
    auto emit = [&](uint32_t f, uint32_t a, uint32_t b, uint32_t c, const void *data, size_t bytes) {
        const size_t slots = bytes <= 64 ? 1 : 1 + (bytes - 64 + sizeof(TileDevOp) - 1) / sizeof(TileDevOp);
        const size_t at = out.size();
        out.resize(at + slots);
        std::memset(&out[at], 0, slots * sizeof(TileDevOp));
        out[at].f = f | (uint32_t)((slots - 1) << 28);
        out[at].a = a;
        out[at].b = b;
        out[at].c = c;
        if (bytes) std::memcpy(out[at].m, data, bytes);
    };
    auto emit_vals = [&](uint32_t f, uint32_t a, uint32_t b, uint32_t c, const double *v, size_t count) {
        if (f64) return emit(f, a, b, c, v, count * 8);
        std::vector<float> w(v, v + count);
        emit(f, a, b, c, w.data(), count * 4);
    };
    out.clear();
    for (size_t i = 0; i < sched.size(); ++i) {
        const qvmhip_tile_op &o = sched[i];
        const uint32_t ln = o.ctrl_mask & lanes, rn = o.ctrl_mask >> tb;
        const uint32_t bit = o.q0 >= tb && o.q0 < m ? kF_Bit0 << (o.q0 - tb) : 0u;
        switch (o.kind) {
            case QVMHIP_TILE_DENSE1:
                emit((o.ctrl_mask ? kF_GenC : kF_Gen) | bit, ln, ln, regs_with(rn, rn), o.m, 8 * ts);
                break;
            case kTileD1Real: emit(kF_Real | bit, 0, 0, 0, o.m, 4 * ts); break;
            case kTileD1RX: emit(kF_RX | bit, 0, 0, 0, o.m, 4 * ts); break;
            case kTileXReg: emit(kF_X | bit, ln, ln, regs_with(rn, rn), nullptr, 0); break;
            case kTileRDiag: emit(kF_RDiag, 0, 0, 0, o.m, 2 * R * ts); break;
            case kTileRemap: emit(kF_Remap, 0, 0, 0, o.m, 16); break;
            case QVMHIP_TILE_DENSE2:
                emit(o.ctrl_mask ? kF_Dense2C : kF_Dense2, ln, ln, regs_with(rn, rn), o.m, 32 * ts);
                break;
            case QVMHIP_TILE_SWAP: emit(kF_SwapC, ln, ln, regs_with(rn, rn), nullptr, 0); break;
            case kTileRSwap: {
                static const uint32_t pairs[6][2] = {{0, 1}, {0, 2}, {0, 3}, {1, 2}, {1, 3}, {2, 3}};
                uint32_t c = 0;
                for (uint32_t k = 0; k < 6; ++k)
                    if (pairs[k][0] == o.q0 && pairs[k][1] == o.q1) c = 1u << k;
                emit(kF_RSwap, 0, 0, c, nullptr, 0);
                break;
            }
            case QVMHIP_TILE_GDIAG: {
                const uint32_t ng = o.q1 >> 16, sels = 1u << ng;
                auto one = [&](uint32_t k) { return val(o, 2 * k) == 1.0 && val(o, 2 * k + 1) == 0.0; };
                uint32_t ident = 0;
                bool id0 = true, neg = true, same = true;  // entry 0 is 1, entry 1 is 1 or -1, no use of the local bit
                for (uint32_t k = 0; k < sels; ++k) {
                    if (one(2 * k) && one(2 * k + 1)) ident |= 1u << k;
                    id0 = id0 && one(2 * k);
                    neg = neg && (one(2 * k + 1) || (val(o, 4 * k + 2) == -1.0 && val(o, 4 * k + 3) == 0.0));
                    same = same && val(o, 4 * k) == val(o, 4 * k + 2) && val(o, 4 * k + 1) == val(o, 4 * k + 3);
                }
                const uint32_t where = o.q1 | (ident << 20);
                if (same) {  // no local qubit: one entry for the whole block
                    emit(kF_DL | kF_Out | (neg ? kF_Neg : 0u), 0, where, 0, o.m, 4 * sels * ts);
                } else if (id0) {  // entry 1 where the local bit is set
                    emit(kF_DL | kF_Out | kF_Id0 | (neg ? kF_Neg : 0u) | bit, bit ? 0u : 1u << o.q0, where, 0, o.m,
                         4 * sels * ts);
                } else {
                    emit(kF_Out | (bit ? kF_DR | bit : kF_DL), bit ? 0u : 1u << o.q0, where, 0, o.m, 4 * sels * ts);
                }
                break;
            }
            case kTileCutPhase: {
                const uint8_t *b = (const uint8_t *)o.m;
                const size_t E = b[0], ndata = b[1];
                std::vector<char> d(kCutHeader + (E + 1) * 2 * ts);
                std::memcpy(d.data(), o.m, kCutHeader);
                for (size_t c = 0; c <= E; ++c)
                    std::memcpy(d.data() + kCutHeader + c * 2 * ts,
                                (const char *)sched[i + 1 + c / 16].m + (c % 16) * 2 * ts, 2 * ts);
                emit(kF_Cut, 0, 0, 0, d.data(), d.size());
                i += ndata;
                break;
            }
            default: {  // DIAG1, DIAG2, CPHASE with at least one lane bit among targets and controls
                const bool two = o.kind != QVMHIP_TILE_DIAG1;
                const bool r0 = o.q0 >= tb, r1 = two && o.q1 >= tb;
                if (o.kind != QVMHIP_TILE_CPHASE && o.ctrl_mask == 0) {
                    if (!two) {
                        emit(kF_DL, 1u << o.q0, 1u << o.q0, 0, o.m, 4 * ts);
                        break;
                    }
                    if (!r0 && !r1) {
                        emit(kF_DL4, o.q0 | (o.q1 << 8), 0, 0, o.m, 8 * ts);
                        break;
                    }
                    // one lane bit, one register bit: entries ordered (lane, register)
                    double v[8];
                    for (int l = 0; l < 2; ++l)
                        for (int r = 0; r < 2; ++r) {
                            const int j = r0 ? (r | (l << 1)) : (l | (r << 1));
                            v[4 * l + 2 * r] = val(o, 2 * j);
                            v[4 * l + 2 * r + 1] = val(o, 2 * j + 1);
                        }
                    const uint32_t lp = r0 ? o.q1 : o.q0, rp = (r0 ? o.q0 : o.q1) - tb;
                    emit_vals(kF_DR | (kF_Bit0 << rp), 1u << lp, 1u << lp, 0, v, 8);
                    break;
                }
                // every entry other than 1 multiplies where the target bits
                // spell it and the controls hold
                const uint32_t tmask = (1u << o.q0) | (two ? 1u << o.q1 : 0u);
                const uint32_t entries = o.kind == QVMHIP_TILE_CPHASE ? 1u : two ? 4u : 2u;
                for (uint32_t j = 0; j < entries; ++j) {
                    const uint32_t jj = o.kind == QVMHIP_TILE_CPHASE ? 3u : j;
                    const double v[4] = {1.0, 0.0, val(o, 2 * (int)j), val(o, 2 * (int)j + 1)};
                    if (v[2] == 1.0 && v[3] == 0.0) continue;
                    const uint32_t mask = o.ctrl_mask | tmask;
                    const uint32_t want = o.ctrl_mask | ((jj & 1u) << o.q0) | (two ? ((jj >> 1) & 1u) << o.q1 : 0u);
                    const uint32_t regs = regs_with(mask >> tb, want >> tb);
                    uint32_t f = kF_DL | kF_Id0 | (v[2] == -1.0 && v[3] == 0.0 ? kF_Neg : 0u);
                    if (regs != all) {
                        f |= kF_Mask;
                        for (uint32_t r = 0; r < rb; ++r)
                            if (regs == regs_with(1u << r, 1u << r)) f = (f & ~kF_Mask) | (kF_Bit0 << r);
                    }
                    emit_vals(f, mask & lanes, want & lanes, regs, v, 4);
                }
            }
        }
    }
    emit(kF_End, 0, 0, 0, nullptr, 0);
}

TileCode compile_tile_ops(int dtype, bool fma, uint32_t m, const qvmhip_tile_op *ops, uint32_t nops) {
    std::vector<qvmhip_tile_op> sched;
    schedule_tile_ops(dtype, fma, m, ops, nops, sched);
    std::vector<TileDevOp> packed;
    pack_tile_ops(dtype, fma, m, sched, packed);
    TileCode c;
    c.bytes.assign((const char *)packed.data(), (const char *)(packed.data() + packed.size()));
    for (const qvmhip_tile_op &o : sched) c.cut = c.cut || o.kind == kTileCutPhase;
    return c;
}

namespace {

// Host-side tile arguments of an n-qubit state and tile qubits tq[0..m).
void make_tile_args(uint32_t n, uint32_t m, const uint32_t *tq, int tb, TileArgs &a) {
    std::memset(&a, 0, sizeof(a));
    a.g.nsorted = m;
    for (uint32_t i = 0; i < m; ++i) {
        a.g.sorted[i] = tq[i];
        a.tq[i] = tq[i];
    }
    a.g.ctrl_mask = 0;
    a.g.ngroups = uint64_t(1) << (n - m);
    const int R = 1 << (m - tb);
    for (int r = 0; r < R; ++r) {
        uint64_t o = 0;
        const uint32_t l = (uint32_t)r << tb;
        for (uint32_t b = 0; b < m; ++b)
            if ((l >> b) & 1u) o |= uint64_t(1) << tq[b];
        a.roff[r] = o;
    }
}

template <typename T, int M, bool FMA, bool CUT>
int run_tile(qvmhip_state *s, const uint32_t *tq, uint32_t m, const TileDevOp *ops_dev) {
    constexpr int RB = tile_reg_bits(M, sizeof(T) == 8, FMA);
    constexpr int NT = 1 << (M - RB);
    TileArgs a;
    make_tile_args(s->n, m, tq, M - RB, a);
    prof_begin(s, QVMHIP_K_TILE);
    const uint32_t grid = (uint32_t)std::min<uint64_t>(a.g.ngroups, kMaxGrid);
    hipLaunchKernelGGL((k_tile<T, M, RB, FMA, CUT>), dim3(grid), dim3(NT), 0, s->stream, (vec2_t<T> *)s->amps, a,
                       ops_dev);
    prof_end(s);
    QH_LAUNCH_CHECK();
    return QVMHIP_OK;
}

template <typename T, int M>
int run_tile_f(qvmhip_state *s, const uint32_t *tq, uint32_t m, const TileDevOp *ops_dev, bool cut) {
    if (!(s->flags & QVMHIP_FLAG_FMA_TILES)) return run_tile<T, M, false, false>(s, tq, m, ops_dev);
    return cut ? run_tile<T, M, true, true>(s, tq, m, ops_dev) : run_tile<T, M, true, false>(s, tq, m, ops_dev);
}

template <typename T>
int run_tile_m(qvmhip_state *s, uint32_t m, const uint32_t *tq, const TileDevOp *ops_dev, bool cut) {
    switch (m) {
        case 8: return run_tile_f<T, 8>(s, tq, m, ops_dev, cut);
        case 9: return run_tile_f<T, 9>(s, tq, m, ops_dev, cut);
        case 10: return run_tile_f<T, 10>(s, tq, m, ops_dev, cut);
        case 11: return run_tile_f<T, 11>(s, tq, m, ops_dev, cut);
        case 12: return run_tile_f<T, 12>(s, tq, m, ops_dev, cut);
        case 13:
            if constexpr (sizeof(T) == 4) return run_tile_f<T, 13>(s, tq, m, ops_dev, cut);
            break;
    }
    return fail(QVMHIP_EINVAL, "tile size m must be 8..12 (F64) or 8..13 (F32)");
}

}  // namespace

int launch_tile_code(qvmhip_state *s, uint32_t m, const uint32_t *tile_qubits, const void *code_dev, bool cut) {
    const TileDevOp *dev = (const TileDevOp *)code_dev;
    return s->dtype == QVMHIP_F64 ? run_tile_m<double>(s, m, tile_qubits, dev, cut)
                                  : run_tile_m<float>(s, m, tile_qubits, dev, cut);
}

// A short op list travels to the state's operand slot in the arguments of
// small launches, which are copied when they are enqueued.
struct OpChunk {
    uint4 w[192];
};
__global__ __launch_bounds__(192) void k_put_ops(uint4 *__restrict__ dst, const OpChunk c, uint32_t n) {
    if (threadIdx.x < n) dst[threadIdx.x] = c.w[threadIdx.x];
}

int launch_tile_pass(qvmhip_state *s, uint32_t m, const uint32_t *tile_qubits, uint32_t nops,
                     const qvmhip_tile_op *ops) {
    const TileCode code = compile_tile_ops(s->dtype, (s->flags & QVMHIP_FLAG_FMA_TILES) != 0, m, ops, nops);
    // Operands go through the matrix slot's first half (64 KiB, some 800
    // ops), ordered on the stream after every earlier reader: up to two chunks
    // (6 KiB, some 75 ops) by launches, which cost 3 us each where a copy costs
    // 10; longer lists get a temporary buffer released after the stream drains.
    const size_t bytes = code.bytes.size();
    if (bytes <= 2 * sizeof(OpChunk)) {
        for (size_t off = 0; off < bytes; off += sizeof(OpChunk)) {
            const size_t n = std::min(sizeof(OpChunk), bytes - off);  // slots: a multiple of 16 bytes
            OpChunk c;
            std::memcpy(&c, code.bytes.data() + off, n);
            hipLaunchKernelGGL(k_put_ops, dim3(1), dim3(192), 0, s->stream, (uint4 *)((char *)s->mat + off), c,
                               (uint32_t)(n / 16));
            QH_LAUNCH_CHECK();
        }
        return launch_tile_code(s, m, tile_qubits, s->mat, code.cut);
    }
    void *dev = s->mat, *tmp = nullptr;
    if (bytes > kFusedMatOffset) {
        QH_CHECK(hipMalloc(&tmp, bytes));
        dev = tmp;
    }
    int rc = upload_operand(s, dev, code.bytes.data(), bytes);
    if (!rc) rc = launch_tile_code(s, m, tile_qubits, dev, code.cut);
    if (tmp) {
        (void)hipStreamSynchronize(s->stream);
        (void)hipFree(tmp);
    }
    return rc;
}

size_t tile_entry_bytes() { return sizeof(TileEntry); }

uint64_t build_tile_entry(void *entry, int dtype, bool fma, uint32_t n, uint32_t m, const uint32_t *tq,
                          uint64_t amp_offset, uint64_t block_start, uint64_t op_off, uint32_t tiles_per_block,
                          bool from_zero, uint64_t zero_mask) {
    TileEntry e;
    std::memset(&e, 0, sizeof(e));
    make_tile_args(n, m, tq, (int)m - tile_reg_bits((int)m, dtype == QVMHIP_F64, fma), e.args);
    e.amp_offset = amp_offset;
    e.block_start = block_start;
    e.op_off = op_off;
    e.from_zero = from_zero ? 1u : 0u;
    e.zero_mask = zero_mask;
    std::memcpy(entry, &e, sizeof(e));
    return (e.args.g.ngroups + tiles_per_block - 1) / tiles_per_block;
}

namespace {
template <typename T, int M, bool FMA, bool CUT>
void tile_batch_go(hipStream_t st, void *base, const void *ent, const uint32_t *blk_ent, uint64_t total,
                   uint32_t tpb, const void *op_buf, bool zero) {
    constexpr int RB = tile_reg_bits(M, sizeof(T) == 8, FMA);
    constexpr int NT = 1 << (M - RB);
    const uint32_t grid = (uint32_t)std::min<uint64_t>(total, kMaxGrid);
    if (zero)
        hipLaunchKernelGGL((k_tile_batch<T, M, RB, FMA, CUT, true>), dim3(grid), dim3(NT), 0, st, (vec2_t<T> *)base,
                           (const TileEntry *)ent, blk_ent, total, tpb, (const char *)op_buf);
    else
        hipLaunchKernelGGL((k_tile_batch<T, M, RB, FMA, CUT, false>), dim3(grid), dim3(NT), 0, st,
                           (vec2_t<T> *)base, (const TileEntry *)ent, blk_ent, total, tpb, (const char *)op_buf);
}
template <typename T, bool FMA, bool CUT>
int tile_batch_m(hipStream_t st, uint32_t m, void *base, const void *ent, const uint32_t *blk_ent, uint64_t total,
                 uint32_t tpb, const void *op_buf, bool zero) {
    switch (m) {
        case 8: tile_batch_go<T, 8, FMA, CUT>(st, base, ent, blk_ent, total, tpb, op_buf, zero); break;
        case 9: tile_batch_go<T, 9, FMA, CUT>(st, base, ent, blk_ent, total, tpb, op_buf, zero); break;
        case 10: tile_batch_go<T, 10, FMA, CUT>(st, base, ent, blk_ent, total, tpb, op_buf, zero); break;
        case 11: tile_batch_go<T, 11, FMA, CUT>(st, base, ent, blk_ent, total, tpb, op_buf, zero); break;
        case 12: tile_batch_go<T, 12, FMA, CUT>(st, base, ent, blk_ent, total, tpb, op_buf, zero); break;
        case 13:
            if constexpr (sizeof(T) == 4) {
                tile_batch_go<T, 13, FMA, CUT>(st, base, ent, blk_ent, total, tpb, op_buf, zero);
                break;
            }
            return fail(QVMHIP_EINVAL, "tile size 13 is FP32 only");
        default:
            return fail(QVMHIP_EINVAL, "tile size m must be 8..13");
    }
    QH_LAUNCH_CHECK();
    return QVMHIP_OK;
}
}  // namespace

int launch_tile_batch(hipStream_t st, int dtype, bool fma, bool cut, bool zero, uint32_t m, void *base,
                      const void *entries_dev, const uint32_t *blk_ent_dev, uint64_t total_blocks,
                      uint32_t tiles_per_block, const void *op_buf) {
    const bool f64 = dtype == QVMHIP_F64;
#define QH_TB(TT, F, C) \
    tile_batch_m<TT, F, C>(st, m, base, entries_dev, blk_ent_dev, total_blocks, tiles_per_block, op_buf, zero)
    if (!fma) return f64 ? QH_TB(double, false, false) : QH_TB(float, false, false);
    if (!cut) return f64 ? QH_TB(double, true, false) : QH_TB(float, true, false);
    return f64 ? QH_TB(double, true, true) : QH_TB(float, true, true);
#undef QH_TB
}

}  // namespace qvmhip
