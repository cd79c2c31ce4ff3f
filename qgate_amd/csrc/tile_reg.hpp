// Register-resident tile passes: device code shared by the single-circuit passes (k_tile.hip)
// and the batched ones (k_batch.hip). Their planning is in reg_plan.hpp.
//
// A pass keeps its tile in registers: each of the T threads holds A = 2^M / T amplitudes of
// each state (one state going forward, phi and lambda in the adjoint sweep). It is split into
// phases; in each phase log2(A) tile bits are register bits (the targets of the phase's
// non-diagonal gates), 6 are lane bits and the rest wave bits, so the phase's pair updates are
// register to register, with no LDS traffic and no barrier. Between phases the tile goes
// through LDS once.
//
// What bounds a pass is instruction issue, so the ops are built to be few and short:
//   * Rotations are applied without their common factor: [[c, -s], [s, c]] is
//     c [[1, -t], [t, 1]] with t = s / c, or s [[k, -1], [1, k]] with k = c / s where that is
//     smaller, one FMA a component instead of a multiply and an FMA. The factors of a phase
//     multiply into one number that is applied at the end of the phase. Uncontrolled general
//     gates arrive split into diagonals and such a rotation (reg_plan.hpp).
//   * Register updates are in-place asm statements with tied operands. Written as expressions,
//     every dispatch arm produced new values and the compiler moved the whole register array at
//     the joins (32 to 64 moves a gate in the sweep, whose rotations take 48).
//   * Diagonal gates on no register bit multiply into one factor per thread, applied at the end
//     of the phase; signs (CZ, Z) into one sign.
//   * Gradient terms are summed over the wavefront by FP64 matrix-core steps, sixteen slots to
//     an accumulator tile: a conversion, two moves and one matrix instruction a term, where a
//     DPP tree took about 20 vector instructions.
//   * A diagonal gate is its first entry, which without controls is a phase of the whole state (one
//     factor per pass, none where only <H> and gradients are wanted), and a ratio.
// Against passes without these steps, the backward sweep of the 24-qubit, 12-layer ansatz takes 15
// passes of 265 us instead of 19 of 353, its forward part 15 of 105 us instead of 22 of 129, and 500
// random gates on 30 qubits 19 of 4.4 ms instead of 20 of 5.8. Vector and scalar issue bound all of
// them: a gate costs about 45 scalar instructions to decode and dispatch beside its arithmetic.
#pragma once

#include <algorithm>
#include <complex>
#include <cstring>
#include <type_traits>
#include <vector>

#include "gate_matrix.hpp"
#include "kernels.hpp"
#include "qg_runtime.hpp"
#include "reg_plan.hpp"
#include "tile_common.hpp"

namespace qg {

namespace {

// Low: the lowest bits that every tile holds, one 128-byte cache line. Each bit less frees one for a
// gate's target: with 256-byte rows the 24-qubit ansatz took 19 sweep and 16 forward passes instead of
// 15 and 15 (sweep 4.36 -> 4.08 ms, forward 1.63 -> 1.59), 500 gates on 30 qubits 22 instead of 19
// (86.2 -> 83.4 ms; with 64-byte rows 110).
template <class R>
struct TileCfg;
template <>
struct TileCfg<float> {
    static constexpr int MaxBits = 12;   // 2^12 x 8 B = 32 KiB of LDS
    static constexpr int MaxOps = 40;    // LDS passes
    static constexpr int MaxRegOps = 72; // register passes: 40 B each in the kernel arguments
    static constexpr int Low = 4;        // 16 contiguous amplitudes = 128 B per row
};
template <>
struct TileCfg<double> {
    static constexpr int MaxBits = 11;   // 2^11 x 16 B = 32 KiB
    static constexpr int MaxOps = 24;
    static constexpr int MaxRegOps = 52; // 56 B each
    static constexpr int Low = 3;        // 8 x 16 B = 128 B per row
};

constexpr int kMaxPhases = 24;

// Bit layout of one register phase, packed in dwords so that a phase read at a runtime
// index takes scalar loads (a byte array read at a runtime index would be a vector load,
// whose wait also waits for HBM traffic in flight). Byte k of `bits` is the local bit of
// register bit k (k < 5), of lane bit k - 5 (5 <= k < 11) or of wave bit k - 11 (k < 16).
struct PhaseBits {
    unsigned bits[4];
    int op_begin, n_ops;   // ops of the pass
    __host__ __device__ int byte(int k) const { return (int)((bits[k >> 2] >> ((k & 3) * 8)) & 0xffu); }
    __host__ __device__ int rb(int k) const { return byte(k); }
    __host__ __device__ int lb(int k) const { return byte(5 + k); }
    __host__ __device__ int wb(int k) const { return byte(11 + k); }
    void set(int k, int v) {
        const int sh = (k & 3) * 8;
        bits[k >> 2] = (bits[k >> 2] & ~(0xffu << sh)) | ((unsigned)v << sh);
    }
};

// Arms of an op. Families of updates on a register position P take codes 4 F + P: rotations
// about Y and X in their two forms (t, k), controlled swaps, general 2x2, a factor or a sign on
// the register indices with bit P set, and a Z rotation on bit P with its gradient term (the term,
// then the factor on the indices with the bit set).
// kArmPair2 + i: a factor on the register indices with both bits of the i-th pair set
// (01, 02, 12, 03, 13, 23), kArmSign2 + i a sign; kArmFactorAny: on those with every bit of creg
// set; kArmZAny: the Z term with controls on register bits. The rest leave the registers alone.
enum : int {
    kFamY = 0, kFamYk = 1, kFamX = 2, kFamXk = 3, kFamSwap = 4, kFamAny = 5, kFamFactor = 6, kFamSign = 7, kFamZ = 8,
    kArmPair2 = 36, kArmSign2 = 42, kArmFactorAny = 48, kArmZAny = 49,
    kArmThread = 50,       // a Z rotation on a lane or wave bit with its gradient term
    kArmThreadCtrl = 51,   // the same with controls on lane and wave bits
    kArmOuter = 52,        // the same on a bit outside the tile, controls allowed
    kArmPhase = 53,        // a factor where every control on lane and wave bits is set
    kArmSign = 54,         // a sign where they are
    kArmU = 55,            // the thread's sum that the Z terms on bits that are no register bits share
    kArmFlush = 56,        // 16 gradient slots are complete
    kArmNone = 57,         // the second half of a general 2x2
    kArmParity = 58        // a factor where two bits differ, with the gradient term of their ZZ
};

// One op of a register pass. code: arm | target << 8 | creg << 16 | generator << 24 | first
// coefficient << 28. Controls are split by where their bits live: outside the tile (gctrl, one
// test per tile), on lane and wave bits (cthr, one test per thread), on register bits (creg).
template <class R>
struct alignas(8) RegOp {
    unsigned code, cthr;
    u64 gctrl;
    int slot;          // gradient slot, -1: none
    int row;           // batched passes: row of the coefficient table
    R c[4];            // else the coefficients (a general 2x2 takes the next op's as well)
};

// An op read whole, as two or three scalar loads: field by field it took five, each with its own
// address.
template <class R>
struct OpWords {
    typedef unsigned u32x8 __attribute__((ext_vector_type(8), aligned(8)));
    typedef unsigned u32x2 __attribute__((ext_vector_type(2), aligned(8)));
    typedef unsigned u32x4 __attribute__((ext_vector_type(4), aligned(8)));
    u32x8 a;
    u32x4 b;
    u32x2 c;
    __device__ __forceinline__ void load(const RegOp<R> *p) {
        const unsigned *w = reinterpret_cast<const unsigned *>(p);
        a = *reinterpret_cast<const u32x8 *>(w);
        if constexpr (sizeof(R) == 8) {
            b = *reinterpret_cast<const u32x4 *>(w + 8);
            c = *reinterpret_cast<const u32x2 *>(w + 12);
        } else {
            c = *reinterpret_cast<const u32x2 *>(w + 8);
        }
    }
    // waits for the words: scalar loads return out of order, so a wait for these after the next
    // op's have been issued would wait for both
    __device__ __forceinline__ void arrive() {
        if constexpr (sizeof(R) == 8)
            asm volatile("; op" : "+s"(a), "+s"(b), "+s"(c));
        else
            asm volatile("; op" : "+s"(a), "+s"(c));
    }
    __device__ __forceinline__ unsigned code() const { return a[0]; }
    __device__ __forceinline__ unsigned cthr() const { return a[1]; }
    __device__ __forceinline__ u64 gctrl() const { return (u64)a[3] << 32 | a[2]; }
    __device__ __forceinline__ int slot() const { return (int)a[4]; }
    __device__ __forceinline__ int row() const { return (int)a[5]; }
    __device__ __forceinline__ R coef(int i) const {
        if constexpr (sizeof(R) == 8) {
            const unsigned lo = i == 0 ? a[6] : i == 1 ? b[0] : i == 2 ? b[2] : c[0];
            const unsigned hi = i == 0 ? a[7] : i == 1 ? b[1] : i == 2 ? b[3] : c[1];
            return __longlong_as_double((long long)((u64)hi << 32 | lo));
        } else {
            return __uint_as_float(i == 0 ? a[6] : i == 1 ? a[7] : i == 2 ? c[0] : c[1]);
        }
    }
};
static_assert(sizeof(RegOp<float>) == 40 && sizeof(RegOp<double>) == 56, "op words");

// Coefficients of a gate, by kind (a row of a batched pass's table):
//   rotation   t or k, 1 if it is k, and the factor left out, in FP64 for complex64 (two
//              entries), as an unevaluated sum of two numbers for complex128
//   diagonal   m00, m11, m11 / m00 (complex)
//   general    m00, m01, m10, m11 (complex)
// The factor is that of the rounded t (or k), which makes good what rounding t does to the norm
// of the state, and the factors of a phase are multiplied in twice the precision of the state
// and rounded once. The rounded matrices of the two-multiply form each shift the norm of the
// whole state; after 530 gates on 30 qubits in complex64 a joint distribution was off by 2.1e-6
// (2-norm), now 0.57e-6.
constexpr int kCoefs = 8;

template <class R>
__host__ __device__ inline void rotation_coefs(R *c, double co, double si) {
    const bool k = (si < 0. ? -si : si) > (co < 0. ? -co : co);
    c[0] = (R)(k ? co / si : si / co);
    c[1] = k ? R(1) : R(0);
    // f (1 + r / 2) = 1 / sqrt(1 + t^2), r the rest of one Newton step in FMAs
    const double t = (double)c[0], t2 = t * t, q = 1. + t2, qe = ((1. - q) + t2) + __builtin_fma(t, t, -t2);
    double f = 1. / sqrt(q);
    const double f2 = f * f, p = f2 * q;
    const double r = ((1. - p) - __builtin_fma(f2, q, -p)) - __builtin_fma(__builtin_fma(f, f, -f2), q, f2 * qe);
    // a matrix that is no rotation but a multiple of one
    const double mag2 = co * co + si * si;
    if (mag2 < 1. - 1e-13 || mag2 > 1. + 1e-13) f *= sqrt(mag2);
    if ((k ? si : co) < 0.) f = -f;
    if constexpr (sizeof(R) == 8) {
        c[2] = f;
        c[3] = 0.5 * f * r;
    } else {
        __builtin_memcpy(c + 2, &f, sizeof(double));
    }
}

// The factors of a phase's rotations (uniform): hi + lo for complex128, hi for complex64.
template <class R>
struct Scale {
    double hi, lo;
    // 1 + carry: what the rounding of the last phase's factor left out
    __device__ __forceinline__ void init(double carry) {
        hi = sizeof(R) == 8 ? 1. : 1. + carry;
        lo = sizeof(R) == 8 ? carry : 0.;
    }
    __device__ __forceinline__ void times(R c2, R c3) {
        if constexpr (sizeof(R) == 8) {
            const double p = hi * c2;
            lo = __builtin_fma(lo, c2, __builtin_fma(hi, c3, __builtin_fma(hi, c2, -p)));
            hi = p;
        } else {
            hi *= __longlong_as_double((long long)(((u64)__float_as_uint(c3) << 32) | __float_as_uint(c2)));
        }
    }
    __device__ __forceinline__ double value() const { return sizeof(R) == 8 ? hi + lo : hi; }
};

template <int A>
struct Log2 {
    static constexpr int v = A <= 1 ? 0 : 1 + Log2<A / 2>::v;
};
template <>
struct Log2<1> {
    static constexpr int v = 0;
};

// f(std::integral_constant<int, J>) for J = B .. E-1: register arrays are only ever indexed
// with compile-time constants, so they stay in registers.
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>());
        static_for<B + 1, E>(f);
    }
}

template <class R>
__device__ __forceinline__ R fma_r(R a, R b, R c) {
    if constexpr (sizeof(R) == 4)
        return __builtin_fmaf(a, b, c);
    else
        return __builtin_fma(a, b, c);
}

// acc + Im(conj(a) b), as two FMAs into the accumulator
template <class R>
__device__ __forceinline__ R add_im_conj_mul(R acc, const Cx<R> &a, const Cx<R> &b) {
    return fma_r(-a.im, b.re, fma_r(a.re, b.im, acc));
}

// acc + the gradient term of a pair (p0, p1) / (l0, l1) for generator G (1 X, 2 Y):
// Im<l|G|p> over the pair, four FMAs into the accumulator
template <class R, int G>
__device__ __forceinline__ R add_pair_term(R acc, const Cx<R> &p0, const Cx<R> &p1, const Cx<R> &l0,
                                           const Cx<R> &l1) {
    if constexpr (G == 1) return add_im_conj_mul(add_im_conj_mul(acc, l0, p1), l1, p0);
    acc = fma_r(l1.re, p0.re, acc);
    acc = fma_r(l1.im, p0.im, acc);
    acc = fma_r(-l0.re, p1.re, acc);
    return fma_r(-l0.im, p1.im, acc);
}

// c ? a : b, component by component: a select of whole structs can be lowered to a select
// of their addresses, which would keep register arrays out of registers.
template <class R>
__device__ __forceinline__ Cx<R> csel(bool c, const Cx<R> &a, const Cx<R> &b) {
    return cx<R>(c ? a.re : b.re, c ? a.im : b.im);
}

// ---- in-place register updates ---------------------------------------------------------------
//
// C is a code of its own per dispatch arm, in the statement as a comment, so that the optimiser
// merges no two arms into one block that would pick register elements through pointers. The
// statements hold vector instructions only, read and write no memory, and leave every output
// written; the matrix-core and cross-lane instructions around them, whose operands need wait
// states after a vector write, take compiler-made values.

// Rotations: (x, y) <- (x + t y, y - t x) for form t, (y + k x, k y - x) for form k. One statement
// takes both components of a register pair, of every state: the compiler puts an idle
// instruction between statements that write vector registers.

template <int C>
__device__ __forceinline__ void rot_t(float &x0, float &y0, float &x1, float &y1, float c) {
    float w, z;
    asm(
        "v_fma_f32 %4, %6, %1, %0\n\t"
        "v_fma_f32 %5, %6, %3, %2\n\t"
        "v_fma_f32 %1, -%6, %0, %1\n\t"
        "v_fma_f32 %3, -%6, %2, %3\n\t"
        "v_mov_b32 %0, %4\n\t"
        "v_mov_b32 %2, %5\n\t"
        "; arm %7"
        : "+v"(x0), "+v"(y0), "+v"(x1), "+v"(y1), "=&v"(w), "=&v"(z)
        : "s"(c), "n"(C));
}

template <int C>
__device__ __forceinline__ void rot_t(float &x0, float &y0, float &x1, float &y1, float &x2, float &y2, float &x3, float &y3, float c) {
    float w, z;
    asm(
        "v_fma_f32 %8, %10, %1, %0\n\t"
        "v_fma_f32 %9, %10, %3, %2\n\t"
        "v_fma_f32 %1, -%10, %0, %1\n\t"
        "v_fma_f32 %3, -%10, %2, %3\n\t"
        "v_mov_b32 %0, %8\n\t"
        "v_mov_b32 %2, %9\n\t"
        "v_fma_f32 %8, %10, %5, %4\n\t"
        "v_fma_f32 %9, %10, %7, %6\n\t"
        "v_fma_f32 %5, -%10, %4, %5\n\t"
        "v_fma_f32 %7, -%10, %6, %7\n\t"
        "v_mov_b32 %4, %8\n\t"
        "v_mov_b32 %6, %9\n\t"
        "; arm %11"
        : "+v"(x0), "+v"(y0), "+v"(x1), "+v"(y1), "+v"(x2), "+v"(y2), "+v"(x3), "+v"(y3), "=&v"(w), "=&v"(z)
        : "s"(c), "n"(C));
}

template <int C>
__device__ __forceinline__ void rot_k(float &x0, float &y0, float &x1, float &y1, float c) {
    float w, z;
    asm(
        "v_fma_f32 %4, %6, %0, %1\n\t"
        "v_fma_f32 %5, %6, %2, %3\n\t"
        "v_fma_f32 %1, %6, %1, -%0\n\t"
        "v_fma_f32 %3, %6, %3, -%2\n\t"
        "v_mov_b32 %0, %4\n\t"
        "v_mov_b32 %2, %5\n\t"
        "; arm %7"
        : "+v"(x0), "+v"(y0), "+v"(x1), "+v"(y1), "=&v"(w), "=&v"(z)
        : "s"(c), "n"(C));
}

template <int C>
__device__ __forceinline__ void rot_k(float &x0, float &y0, float &x1, float &y1, float &x2, float &y2, float &x3, float &y3, float c) {
    float w, z;
    asm(
        "v_fma_f32 %8, %10, %0, %1\n\t"
        "v_fma_f32 %9, %10, %2, %3\n\t"
        "v_fma_f32 %1, %10, %1, -%0\n\t"
        "v_fma_f32 %3, %10, %3, -%2\n\t"
        "v_mov_b32 %0, %8\n\t"
        "v_mov_b32 %2, %9\n\t"
        "v_fma_f32 %8, %10, %4, %5\n\t"
        "v_fma_f32 %9, %10, %6, %7\n\t"
        "v_fma_f32 %5, %10, %5, -%4\n\t"
        "v_fma_f32 %7, %10, %7, -%6\n\t"
        "v_mov_b32 %4, %8\n\t"
        "v_mov_b32 %6, %9\n\t"
        "; arm %11"
        : "+v"(x0), "+v"(y0), "+v"(x1), "+v"(y1), "+v"(x2), "+v"(y2), "+v"(x3), "+v"(y3), "=&v"(w), "=&v"(z)
        : "s"(c), "n"(C));
}

template <int C>
__device__ __forceinline__ void rot_t(double &x0, double &y0, double &x1, double &y1, double c) {
    double w, z;
    asm(
        "v_fma_f64 %4, %6, %1, %0\n\t"
        "v_fma_f64 %5, %6, %3, %2\n\t"
        "v_fma_f64 %1, -%6, %0, %1\n\t"
        "v_fma_f64 %3, -%6, %2, %3\n\t"
        "v_mov_b64 %0, %4\n\t"
        "v_mov_b64 %2, %5\n\t"
        "; arm %7"
        : "+v"(x0), "+v"(y0), "+v"(x1), "+v"(y1), "=&v"(w), "=&v"(z)
        : "s"(c), "n"(C));
}

template <int C>
__device__ __forceinline__ void rot_t(double &x0, double &y0, double &x1, double &y1, double &x2, double &y2, double &x3, double &y3, double c) {
    double w, z;
    asm(
        "v_fma_f64 %8, %10, %1, %0\n\t"
        "v_fma_f64 %9, %10, %3, %2\n\t"
        "v_fma_f64 %1, -%10, %0, %1\n\t"
        "v_fma_f64 %3, -%10, %2, %3\n\t"
        "v_mov_b64 %0, %8\n\t"
        "v_mov_b64 %2, %9\n\t"
        "v_fma_f64 %8, %10, %5, %4\n\t"
        "v_fma_f64 %9, %10, %7, %6\n\t"
        "v_fma_f64 %5, -%10, %4, %5\n\t"
        "v_fma_f64 %7, -%10, %6, %7\n\t"
        "v_mov_b64 %4, %8\n\t"
        "v_mov_b64 %6, %9\n\t"
        "; arm %11"
        : "+v"(x0), "+v"(y0), "+v"(x1), "+v"(y1), "+v"(x2), "+v"(y2), "+v"(x3), "+v"(y3), "=&v"(w), "=&v"(z)
        : "s"(c), "n"(C));
}

template <int C>
__device__ __forceinline__ void rot_k(double &x0, double &y0, double &x1, double &y1, double c) {
    double w, z;
    asm(
        "v_fma_f64 %4, %6, %0, %1\n\t"
        "v_fma_f64 %5, %6, %2, %3\n\t"
        "v_fma_f64 %1, %6, %1, -%0\n\t"
        "v_fma_f64 %3, %6, %3, -%2\n\t"
        "v_mov_b64 %0, %4\n\t"
        "v_mov_b64 %2, %5\n\t"
        "; arm %7"
        : "+v"(x0), "+v"(y0), "+v"(x1), "+v"(y1), "=&v"(w), "=&v"(z)
        : "s"(c), "n"(C));
}

template <int C>
__device__ __forceinline__ void rot_k(double &x0, double &y0, double &x1, double &y1, double &x2, double &y2, double &x3, double &y3, double c) {
    double w, z;
    asm(
        "v_fma_f64 %8, %10, %0, %1\n\t"
        "v_fma_f64 %9, %10, %2, %3\n\t"
        "v_fma_f64 %1, %10, %1, -%0\n\t"
        "v_fma_f64 %3, %10, %3, -%2\n\t"
        "v_mov_b64 %0, %8\n\t"
        "v_mov_b64 %2, %9\n\t"
        "v_fma_f64 %8, %10, %4, %5\n\t"
        "v_fma_f64 %9, %10, %6, %7\n\t"
        "v_fma_f64 %5, %10, %5, -%4\n\t"
        "v_fma_f64 %7, %10, %7, -%6\n\t"
        "v_mov_b64 %4, %8\n\t"
        "v_mov_b64 %6, %9\n\t"
        "; arm %11"
        : "+v"(x0), "+v"(y0), "+v"(x1), "+v"(y1), "+v"(x2), "+v"(y2), "+v"(x3), "+v"(y3), "=&v"(w), "=&v"(z)
        : "s"(c), "n"(C));
}

// x, y <- m ? y, x : x, y (m: lane mask)
template <int C>
__device__ __forceinline__ void swap_if(Cx<float> &x, Cx<float> &y, u64 m) {
    float w, z;
    asm("v_cndmask_b32 %4, %0, %1, %6\n\tv_cndmask_b32 %5, %2, %3, %6\n\tv_cndmask_b32 %1, %1, %0, %6\n\t"
        "v_cndmask_b32 %3, %3, %2, %6\n\tv_mov_b32 %0, %4\n\tv_mov_b32 %2, %5 ; arm %7"
        : "+v"(x.re), "+v"(y.re), "+v"(x.im), "+v"(y.im), "=&v"(w), "=&v"(z) : "s"(m), "n"(C));
}
template <int C>
__device__ __forceinline__ void swap_if(Cx<double> &x, Cx<double> &y, u64 m) {
    // under a lane mask: a 64-bit value has no select of its own
    double w, z;
    u64 saved;
    asm("s_mov_b64 %6, exec\n\ts_and_b64 exec, exec, %7\n\tv_mov_b64 %4, %0\n\tv_mov_b64 %5, %2\n\t"
        "v_mov_b64 %0, %1\n\tv_mov_b64 %2, %3\n\tv_mov_b64 %1, %4\n\tv_mov_b64 %3, %5\n\ts_mov_b64 exec, %6 ; arm %8"
        : "+v"(x.re), "+v"(y.re), "+v"(x.im), "+v"(y.im), "=&v"(w), "=&v"(z), "=&s"(saved)
        : "s"(m), "n"(C)
        : "scc");
}

// (re, im) <- (re, im) (fr, fi)
template <int C>
__device__ __forceinline__ void mul_by(Cx<float> &v, const Cx<float> &f) {
    float w;
    asm("v_mul_f32 %2, %0, %3\n\tv_fma_f32 %2, -%1, %4, %2\n\tv_mul_f32 %1, %1, %3\n\tv_fma_f32 %1, %0, %4, %1\n\t"
        "v_mov_b32 %0, %2 ; arm %5"
        : "+v"(v.re), "+v"(v.im), "=&v"(w) : "v"(f.re), "v"(f.im), "n"(C));
}
template <int C>
__device__ __forceinline__ void mul_by(Cx<double> &v, const Cx<double> &f) {
    double w;
    asm("v_mul_f64 %2, %0, %3\n\tv_fma_f64 %2, -%1, %4, %2\n\tv_mul_f64 %1, %1, %3\n\tv_fma_f64 %1, %0, %4, %1\n\t"
        "v_mov_b64 %0, %2 ; arm %5"
        : "+v"(v.re), "+v"(v.im), "=&v"(w) : "v"(f.re), "v"(f.im), "n"(C));
}

// v <- v s
template <int C>
__device__ __forceinline__ void scale_by(Cx<float> &v, float s) {
    asm("v_mul_f32 %0, %0, %2\n\tv_mul_f32 %1, %1, %2 ; arm %3" : "+v"(v.re), "+v"(v.im) : "v"(s), "n"(C));
}
template <int C>
__device__ __forceinline__ void scale_by(Cx<double> &v, double s) {
    asm("v_mul_f64 %0, %0, %2\n\tv_mul_f64 %1, %1, %2 ; arm %3" : "+v"(v.re), "+v"(v.im) : "v"(s), "n"(C));
}

// (x0, x1) <- M (x0, x1) where c, in place; general 2x2
template <class R, int C>
__device__ __forceinline__ void mix(Cx<R> &x0, Cx<R> &x1, const R (&m)[8], bool c) {
    const Cx<R> y0 = cx<R>(fma_r(m[0], x0.re, fma_r(-m[1], x0.im, fma_r(m[2], x1.re, -m[3] * x1.im))),
                           fma_r(m[0], x0.im, fma_r(m[1], x0.re, fma_r(m[2], x1.im, m[3] * x1.re))));
    const Cx<R> y1 = cx<R>(fma_r(m[4], x0.re, fma_r(-m[5], x0.im, fma_r(m[6], x1.re, -m[7] * x1.im))),
                           fma_r(m[4], x0.im, fma_r(m[5], x0.re, fma_r(m[6], x1.im, m[7] * x1.re))));
    x0 = csel(c, y0, x0);
    x1 = csel(c, y1, x1);
    asm volatile("; arm %0" ::"n"(C));
}

// Every component in a register of its own: LDS reads and stores take register pairs, and a pair
// that stayed one through the phase could be no operand of the updates above, so that each of
// them copied it out and back. These statements keep the copies at the two ends of the phase.
template <class R>
__device__ __forceinline__ void own_register(R &x) {
    asm("; own register" : "+v"(x));
}

template <class R, int A>
__device__ __forceinline__ void apart(Cx<R> (&v)[A]) {
    static_for<0, A>([&](auto jc) __attribute__((always_inline)) {
        constexpr int j = decltype(jc)::value;
        own_register(v[j].re);
        own_register(v[j].im);
    });
}

// The register bits of the i-th pair of kArmPair2 / kArmSign2.
__host__ __device__ constexpr int pair2_mask(int i) {
    return i == 0 ? 3 : i == 1 ? 5 : i == 2 ? 6 : i == 3 ? 9 : i == 4 ? 10 : 12;
}

// ---- gradient terms --------------------------------------------------------------------------

typedef double f64x4 __attribute__((ext_vector_type(4)));

// Sums over the wavefront of up to 16 consecutive slots: one v_mfma_f64_16x16x4f64 per term
// multiplies the 64 lanes' values, as a 16 x 4 matrix, by a 4 x 16 matrix whose column `slot` is
// their scale, so column slot of the accumulator collects the sums over groups of four lanes; flush
// adds the accumulator's rows, in a fixed order, and leaves them in red[slot].
template <int NW>
struct SlotSums {
    f64x4 acc;
    __device__ __forceinline__ void init() { acc = f64x4{0., 0., 0., 0.}; }
    __device__ __forceinline__ void flush(int group, double (*red)[NW], int n_slots, unsigned lane, unsigned wave) {
        double s = (acc[0] + acc[1]) + (acc[2] + acc[3]);
        s += __shfl_xor(s, 16, 64);
        s += __shfl_xor(s, 32, 64);
        const int slot = group * 16 + (int)lane;
        if (lane < 16 && slot < n_slots) red[slot][wave] = s;
        acc = f64x4{0., 0., 0., 0.};
    }
    __device__ __forceinline__ void add(double v, double scale, int slot, unsigned lane) {
        const double b = (lane & 15u) == (unsigned)(slot & 15) ? scale : 0.;
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(v, b, acc, 0, 0, 0);
    }
};

constexpr int kMaxSweepSlots = 96;

// ---- register ops ----------------------------------------------------------------------------

// The op of code C on the registers. m: coefficients; f: its factor in this thread (1 where its
// controls on lane and wave bits fail, ok); acc receives the gradient term (NS == 2).
template <int C, class R, int A, int NS>
__device__ __forceinline__ void reg_arm(Cx<R> (&v)[NS][A], const R (&m)[8], const Cx<R> &f, int creg, bool ok,
                                        int pauli, int tgt, u64 zsrc, R &acc) {
    constexpr int RB = Log2<A>::v, F = C / 4, P = C % 4;
    constexpr bool subset = F == kFamFactor || F == kFamSign || (C >= kArmPair2 && C < kArmFactorAny);
    constexpr int mask = F == kFamFactor || F == kFamSign ? 1 << P
                         : C >= kArmSign2                 ? pair2_mask(C - kArmSign2)
                                                          : pair2_mask(C - kArmPair2);
    constexpr bool sign = F == kFamSign || (C >= kArmSign2 && C < kArmFactorAny);
    if constexpr (F <= kFamAny) {
        if constexpr (P >= RB) {
            __builtin_unreachable();
        } else {
            const R t = m[0];
            const u64 okm = F == kFamSwap ? __ballot(ok) : 0;
            static_for<0, A>([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                if constexpr (((j >> P) & 1) == 0) {
                    constexpr int j1 = j + (1 << P);
                    const bool c = ok && (j & creg) == creg;
                    if constexpr (NS == 2 && F <= kFamXk)
                        acc = add_pair_term<R, (F <= kFamYk ? 2 : 1)>(acc, v[0][j], v[0][j1], v[NS - 1][j],
                                                                      v[NS - 1][j1]);
                    if constexpr (NS == 2 && F == kFamAny) {
                        R w = R(0);
                        if (pauli == 1) w = add_pair_term<R, 1>(w, v[0][j], v[0][j1], v[NS - 1][j], v[NS - 1][j1]);
                        if (pauli == 2) w = add_pair_term<R, 2>(w, v[0][j], v[0][j1], v[NS - 1][j], v[NS - 1][j1]);
                        acc += c ? w : R(0);
                    }
                    if constexpr (F <= kFamXk) {
                        constexpr bool X = F >= kFamX, K = F == kFamYk || F == kFamXk;
                        Cx<R> &a0 = v[0][j], &a1 = v[0][j1], &b0 = v[NS - 1][j], &b1 = v[NS - 1][j1];
                        if constexpr (NS == 1 && !X && !K) rot_t<C>(a0.re, a1.re, a0.im, a1.im, t);
                        if constexpr (NS == 1 && !X && K) rot_k<C>(a0.re, a1.re, a0.im, a1.im, t);
                        if constexpr (NS == 1 && X && !K) rot_t<C>(a0.re, a1.im, a1.re, a0.im, t);
                        if constexpr (NS == 1 && X && K) rot_k<C>(a0.re, a1.im, a1.re, a0.im, t);
                        if constexpr (NS == 2 && !X && !K)
                            rot_t<C>(a0.re, a1.re, a0.im, a1.im, b0.re, b1.re, b0.im, b1.im, t);
                        if constexpr (NS == 2 && !X && K)
                            rot_k<C>(a0.re, a1.re, a0.im, a1.im, b0.re, b1.re, b0.im, b1.im, t);
                        if constexpr (NS == 2 && X && !K)
                            rot_t<C>(a0.re, a1.im, a1.re, a0.im, b0.re, b1.im, b1.re, b0.im, t);
                        if constexpr (NS == 2 && X && K)
                            rot_k<C>(a0.re, a1.im, a1.re, a0.im, b0.re, b1.im, b1.re, b0.im, t);
                    } else {
#pragma unroll
                        for (int s = 0; s < NS; ++s) {
                            Cx<R> &x0 = v[s][j], &x1 = v[s][j1];
                            if constexpr (F == kFamSwap) {
                                const u64 mk = (j & creg) == creg ? okm : 0;
                                swap_if<C>(x0, x1, mk);
                            } else {
                                mix<R, C>(x0, x1, m, c);
                            }
                        }
                    }
                }
            });
        }
    } else if constexpr (subset) {
        if constexpr (mask >= A) {
            __builtin_unreachable();
        } else {
            const R sg = ok ? R(-1) : R(1);
            static_for<0, A>([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                if constexpr ((j & mask) == mask) {
#pragma unroll
                    for (int s = 0; s < NS; ++s) {
                        if constexpr (sign) {
                            scale_by<C>(v[s][j], sg);
                        } else {
                            mul_by<C>(v[s][j], f);
                        }
                    }
                }
            });
        }
    } else if constexpr (F == kFamZ) {
        if constexpr (NS == 1 || P >= RB) {
            __builtin_unreachable();
        } else {
            static_for<0, A>([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                if constexpr (((j >> P) & 1) == 0)
                    acc = add_im_conj_mul(acc, v[1][j], v[0][j]);
                else
                    acc = add_im_conj_mul(acc, v[0][j], v[1][j]);
            });
            acc = ok ? acc : R(0);
            static_for<0, A>([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                if constexpr (((j >> P) & 1) != 0) {
#pragma unroll
                    for (int s = 0; s < NS; ++s) mul_by<C>(v[s][j], f);
                }
            });
        }
    } else if constexpr (C == kArmFactorAny) {
        static_for<0, A>([&](auto jc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value;
            const Cx<R> fj = csel((j & creg) == creg, f, cx<R>(R(1), R(0)));
#pragma unroll
            for (int s = 0; s < NS; ++s) mul_by<C>(v[s][j], fj);
        });
    } else {   // Z term with controls on register bits; target: register position, or RB + bit
        if constexpr (NS == 1) {
            __builtin_unreachable();
        } else {
            const bool reg = tgt < RB, tb = !reg && ((zsrc >> ((tgt & 0x7f) - RB)) & 1) != 0;
            static_for<0, A>([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                const R w = add_im_conj_mul(R(0), v[1][j], v[0][j]);
                const bool b = reg ? ((j >> tgt) & 1) != 0 : tb;
                acc += ok && (j & creg) == creg ? (b ? -w : w) : R(0);
            });
        }
    }
}

// ---- one phase -------------------------------------------------------------------------------

// What a thread carries through a phase besides its amplitudes.
template <class R>
struct PhaseState {
    Cx<R> tf;          // factor per thread, pending: there is one
    Scale<R> sc;       // factor left out of the rotations, scaled: there is one
    unsigned sign;     // sign bit of the factor per thread
    bool pending, scaled;   // scaled: there is a real factor, the one left out or a sign
    __device__ __forceinline__ void init(double carry) {
        tf = cx<R>(R(1), R(0));
        sc.init(carry);
        sign = 0;
        pending = scaled = false;
    }
    // At the end of the phase: f is the factor to apply (its imaginary part only if pending), and
    // carry what rounding it left out, for the next phase (the norm of the whole state would
    // otherwise be off by up to half a unit in the last place per phase).
    __device__ __forceinline__ Cx<R> finish(double &carry) const {
        if (!pending && !scaled) return cx<R>(R(1), R(0));
        const double s = sizeof(R) == 8 ? sc.value() : pending ? sc.hi : (double)(R)sc.hi;
        carry = ((sc.hi - s) + sc.lo) * __builtin_amdgcn_rcp(s);
        const double t = __longlong_as_double(__double_as_longlong(s) ^ (long long)((u64)sign << 32));
        if (!pending) return cx<R>((R)t, R(0));
        return cx<R>((R)((double)tf.re * t), (R)((double)tf.im * t));
    }
};

// The ops of a phase on NS states in registers. ops: the pass's ops (one more is read than there
// are); tm: the item's coefficient table (B), kCoefs to a row; sums, red: the gradient terms of
// the sweep (NS == 2). One loop with one exit: with two, or with a loop inside for the ops that
// leave the registers alone, the compiler kept the registers of several iterations alive and
// copied them.
template <class R, int A, int NS, bool B, int NW>
__device__ __forceinline__ void run_phase(Cx<R> (&v)[NS][A], const RegOp<R> *ops, int op_begin, int n_ops, u64 base,
                                          unsigned off, const R *tm, PhaseState<R> &st, SlotSums<NW> &sums,
                                          double (*red)[NW], int n_slots, unsigned lane, unsigned wave) {
    const Cx<R> one = cx<R>(R(1), R(0));
#pragma unroll
    for (int s = 0; s < NS; ++s) apart(v[s]);
    R u = R(0);   // sum of Im(conj(lambda) phi), in the registers' scale
    OpWords<R> op, next;
    op.load(ops + op_begin);
    for (int k = op_begin; k < op_begin + n_ops; ++k) {
        op.arrive();
        next.load(ops + k + 1);   // read while this op runs
        const int slot = op.slot();
        if ((base & op.gctrl()) == op.gctrl()) {
            const unsigned code = op.code(), cthr = op.cthr();
            const auto controls = [&] { return (off & cthr) == cthr; };   // formed where an arm asks for it
            const int tgt = (int)((code >> 8) & 0xffu), creg = (int)((code >> 16) & 0xffu);
            R m[8];
            if constexpr (B) {
                const R *row = tm + (size_t)op.row() * kCoefs + (code >> 28);
                for (int i = 0; i < 4; ++i) m[i] = row[i];
            } else {
                for (int i = 0; i < 4; ++i) m[i] = op.coef(i);
            }
            R acc = R(0);   // gradient term, in the registers' scale
            int arm = (int)(code & 0xffu);
            if (arm < 16) arm += m[1] != R(0) ? 4 : 0;   // rotations: the form comes with the coefficients
            const u64 zsrc = (tgt & 0x80) ? base : (u64)off;
            const double scale = st.sc.hi;   // of the registers, before the op
#define QG_ARM(C_)                                                                                  \
    case C_: {                                                                                      \
        const bool ok = (C_) < 16 || controls();                                                   \
        const Cx<R> f = csel(ok, cx<R>(m[0], m[1]), one);                                          \
        if constexpr ((C_) / 4 == kFamAny) {   /* the second half of the matrix */                    \
            if constexpr (B) {                                                                     \
                for (int i = 4; i < 8; ++i) m[i] = tm[(size_t)op.row() * kCoefs + i];                 \
            } else {                                                                               \
                for (int i = 4; i < 8; ++i) m[i] = next.coef(i - 4);                                \
            }                                                                                      \
        }                                                                                          \
        reg_arm<(C_), R, A, NS>(v, m, f, creg, ok, (int)((code >> 24) & 0xfu), tgt, zsrc, acc);          \
        if constexpr ((C_) < 16) {                                                                    \
            st.sc.times(m[2], m[3]);                                                               \
            st.scaled = true;                                                                      \
        }                                                                                          \
        break;                                                                                     \
    }
#define QG_ARMS(C_) QG_ARM(C_) QG_ARM(C_ + 1) QG_ARM(C_ + 2) QG_ARM(C_ + 3)
            switch (arm) {
                QG_ARMS(0) QG_ARMS(4) QG_ARMS(8) QG_ARMS(12) QG_ARMS(16) QG_ARMS(20) QG_ARMS(24) QG_ARMS(28)
                QG_ARMS(32) QG_ARMS(36) QG_ARMS(40) QG_ARMS(44) QG_ARM(48) QG_ARM(49)
                case kArmThread:
                case kArmThreadCtrl: {
                    const bool b = ((off >> tgt) & 1u) != 0;
                    Cx<R> f = csel(b, cx<R>(m[0], m[1]), one);
                    if constexpr (NS == 2) acc = b ? -u : u;
                    if (arm == kArmThreadCtrl) {
                        const bool ok = controls();
                        f = csel(ok, f, one);
                        acc = ok ? acc : R(0);
                    }
                    st.tf = cmul(st.tf, f);
                    st.pending = true;
                    break;
                }
                case kArmOuter: {
                    const bool b = ((base >> tgt) & 1u) != 0, ok = controls();
                    const Cx<R> f = csel(ok && b, cx<R>(m[0], m[1]), one);
                    st.tf = cmul(st.tf, f);
                    st.pending = true;
                    if constexpr (NS == 2) acc = ok ? (b ? -u : u) : R(0);
                    break;
                }
                case kArmParity: {   // bits: of the tile, or 0x80 | of the state
                    const auto bit = [&](int x) {
                        return (x & 0x80) ? (unsigned)(base >> (x & 0x7f)) & 1u : (off >> x) & 1u;
                    };
                    const bool b = (bit(tgt) ^ bit(creg)) != 0;
                    if constexpr (NS == 2) acc = b ? -u : u;
                    st.tf = cmul(st.tf, csel(b, cx<R>(m[0], m[1]), one));
                    st.pending = true;
                    break;
                }
                case kArmPhase:
                    st.tf = cmul(st.tf, csel(controls(), cx<R>(m[0], m[1]), one));
                    st.pending = true;
                    break;
                case kArmSign:
                    st.sign ^= controls() ? 0x80000000u : 0u;
                    st.scaled = true;
                    break;
                case kArmU:
                    if constexpr (NS == 2) {
                        R w = R(0);
                        static_for<0, A>([&](auto jc) __attribute__((always_inline)) {
                            constexpr int j = decltype(jc)::value;
                            w = add_im_conj_mul(w, v[1][j], v[0][j]);
                        });
                        u = w;
                    }
                    break;
                case kArmFlush:
                    if constexpr (NS == 2) sums.flush(tgt, red, n_slots, lane, wave);
                    break;
                default: break;
            }
#undef QG_ARM
#undef QG_ARMS
            if constexpr (NS == 2)
                if (slot >= 0) sums.add((double)acc, scale * scale, slot, lane);
        }
        op = next;
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) apart(v[s]);
}

// ---- layouts ---------------------------------------------------------------------------------

// LDS index of local tile index l: bits 5 to 9 and 10 to 12 folded onto the low five, so that a
// wavefront whose lane bits start above bit 0 still spreads over the banks. Linear over XOR:
// swizzle(a ^ b) = swizzle(a) ^ swizzle(b).
__host__ __device__ __forceinline__ unsigned swizzle(unsigned l) { return l ^ ((l >> 5) & 31u) ^ ((l >> 10) & 31u); }

// Local-index bits of register index j in phase P (uniform: a scalar value).
template <int RB>
__device__ __forceinline__ unsigned reg_bits(const PhaseBits &P, int j) {
    unsigned l = 0;
#pragma unroll
    for (int k = 0; k < RB; ++k) l |= (((unsigned)j >> k) & 1u) << P.rb(k);
    return l;
}

template <int WB>
__device__ __forceinline__ unsigned phase_offset(const PhaseBits &P, unsigned lane, unsigned wave) {
    unsigned off = 0;
#pragma unroll
    for (int k = 0; k < 6; ++k) off |= ((lane >> k) & 1u) << P.lb(k);
#pragma unroll
    for (int k = 0; k < WB; ++k) off |= ((wave >> k) & 1u) << P.wb(k);
    return off;
}

// Registers of one state in phase layout (off, P) <- LDS tile t.
template <class R, int A, int RB>
__device__ __forceinline__ void regs_from_lds(Cx<R> (&v)[A], const Cx<R> *t, unsigned soff, const PhaseBits &P) {
    static_for<0, A>([&](auto jc) __attribute__((always_inline)) {
        constexpr int j = decltype(jc)::value;
        v[j] = t[soff ^ swizzle(reg_bits<RB>(P, j))];
    });
}

// LDS tile t <- registers, times the factor f of the phase.
template <class R, int A, int RB>
__device__ __forceinline__ void regs_to_lds(Cx<R> *t, const Cx<R> (&v)[A], unsigned soff, const PhaseBits &P,
                                            const PhaseState<R> &st, const Cx<R> &f) {
    // an opaque copy of soff: the addresses are formed here again (one XOR each) instead of being
    // kept from the phase's load through every op
    asm volatile("; phase store" : "+v"(soff));
    if (st.pending) {
        static_for<0, A>([&](auto jc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value;
            t[soff ^ swizzle(reg_bits<RB>(P, j))] = cmul(f, v[j]);
        });
    } else if (st.scaled) {
        static_for<0, A>([&](auto jc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value;
            t[soff ^ swizzle(reg_bits<RB>(P, j))] = cx<R>(v[j].re * f.re, v[j].im * f.re);
        });
    } else {
        static_for<0, A>([&](auto jc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value;
            t[soff ^ swizzle(reg_bits<RB>(P, j))] = v[j];
        });
    }
}

// HBM <-> swizzled LDS tile of 2^M amplitudes, all of a thread's 16-byte accesses in flight at
// once. Unit c T + tid has local index (c T + tid) << lw, whose two parts occupy disjoint bits:
// one deposit per thread and one per chunk (the same for the whole workgroup).
template <class R, int T, int M>
__device__ __forceinline__ void tile_in(Cx<R> *t, const Cx<R> *a, u64 base, const signed char *pos, int low) {
    constexpr int W = Unit<R>::W, lw = W == 2 ? 1 : 0, N = (1 << (M - lw)) / T;
    const u64 dt = base | deposit((unsigned)threadIdx.x << lw, pos, M, low);
    Amps<R> x[N];
#pragma unroll
    for (int c = 0; c < N; ++c) x[c] = load_unit(a, (dt | deposit((unsigned)(c * T) << lw, pos, M, low)) >> lw);
    const unsigned s = swizzle((unsigned)threadIdx.x << lw);
#pragma unroll
    for (int c = 0; c < N; ++c)
#pragma unroll
        for (int j = 0; j < W; ++j) t[s ^ swizzle(((unsigned)(c * T) << lw) | (unsigned)j)] = x[c].v[j];
}

template <class R, int T, int M>
__device__ __forceinline__ void tile_out(Cx<R> *a, const Cx<R> *t, u64 base, const signed char *pos, int low) {
    constexpr int W = Unit<R>::W, lw = W == 2 ? 1 : 0, N = (1 << (M - lw)) / T;
    const u64 dt = base | deposit((unsigned)threadIdx.x << lw, pos, M, low);
    const unsigned s = swizzle((unsigned)threadIdx.x << lw);
    Amps<R> x[N];
#pragma unroll
    for (int c = 0; c < N; ++c)
#pragma unroll
        for (int j = 0; j < W; ++j) x[c].v[j] = t[s ^ swizzle(((unsigned)(c * T) << lw) | (unsigned)j)];
#pragma unroll
    for (int c = 0; c < N; ++c) store_unit(a, (dt | deposit((unsigned)(c * T) << lw, pos, M, low)) >> lw, x[c]);
}

// ---- forward pass ----------------------------------------------------------------------------

// The program of a forward pass travels in the kernel arguments (under 4 KiB).
template <class R>
struct RegProgram {
    int n_ops, n_phases, low;
    alignas(4) signed char pos[kTilePosMax];
    PhaseBits phases[kMaxPhases];
    RegOp<R> ops[TileCfg<R>::MaxRegOps + 1];   // one more is read than there are
};
static_assert(sizeof(RegProgram<float>) <= 3584 && sizeof(RegProgram<double>) <= 3584, "kernel argument size");

// Batched passes (B): the state vector holds many circuits of one gate structure, item i's
// amplitudes at [i << item_shift, (i + 1) << item_shift), and no tile spans two items. An op
// then takes its coefficients from the tile item's table of n_rows rows of kCoefs.
// One tile per workgroup: persistent workgroups that load the next tile into registers while
// they work on the current one need 32 more VGPRs (3 workgroups per CU instead of 4) and
// measured slower.
template <class R, int M, int T, bool B>
__global__ __launch_bounds__(T) void k_tile_reg(Cx<R> *__restrict__ a, const RegProgram<R> prog, u64 first,
                                                const R *__restrict__ coefs, int n_rows, int item_shift) {
    constexpr int A = (1 << M) / T, RB = Log2<A>::v, WB = Log2<T / 64>::v;
    __shared__ Cx<R> t[1 << M];
    const u64 base = tile_base(first + blockIdx.x, prog.pos, M);
    const R *tm = nullptr;
    if constexpr (B) tm = coefs + (base >> item_shift) * (u64)n_rows * kCoefs;
    tile_in<R, T, M>(t, a, base, prog.pos, prog.low);
    __syncthreads();
    const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    Cx<R> v[1][A];
    SlotSums<1> none;
    double carry = 0.;
    for (int ph = 0; ph < prog.n_phases; ++ph) {
        const PhaseBits P = prog.phases[ph];
        const unsigned off = phase_offset<WB>(P, lane, wave);
        regs_from_lds<R, A, RB>(v[0], t, swizzle(off), P);
        PhaseState<R> st;
        st.init(carry);
        run_phase<R, A, 1, B, 1>(v, prog.ops, P.op_begin, P.n_ops, base, off, tm, st, none, nullptr, 0, lane, wave);
        const Cx<R> f = st.finish(carry);
        regs_to_lds<R, A, RB>(t, v[0], swizzle(off), P, st, f);
        __syncthreads();
    }
    tile_out<R, T, M>(a, t, base, prog.pos, prog.low);
}

// ---- adjoint sweep ---------------------------------------------------------------------------

struct SweepPass {
    int low;
    int op_begin;          // ops of the pass in the op table; its phases count from there
    int phase_begin, n_phases, n_slots;
    alignas(4) signed char pos[kTilePosMax];
};

// phi and lambda tiles in registers, one LDS tile each for the layout changes. Every LDS
// location written at the end of a phase is the one the same thread read at its start, so
// only the hand-overs between layouts need barriers. Each rotation's tile term is left in
// partial[slot * n_tiles + tile].
template <class R, int M, int T, bool B>
__global__ __launch_bounds__(T) void k_tile_sweep_reg(Cx<R> *__restrict__ phi, Cx<R> *__restrict__ lam,
                                                      const SweepPass pass, const RegOp<R> *__restrict__ ops,
                                                      const PhaseBits *__restrict__ phases,
                                                      double *__restrict__ partial, u64 n_tiles, u64 first,
                                                      const R *__restrict__ coefs, int n_rows, int item_shift) {
    constexpr int A = (1 << M) / T, RB = Log2<A>::v, WB = Log2<T / 64>::v, NW = T / 64;
    __shared__ Cx<R> tp[1 << M];
    __shared__ Cx<R> tl[1 << M];
    __shared__ double red[kMaxSweepSlots][NW];
    const u64 tile = first + blockIdx.x;
    const u64 base = tile_base(tile, pass.pos, M);
    const R *tm = nullptr;
    if constexpr (B) tm = coefs + (base >> item_shift) * (u64)n_rows * kCoefs;
    const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    Cx<R> v[2][A];
    tile_in<R, T, M>(tp, phi, base, pass.pos, pass.low);
    tile_in<R, T, M>(tl, lam, base, pass.pos, pass.low);
    for (int k = threadIdx.x; k < pass.n_slots * NW; k += T) red[k / NW][k % NW] = 0.;   // slots off in this tile
    __syncthreads();
    SlotSums<NW> sums;
    sums.init();
    double carry = 0.;
    for (int ph = 0; ph < pass.n_phases; ++ph) {
        const PhaseBits P = phases[pass.phase_begin + ph];
        const unsigned off = phase_offset<WB>(P, lane, wave);
        const unsigned soff = swizzle(off);
        regs_from_lds<R, A, RB>(v[0], tp, soff, P);
        regs_from_lds<R, A, RB>(v[1], tl, soff, P);
        PhaseState<R> st;
        st.init(carry);
        run_phase<R, A, 2, B, NW>(v, ops, pass.op_begin + P.op_begin, P.n_ops, base, off, tm, st, sums, red,
                                  pass.n_slots, lane, wave);
        const Cx<R> f = st.finish(carry);
        regs_to_lds<R, A, RB>(tp, v[0], soff, P, st, f);
        regs_to_lds<R, A, RB>(tl, v[1], soff, P, st, f);
        __syncthreads();
    }
    tile_out<R, T, M>(phi, tp, base, pass.pos, pass.low);
    tile_out<R, T, M>(lam, tl, base, pass.pos, pass.low);
    for (int k = threadIdx.x; k < pass.n_slots; k += T) {
        double s = 0.;
#pragma unroll
        for (int w = 0; w < NW; ++w) s += red[k][w];
        partial[(u64)k * n_tiles + tile] = s;
    }
}

// ---- ops of a planned phase (host) -------------------------------------------------------------

// Packed form of a phase layout (ops [begin, begin + n) of its pass).
inline PhaseBits phase_bits(const PhasePlan &P, int begin, int n) {
    QG_REQUIRE(P.regs.size() <= 5 && P.lanes.size() <= 6 && P.waves.size() <= 5, "register phase: too many bits");
    PhaseBits h;
    std::memset(&h, 0, sizeof(h));
    for (int b = 0; b < (int)P.regs.size(); ++b) h.set(b, P.regs[b]);
    for (int b = 0; b < (int)P.lanes.size(); ++b) h.set(5 + b, P.lanes[b]);
    for (int b = 0; b < (int)P.waves.size(); ++b) h.set(11 + b, P.waves[b]);
    h.op_begin = begin;
    h.n_ops = n;
    return h;
}

// Coefficients of a gate (kCoefs of them), as the ops read them.
template <class R>
void gate_coefs(const RegGate &g, R *c) {
    for (int i = 0; i < kCoefs; ++i) c[i] = R(0);
    if (g.kind == kGateY) {
        rotation_coefs(c, g.m.m[0][0].real(), g.m.m[0][1].real());
    } else if (g.kind == kGateX) {
        rotation_coefs(c, g.m.m[0][0].real(), -g.m.m[0][1].imag());
    } else if (g.kind == kGateDiag) {
        const std::complex<long double> r =
            std::complex<long double>(g.m.m[1][1]) / std::complex<long double>(g.m.m[0][0]);
        c[0] = (R)g.m.m[0][0].real(); c[1] = (R)g.m.m[0][0].imag();
        c[2] = (R)g.m.m[1][1].real(); c[3] = (R)g.m.m[1][1].imag();
        c[4] = (R)r.real(); c[5] = (R)r.imag();
    } else if (g.kind == kGateAny) {
        double a[8];
        gate_matrix_to_array(g.m, a);
        for (int i = 0; i < 8; ++i) c[i] = (R)a[i];
    }
}

template <class R>
void append_flush(std::vector<RegOp<R>> &out, int group) {
    RegOp<R> op;
    std::memset(&op, 0, sizeof(op));
    op.code = (unsigned)kArmFlush | (unsigned)group << 8;
    op.slot = -1;
    out.push_back(op);
}

// A phase of the whole state: diagonal gates on register bits leave one each.
typedef std::complex<long double> GlobalPhase;

// Appends the ops of gate g (index `row` in the coefficient table) in phase P. local: tile bit
// of a state lane, -1 outside the tile. n_slots counts the gradient slots given out; have_u: the
// sum of kArmU is that of the registers as they are; global takes the phases of the whole state.
template <class R>
void append_ops(std::vector<RegOp<R>> &out, const RegGate &g, int row, const PhasePlan &P, const int *local,
                int &n_slots, bool &have_u, GlobalPhase &global) {
    if (g.pauli != 0 && n_slots > 0 && n_slots % 16 == 0) append_flush(out, n_slots / 16 - 1);
    const int rb = (int)P.regs.size();
    auto position = [&](int bit) { return (int)(std::find(P.regs.begin(), P.regs.end(), bit) - P.regs.begin()); };
    RegOp<R> op;
    std::memset(&op, 0, sizeof(op));
    op.row = row;
    op.slot = -1;
    int creg = 0;
    for (int c : g.ctrl) {
        if (local[c] < 0)
            op.gctrl |= u64(1) << c;
        else if (position(local[c]) < rb)
            creg |= 1 << position(local[c]);
        else
            op.cthr |= 1u << local[c];
    }
    R c[kCoefs];
    gate_coefs<R>(g, c);
    auto push = [&](int arm, int tgt, int regs, int coff, int slot, const RegOp<R> &base) {
        RegOp<R> o = base;
        o.code = (unsigned)arm | (unsigned)tgt << 8 | (unsigned)regs << 16 |
                 (unsigned)(slot >= 0 ? g.pauli : 0) << 24 | (unsigned)coff << 28;
        o.slot = slot;
        for (int i = 0; i < 4; ++i) o.c[i] = c[coff + i];
        out.push_back(o);
    };
    const int lt = local[g.target];
    const int tp = lt < 0 ? rb : position(lt);
    if (g.kind != kGateDiag) {
        QG_REQUIRE(tp < rb, "register phase: pair target is not a register bit");
        const int fam = g.kind == kGateY ? kFamY : g.kind == kGateX ? kFamX : g.kind == kGateSwap ? kFamSwap : kFamAny;
        QG_REQUIRE((fam != kFamY && fam != kFamX) || g.ctrl.empty(), "register phase: controlled rotation");
        push(4 * fam + tp, 0, creg, 0, g.pauli != 0 ? n_slots++ : -1, op);
        if (fam == kFamAny) push(kArmNone, 0, 0, 4, -1, op);   // m10, m11
        have_u = false;
        return;
    }
    const std::complex<double> d0 = g.m.m[0][0], d1 = g.m.m[1][1];
    int slot = g.pauli != 0 ? n_slots++ : -1;
    // factor on the amplitudes whose bits (masks of o, regs) are all set
    auto factor = [&](RegOp<R> o, int regs, int coff, std::complex<double> f) {
        const bool sign = f == -1. && g.pauli == 0;
        const int n = __builtin_popcount((unsigned)regs);
        if (n == 0) {
            push(sign ? kArmSign : kArmPhase, 0, 0, coff, -1, o);
        } else if (n == 1) {
            push(4 * (sign ? kFamSign : kFamFactor) + __builtin_ctz((unsigned)regs), 0, regs, coff, -1, o);
        } else if (n == 2) {
            int i = 0;
            while (pair2_mask(i) != regs) ++i;
            push((sign ? kArmSign2 : kArmPair2) + i, 0, regs, coff, -1, o);
        } else {
            push(kArmFactorAny, 0, regs, coff, -1, o);
        }
    };
    // diag(m00, m11) = m00 on the controls, then the ratio m11 / m00 on the controls and the target.
    // With both entries as factors, each rounded, their moduli (equal, and off by the same rounding)
    // would scale the whole state; of many rotations by one angle these errors add up.
    const bool one0 = d0 == 1. && g.pauli == 0;   // m00 == 1 whatever the parameter
    if (!one0) {
        const long double n = std::norm(GlobalPhase(d0));
        if (g.ctrl.empty() && std::abs(n - 1.L) < 1e-14L)
            global *= GlobalPhase(d0) / std::sqrt(n);
        else
            factor(op, creg, 0, d0);
    }
    const int coff = one0 ? 2 : 4;
    if (g.parity >= 0) {
        auto where = [&](int lane) { return local[lane] >= 0 ? local[lane] : 0x80 | lane; };
        for (int lane : {g.target, g.parity})
            QG_REQUIRE(local[lane] < 0 || position(local[lane]) >= rb, "register phase: parity on a register bit");
        if (slot >= 0 && !have_u) {
            RegOp<R> u;
            std::memset(&u, 0, sizeof(u));
            push(kArmU, 0, 0, 0, -1, u);
            have_u = true;
        }
        push(kArmParity, where(g.target), where(g.parity), coff, slot, op);
        return;
    }
    if (slot >= 0 && creg == 0 && tp < rb) {   // term and factor in one op
        push(4 * kFamZ + tp, 0, 1 << tp, coff, slot, op);
        return;
    }
    if (slot >= 0 && creg == 0) {
        if (!have_u) {
            RegOp<R> u;
            std::memset(&u, 0, sizeof(u));
            push(kArmU, 0, 0, 0, -1, u);
            have_u = true;
        }
        push(lt < 0 ? kArmOuter : op.cthr != 0 ? kArmThreadCtrl : kArmThread, lt >= 0 ? lt : g.target, 0, coff, slot,
             op);
        return;
    }
    if (slot >= 0)   // target: register position, or RB + local bit, or 0x80 | RB + state bit
        push(kArmZAny, tp < rb ? tp : lt >= 0 ? rb + lt : 0x80 | (rb + g.target), creg, 0, slot, op);
    int treg = creg;
    if (lt < 0)
        op.gctrl |= u64(1) << g.target;
    else if (tp < rb)
        treg |= 1 << tp;
    else
        op.cthr |= 1u << lt;
    factor(op, treg, coff, one0 ? d1 : d1 / d0);
}

// The register gates of the gate list of a sweep: rotations whole (their gradient terms are
// taken right before them), fixed gates split as in the forward pass.
inline std::vector<RegGate> sweep_gates(const std::vector<SweepGate> &gates, int n_lanes) {
    std::vector<RegGate> out;
    out.reserve(gates.size() + gates.size() / 4);
    const std::vector<int> role = parity_roles(
        (int)gates.size(), n_lanes, [&](int i) -> const SweepGate & { return gates[i]; },
        [&](int i) { return gates[i].pauli == 0 && gates[i].ctrl.size() == 1 && is_x(gates[i].udag); },
        [&](int i) {
            const SweepGate &g = gates[i];
            return g.ctrl.empty() && (g.pauli == 3 || (g.pauli == 0 && diag2(g.udag) && has_ratio(g.udag)));
        });
    for (int i = 0; i < (int)gates.size(); ++i) {
        const SweepGate &g = gates[i];
        if (role[i] == kDropped) continue;
        const size_t at = out.size();
        if (g.pauli == 0) {
            append_fixed(out, g.udag, g.ctrl, g.target, i);
        } else {
            RegGate r;
            r.kind = g.pauli == 3 ? kGateDiag : !g.ctrl.empty() ? kGateAny : g.pauli == 1 ? kGateX : kGateY;
            r.target = g.target;
            r.pauli = g.pauli;
            r.source = i;
            r.ctrl = g.ctrl;
            r.m = g.udag;
            out.push_back(r);
        }
        if (role[i] != kKept && out.size() > at) out.back().parity = role[i];
    }
    return out;
}

// A planned register pass: phases (op_begin from 0) and ops.
template <class R>
struct BuiltPass {
    std::vector<int> bits;
    int low = 0;
    std::vector<PhaseBits> phases;
    std::vector<RegOp<R>> ops;
    std::vector<int> slot_gate;    // gate of each gradient slot
    std::vector<int> gates;        // gates of the pass
};

// Passes over a gate list: tiles of m of n lanes that hold the lowest `low`, rb register and wb
// wave bits, at most max_gates gates, max_ops ops and max_phases phases a pass. Gates whose tile has no bit left
// for them (tile bits == low bits) are refused by the caller's choice of m > low. Phases of the whole
// state are applied once per pass (the amplitudes are wanted) or left out (kNoGlobalPhase:
// expectation values and gradients do not depend on them; batched rotations have theirs in no table).
enum GlobalPhases { kGlobalPhase, kNoGlobalPhase };
//
// take(pass) is called with each pass as it is planned, so that the first ones can run meanwhile.
template <class R, class Take>
void for_each_pass(const std::vector<RegGate> &gates, int n, int m, int low, int rb, int wb, int max_gates,
                   int max_ops, int max_phases, GlobalPhases keep, Take take) {
    QG_REQUIRE(low < m && m <= n, "register pass: %d tile bits, %d low, %d lanes", m, low, n);
    const int ng = (int)gates.size();
    std::vector<PlanGate> pg(ng);
    for (int i = 0; i < ng; ++i)
        pg[i] = PlanGate{gates[i].target, &gates[i].ctrl, gates[i].kind == kGateDiag,
                         gates[i].kind == kGateAny ? 2 : 1, gates[i].pauli != 0 ? 1 : 0, gates[i].parity};
    std::vector<char> done(ng, 0);
    for (int first = 0; first < ng;) {
        // a diagonal gate on a register bit can take two ops: a pass that comes out too long is
        // planned again with fewer gates
        for (int limit = std::min(max_gates, max_ops);;) {
            std::vector<char> now(done);
            const PassBits pb = next_pass(pg, now, first, n, m, low, limit, kMaxSweepSlots);
            QG_REQUIRE(!pb.gates.empty(), "register pass takes no gate");
            int local[64];
            for (int b = 0; b < 64; ++b) local[b] = -1;
            for (int j = 0; j < m; ++j) local[pb.bits[j]] = j;
            BuiltPass<R> bp;
            bp.bits = pb.bits;
            bp.low = pb.low;
            bp.gates = pb.gates;
            int slots = 0;
            GlobalPhase global(1.L);
            for (const PhasePlan &P : plan_phases(pg, pb.gates, local, n, m, rb, wb)) {
                const int begin = (int)bp.ops.size();
                bool have_u = false;
                for (int gi : P.order) {
                    append_ops<R>(bp.ops, gates[gi], gi, P, local, slots, have_u, global);
                    if (gates[gi].pauli != 0) bp.slot_gate.push_back(gi);
                }
                bp.phases.push_back(phase_bits(P, begin, (int)bp.ops.size() - begin));
            }
            if (keep == kGlobalPhase && global != GlobalPhase(1.L)) {
                RegOp<R> op;
                std::memset(&op, 0, sizeof(op));
                op.code = (unsigned)kArmPhase;
                op.slot = -1;
                op.c[0] = (R)global.real();
                op.c[1] = (R)global.imag();
                bp.ops.push_back(op);
                bp.phases.back().n_ops += 1;
            }
            if (slots > 0) {   // the last slots
                append_flush(bp.ops, (slots - 1) / 16);
                bp.phases.back().n_ops += 1;
            }
            if ((int)bp.ops.size() > max_ops || (int)bp.phases.size() > max_phases) {
                QG_REQUIRE(limit > 2, "register pass: a gate takes too many ops");
                int weight = 0;
                for (int gi : pb.gates) weight += pg[gi].weight;
                limit = std::min(weight - 1, (int)bp.phases.size() > max_phases
                                                 ? weight * 3 / 4
                                                 : weight * max_ops / (int)bp.ops.size());
                continue;
            }
            done.swap(now);
            take(std::move(bp));
            break;
        }
        while (first < ng && done[first]) ++first;
    }
}

template <class R>
std::vector<BuiltPass<R>> build_passes(const std::vector<RegGate> &gates, int n, int m, int low, int rb, int wb,
                                       int max_gates, int max_ops, int max_phases, GlobalPhases keep) {
    std::vector<BuiltPass<R>> out;
    for_each_pass<R>(gates, n, m, low, rb, wb, max_gates, max_ops, max_phases, keep,
                     [&](BuiltPass<R> &&bp) { out.push_back(std::move(bp)); });
    return out;
}

inline void set_positions(signed char *pos, const std::vector<int> &bits) {
    for (int j = 0; j < kTilePosMax; ++j) pos[j] = j < (int)bits.size() ? (signed char)bits[j] : (signed char)0;
}

template <class R>
RegProgram<R> reg_program(const BuiltPass<R> &bp) {
    RegProgram<R> rp;
    std::memset(&rp, 0, sizeof(rp));
    rp.n_ops = (int)bp.ops.size();
    rp.n_phases = (int)bp.phases.size();
    rp.low = bp.low;
    set_positions(rp.pos, bp.bits);
    std::copy(bp.phases.begin(), bp.phases.end(), rp.phases);
    std::copy(bp.ops.begin(), bp.ops.end(), rp.ops);
    return rp;
}

}  // namespace

}  // namespace qg
