// lambda (+)= H psi over a full-size tile, for Pauli sums grouped by X mask: device code shared by
// the single-circuit passes (k_tile.hip) and the batched ones (k_batch.hip), and its planning.
//
// Amplitude x of lambda takes sum over groups g of c_g(x) psi[x ^ xmask_g], where c_g(x) is the sum
// over the group's terms k of c_k (-1)^popcount(x & z_k). A thread holds E amplitudes of the tile,
// whose indices differ in log2(E) bits that are the same for every thread and tile, so a term
// enters the E coefficients of a thread with one sign of the thread times a Walsh pattern of E
// signs known on the host. The terms of a group are sorted by pattern: a thread sums each
// pattern's terms (one parity and one FMA a term instead of one per term and amplitude) and one
// Walsh-Hadamard transform of the E sums gives its coefficients. FP64 throughout, fixed order.
// (24-qubit ZZ and X sum in complex64, three passes: 202 us each before, when every amplitude took
// the parity of every term; 87 us now, 4.1 TB/s of the 2.7 passes over a state that each makes.)
#pragma once

#include <algorithm>
#include <vector>

#include "kernels.hpp"
#include "tile_common.hpp"

namespace qg {

namespace {

// Threads of a workgroup: 8 amplitudes each (with 16, the coefficients and sums take 188 registers
// and two waves share a SIMD instead of four).
template <class R>
constexpr int kPauliThreads = sizeof(R) == 4 ? 512 : 256;
constexpr int kPauliPatterns = 8;   // amplitudes a thread holds

struct PauliZ {
    u64 zmask;
    int coef;      // index in the coefficient array: 2 k, or 2 k + 1 for an imaginary coefficient
    int pad;
};

// A group within its pass: terms [begin[p], begin[p + 1]) of the sorted list have pattern p with
// real coefficients, [ibegin[p], ibegin[p + 1]) with imaginary ones.
struct PauliWork {
    unsigned xlocal;
    int plain;     // only pattern 0, real: one coefficient for all of a thread's amplitudes
    int imag;      // there are imaginary coefficients
    int begin[kPauliPatterns + 1], ibegin[kPauliPatterns + 1];
};

// Sums of the terms of each pattern, then the coefficients of the thread's E amplitudes.
template <int E>
__device__ __forceinline__ void pauli_coefs(double (&c)[E], const int *begin, const PauliZ *zs, const double *coefs,
                                            u64 dt) {
#pragma unroll
    for (int p = 0; p < E; ++p) {
        double s = 0.;
        for (int k = begin[p]; k < begin[p + 1]; ++k) {
            const PauliZ z = zs[k];
            s = __builtin_fma((__popcll(dt & z.zmask) & 1) ? -1. : 1., coefs[z.coef], s);
        }
        c[p] = s;
    }
#pragma unroll
    for (int h = 1; h < E; h <<= 1)
#pragma unroll
        for (int p = 0; p < E; ++p)
            if ((p & h) == 0) {
                const double a = c[p], b = c[p + h];
                c[p] = a + b;
                c[p + h] = a - b;
            }
}

// H psi of a thread's E amplitudes, added to (ar, ai). l0: local index of the first one (the others
// differ from it by the constant bits at(e)); dt: its state index; psi(l, c): the tile's amplitude of
// local index l ^ c, c constant.
template <class R, int E, class At, class Psi>
__device__ __forceinline__ void pauli_apply(double (&ar)[E], double (&ai)[E], unsigned l0, u64 dt, At at, Psi psi,
                                            const PauliWork *__restrict__ works, int n_groups,
                                            const PauliZ *__restrict__ zs, const double *__restrict__ coefs) {
    for (int g = 0; g < n_groups; ++g) {
        const PauliWork &w = works[g];
        const unsigned lx = l0 ^ w.xlocal;
        if (w.plain) {
            double s = 0.;
            for (int k = w.begin[0]; k < w.begin[1]; ++k) {
                const PauliZ z = zs[k];
                s = __builtin_fma((__popcll(dt & z.zmask) & 1) ? -1. : 1., coefs[z.coef], s);
            }
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const Cx<R> v = psi(lx, at(e));
                ar[e] = __builtin_fma(s, (double)v.re, ar[e]);
                ai[e] = __builtin_fma(s, (double)v.im, ai[e]);
            }
            continue;
        }
        double c[E];
        pauli_coefs<E>(c, w.begin, zs, coefs, dt);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const Cx<R> v = psi(lx, at(e));
            ar[e] = __builtin_fma(c[e], (double)v.re, ar[e]);
            ai[e] = __builtin_fma(c[e], (double)v.im, ai[e]);
        }
        if (w.imag) {
            pauli_coefs<E>(c, w.ibegin, zs, coefs, dt);
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const Cx<R> v = psi(lx, at(e));
                ar[e] = __builtin_fma(-c[e], (double)v.im, ar[e]);
                ai[e] = __builtin_fma(c[e], (double)v.re, ai[e]);
            }
        }
    }
}

// One full-size tile (2^MB amplitudes, kPauliThreads<R> threads); returns the thread's part of
// Re<psi|lambda> if `dot` is set. tp: the psi tile, in the order of its local index.
template <class R, int MB>
__device__ __forceinline__ double pauli_full_tile(const Cx<R> *tp, Cx<R> *__restrict__ lam, u64 base,
                                                  const signed char *pos, int low, bool accumulate, bool dot,
                                                  const PauliWork *__restrict__ works, int n_groups,
                                                  const PauliZ *__restrict__ zs, const double *__restrict__ coefs) {
    constexpr int W = Unit<R>::W, lw = W == 2 ? 1 : 0, T = kPauliThreads<R>, N = (1 << (MB - lw)) / T, E = N * W;
    static_assert(E == kPauliPatterns, "amplitudes a thread");
    const u64 dt = base | deposit((unsigned)threadIdx.x << lw, pos, MB, low);
    double ar[E], ai[E];
    u64 unit[N];
#pragma unroll
    for (int c = 0; c < N; ++c) unit[c] = (dt | deposit((unsigned)(c * T) << lw, pos, MB, low)) >> lw;
    if (accumulate) {
        Amps<R> x[N];
#pragma unroll
        for (int c = 0; c < N; ++c) x[c] = load_unit(lam, unit[c]);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            ar[e] = (double)x[e / W].v[e % W].re;
            ai[e] = (double)x[e / W].v[e % W].im;
        }
    } else {
#pragma unroll
        for (int e = 0; e < E; ++e) ar[e] = ai[e] = 0.;
    }
    // local index of amplitude e: unit (e / W) T + tid, amplitude e % W of it
    const unsigned l0 = (unsigned)threadIdx.x << lw;
    const auto at = [](int e) { return ((unsigned)(e / W * T) << lw) | (unsigned)(e % W); };
    pauli_apply<R, E>(ar, ai, l0, dt, at, [&](unsigned l, unsigned c) { return tp[l ^ c]; }, works, n_groups, zs,
                      coefs);
    double sum = 0.;
#pragma unroll
    for (int q = 0; q < N; ++q) {
        Amps<R> out;
#pragma unroll
        for (int j = 0; j < W; ++j) {
            const int e = q * W + j;
            out.v[j] = cx<R>((R)ar[e], (R)ai[e]);
            if (dot) {
                const Cx<R> v = tp[l0 | at(e)];
                sum += (double)v.re * (double)out.v[j].re + (double)v.im * (double)out.v[j].im;
            }
        }
        store_unit(lam, unit[q], out);
    }
    return sum;
}

// The groups [first, first + n) of a pass on tiles whose bits are `bits` (ascending), in workgroups
// of `threads` with kPauliPatterns amplitudes a thread: their works and sorted terms. n_y(k): number
// of Y factors of term k.
template <class R, class NY>
void plan_pauli_pass(const std::vector<PauliGroup> &groups, int first, int n, const std::vector<u64> &zmask, NY n_y,
                     const std::vector<int> &bits, int threads, std::vector<PauliWork> &works,
                     std::vector<PauliZ> &zs) {
    constexpr int W = Unit<R>::W, lw = W == 2 ? 1 : 0;
    // state bits in which a thread's amplitudes differ: unit bits above the workgroup's, and (W ==
    // 2) the amplitude inside the unit
    std::vector<int> own;
    if (W == 2) own.push_back(bits[0]);
    int tb = 0;
    while ((1 << tb) < threads) ++tb;
    for (int j = lw + tb; j < (int)bits.size(); ++j) own.push_back(bits[j]);
    auto pattern = [&](u64 z) {
        int p = 0;
        for (size_t b = 0; b < own.size(); ++b) p |= (int)((z >> own[b]) & 1) << b;
        return p;
    };
    for (int i = first; i < first + n; ++i) {
        const PauliGroup &g = groups[i];
        PauliWork w;
        w.xlocal = g.xlocal;
        w.imag = 0;
        w.plain = 1;
        for (int im = 0; im < 2; ++im) {
            int *begin = im ? w.ibegin : w.begin;
            for (int p = 0; p < kPauliPatterns; ++p) {
                begin[p] = (int)zs.size();
                for (int k = g.first; k < g.first + g.count; ++k) {
                    if ((n_y(k) & 1) != im || pattern(zmask[k]) != p) continue;
                    zs.push_back(PauliZ{zmask[k], 2 * k + im, 0});
                    if (im) w.imag = 1;
                    if (im || p != 0) w.plain = 0;
                }
            }
            begin[kPauliPatterns] = (int)zs.size();
        }
        works.push_back(w);
    }
}

}  // namespace

}  // namespace qg
