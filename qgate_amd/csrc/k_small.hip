// Circuits whose whole state fits one workgroup: <H> and the gradient without a pass over HBM.
//
// Small circuits are bound by latency: a pass over a few tiles takes about 10 us however little it
// does, and a gradient was 5 to 20 such launches, the copies of their tables and the waits between
// them. Here the state stays in one workgroup from |0...0> to the last gradient term: 2^M
// amplitudes (M >= n; amplitudes above 2^n are zero and stay zero) in 2^(M - 3) threads, 8 each,
// worked on by the register engine of the tile passes (tile_reg.hpp), with LDS for its layout
// changes. No op has a bit outside the tile.
// What is left is latency too: at 13 qubits an op takes 0.4 to 0.6 us, of decoding, LDS hand-overs and
// table lines, with 4 waves on each SIMD of one compute unit (307 gates, 176 ops forward: 99 us, the
// sweep 137 us).
// <H> and gradient, whole calls, on the tile passes and here: 6 qubits complex128 337 -> 257 us (their
// host part differs by 60 us from process to process); 13 qubits complex64, 307 gates, 808 -> 671 us
// (540 since its ZZ rotations are parity gates); 96 circuits of 6 to 11 qubits 1580 -> 507 us.
//   one circuit      k_small_expect and k_small_sweep, one launch for each of the two calls
//   a batch          k_small_rows (coefficients of every item, from its parameters), then one
//                    workgroup an item, k_small_batch, from |0...0> to the item's gradient
#include <algorithm>
#include <complex>
#include <cstring>
#include <vector>

#include "circuit_rows.hpp"
#include "kernels.hpp"
#include "qg_runtime.hpp"
#include "small.hpp"
#include "table_layout.hpp"
#include "tile_common.hpp"
#include "tile_pauli.hpp"
#include "tile_reg.hpp"

namespace qg {

namespace {

constexpr int kSmallAmps = kPauliPatterns;   // amplitudes a thread
template <int M>
constexpr int kSmallThreads = (1 << M) / kSmallAmps;

// Largest state: two of them in LDS (128 KiB), 1024 threads at most. At these sizes the tile
// passes are still slower: 13 lanes in complex64, 12 layers of the RY RZ CZ ansatz, one circuit
// 936 us against 905 here, 512 of them (6 layers) 2.41 ms against 2.28; 12 lanes in complex128 921 us
// against 804, 400 of them 1.78 ms against 1.57.
template <class R>
constexpr int kSmallMaxBits = sizeof(R) == 4 ? 13 : 12;
// X and Y factors of a Pauli term that the general path takes.
template <class R>
constexpr int kPauliTileBits = sizeof(R) == 4 ? 12 : 11;

struct SmallPass {
    int op_begin, phase_begin, n_phases, n_slots, slot_begin;
};

// ---- device --------------------------------------------------------------------------------

// Brings a table that scalar loads will read entry by entry into this chip's L2, by vector loads of
// all its 64-byte lines at once: a scalar load that misses L2 too (the table was written by a copy or
// by another chip) took longer than an op, and a lone workgroup waited for it at every second op.
// The value is given to arrived() once other loads have been issued.
template <int T>
__device__ __forceinline__ unsigned touch(const void *table, int bytes) {
    const unsigned *w = static_cast<const unsigned *>(table);
    const int lines = (bytes + 63) / 64;
    unsigned x = 0;
#pragma unroll 4
    for (int i = threadIdx.x; i < lines; i += T) x |= w[i * 16];
    return x;
}
__device__ __forceinline__ void arrived(unsigned x) { asm volatile("; touched" ::"v"(x)); }

template <class R, int M>
__device__ __forceinline__ void small_zero(Cx<R> *t) {
    constexpr int T = kSmallThreads<M>;
#pragma unroll
    for (int c = 0; c < kSmallAmps; ++c) {
        const unsigned l = (unsigned)(c * T) + threadIdx.x;
        t[l] = cx<R>(l == 0 ? R(1) : R(0), R(0));   // swizzle(0) == 0
    }
    __syncthreads();
}

template <class R, int M, bool B>
__device__ __forceinline__ void small_forward(Cx<R> *t, const RegOp<R> *__restrict__ ops,
                                              const PhaseBits *__restrict__ phases, int n_phases, const R *tm) {
    constexpr int T = kSmallThreads<M>, A = kSmallAmps, RB = Log2<A>::v, WB = Log2<T / 64>::v;
    const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    Cx<R> v[1][A];
    SlotSums<1> none;
    double carry = 0.;
    for (int ph = 0; ph < n_phases; ++ph) {
        const PhaseBits P = phases[ph];
        const unsigned off = phase_offset<WB>(P, lane, wave), soff = swizzle(off);
        regs_from_lds<R, A, RB>(v[0], t, soff, P);
        PhaseState<R> st;
        st.init(carry);
        run_phase<R, A, 1, B, 1>(v, ops, P.op_begin, P.n_ops, 0, off, tm, st, none, nullptr, 0, lane, wave);
        const Cx<R> f = st.finish(carry);
        regs_to_lds<R, A, RB>(t, v[0], soff, P, st, f);
        __syncthreads();
    }
}

// put(l, a): lambda's amplitude of index l. Returns the thread's part of Re<psi|lambda>.
template <class R, int M, class Put>
__device__ __forceinline__ double small_pauli(const Cx<R> *t, const PauliWork *__restrict__ works, int n_works,
                                              const PauliZ *__restrict__ zs, const double *__restrict__ coefs,
                                              Put put) {
    constexpr int W = Unit<R>::W, lw = W == 2 ? 1 : 0, T = kSmallThreads<M>, E = kSmallAmps;
    const unsigned l0 = threadIdx.x << lw;
    const auto at = [](int e) { return ((unsigned)(e / W * T) << lw) | (unsigned)(e % W); };
    double ar[E], ai[E];
#pragma unroll
    for (int e = 0; e < E; ++e) ar[e] = ai[e] = 0.;
    pauli_apply<R, E>(ar, ai, l0, l0, at, [&](unsigned l, unsigned c) { return t[swizzle(l) ^ swizzle(c)]; }, works,
                      n_works, zs, coefs);
    double sum = 0.;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const Cx<R> out = cx<R>((R)ar[e], (R)ai[e]), v = t[swizzle(l0) ^ swizzle(at(e))];
        sum += (double)v.re * (double)out.re + (double)v.im * (double)out.im;
        put(l0 | at(e), out);
    }
    return sum;
}

template <class R, int M, bool B>
__device__ __forceinline__ void small_back(Cx<R> *tp, Cx<R> *tl, double (*red)[kSmallThreads<M> / 64],
                                           const RegOp<R> *__restrict__ ops, const PhaseBits *__restrict__ phases,
                                           const SmallPass *__restrict__ passes, int n_passes,
                                           const int *__restrict__ slot_gate, double *terms, const R *tm) {
    constexpr int T = kSmallThreads<M>, A = kSmallAmps, RB = Log2<A>::v, NW = T / 64, WB = Log2<NW>::v;
    const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    Cx<R> v[2][A];
    SlotSums<NW> sums;
    sums.init();
    double carry = 0.;
    for (int p = 0; p < n_passes; ++p) {
        const SmallPass ps = passes[p];
        for (int ph = 0; ph < ps.n_phases; ++ph) {
            const PhaseBits P = phases[ps.phase_begin + ph];
            const unsigned off = phase_offset<WB>(P, lane, wave), soff = swizzle(off);
            regs_from_lds<R, A, RB>(v[0], tp, soff, P);
            regs_from_lds<R, A, RB>(v[1], tl, soff, P);
            PhaseState<R> st;
            st.init(carry);
            run_phase<R, A, 2, B, NW>(v, ops, ps.op_begin + P.op_begin, P.n_ops, 0, off, tm, st, sums, red,
                                      ps.n_slots, lane, wave);
            const Cx<R> f = st.finish(carry);
            regs_to_lds<R, A, RB>(tp, v[0], soff, P, st, f);
            regs_to_lds<R, A, RB>(tl, v[1], soff, P, st, f);
            __syncthreads();
        }
        for (int k = threadIdx.x; k < ps.n_slots; k += T) {
            double s = 0.;
#pragma unroll
            for (int w = 0; w < NW; ++w) s += red[k][w];
            terms[slot_gate[ps.slot_begin + k]] = s;
        }
        __syncthreads();
    }
}

// The state's 2^n amplitudes between HBM and the swizzled LDS tile (zero above).
template <class R, int M>
__device__ __forceinline__ void small_store(Cx<R> *a, const Cx<R> *t, int n) {
    constexpr int W = Unit<R>::W, lw = W == 2 ? 1 : 0, T = kSmallThreads<M>, N = kSmallAmps / W;
#pragma unroll
    for (int c = 0; c < N; ++c) {
        const unsigned u = (unsigned)(c * T) + threadIdx.x;
        Amps<R> x;
#pragma unroll
        for (int j = 0; j < W; ++j) x.v[j] = t[swizzle(u << lw | (unsigned)j)];
        if (u < (1u << n) >> lw) store_unit(a, u, x);
    }
}

template <class R, int M>
__device__ __forceinline__ void small_load(Cx<R> *t, const Cx<R> *a, int n) {
    constexpr int W = Unit<R>::W, lw = W == 2 ? 1 : 0, T = kSmallThreads<M>, N = kSmallAmps / W;
    Amps<R> x[N];
#pragma unroll
    for (int c = 0; c < N; ++c) {
        const unsigned u = (unsigned)(c * T) + threadIdx.x;
        if (u < (1u << n) >> lw) {
            x[c] = load_unit(a, u);
        } else {
#pragma unroll
            for (int j = 0; j < W; ++j) x[c].v[j] = cx<R>(R(0), R(0));
        }
    }
#pragma unroll
    for (int c = 0; c < N; ++c)
#pragma unroll
        for (int j = 0; j < W; ++j) t[swizzle(((unsigned)(c * T) + threadIdx.x) << lw | (unsigned)j)] = x[c].v[j];
}

template <class R, int M>
__global__ __launch_bounds__((kSmallThreads<M>)) void k_small_expect(Cx<R> *__restrict__ psi, Cx<R> *__restrict__ lam,
                                                                   int n, const RegOp<R> *__restrict__ ops, int n_ops,
                                                                   const PhaseBits *__restrict__ phases, int n_phases,
                                                                   const PauliWork *__restrict__ works, int n_works,
                                                                   const PauliZ *__restrict__ zs,
                                                                   const double *__restrict__ coefs, double *value) {
    __shared__ Cx<R> t[1 << M];
    __shared__ Cx<R> tl[1 << M];
    __shared__ double scratch[kSmallThreads<M> / 64];
    const unsigned warm = touch<kSmallThreads<M>>(ops, n_ops * (int)sizeof(RegOp<R>)) |
                          touch<kSmallThreads<M>>(phases, n_phases * (int)sizeof(PhaseBits));
    small_zero<R, M>(t);
    arrived(warm);
    small_forward<R, M, false>(t, ops, phases, n_phases, nullptr);
    const double dot = small_pauli<R, M>(t, works, n_works, zs, coefs,
                                         [&](unsigned l, const Cx<R> &a) { tl[swizzle(l)] = a; });
    small_store<R, M>(psi, t, n);
    const double s = block_sum_tile<kSmallThreads<M>>(dot, scratch);
    if (threadIdx.x == 0) value[0] = s;
    small_store<R, M>(lam, tl, n);
}

template <class R, int M>
__global__ __launch_bounds__((kSmallThreads<M>)) void k_small_sweep(const Cx<R> *__restrict__ phi,
                                                                  const Cx<R> *__restrict__ lam, int n,
                                                                  const RegOp<R> *__restrict__ ops, int n_ops,
                                                                  const PhaseBits *__restrict__ phases, int n_phases,
                                                                  const SmallPass *__restrict__ passes, int n_passes,
                                                                  const int *__restrict__ slot_gate, double *terms) {
    __shared__ Cx<R> tp[1 << M];
    __shared__ Cx<R> tl[1 << M];
    __shared__ double red[kMaxSweepSlots][kSmallThreads<M> / 64];
    const unsigned warm = touch<kSmallThreads<M>>(ops, n_ops * (int)sizeof(RegOp<R>)) |
                          touch<kSmallThreads<M>>(phases, n_phases * (int)sizeof(PhaseBits));
    small_load<R, M>(tp, phi, n);
    small_load<R, M>(tl, lam, n);
    arrived(warm);
    __syncthreads();
    small_back<R, M, false>(tp, tl, red, ops, phases, passes, n_passes, slot_gate, terms, nullptr);
}

// A group of a batch: where its tables and its items' data begin.
struct SmallGroup {
    int n_params, n_gates, n_terms;
    int f_rows, s_rows, f_row, s_row;   // coefficient rows: counts, first ones
    int f_phase, f_phases, f_op, n_ops; // ops of the sweep follow those of the forward pass
    int pass, n_passes;
    int work, n_works;
    int param;                          // first of its entries in the parameter map
    u64 params, obs, coefs, terms, value, grad;   // of its first item
};
struct SmallItem {
    int group, index;
};

template <class R>
__global__ __launch_bounds__(256) void k_small_rows(const SmallGroup *__restrict__ groups,
                                                    const SmallItem *__restrict__ items,
                                                    const BRow<R> *__restrict__ rows,
                                                    const double *__restrict__ params, R *__restrict__ coefs) {
    const SmallItem it = items[blockIdx.x];
    const SmallGroup g = groups[it.group];
    const int n = g.f_rows + g.s_rows;
    const double *p = params + g.params + (u64)it.index * (u64)g.n_params;
    R *out = coefs + (g.coefs + (u64)it.index * (u64)n) * kCoefs;
    for (int k = threadIdx.x; k < n; k += 256)
        row_coefs(rows[k < g.f_rows ? g.f_row + k : g.s_row + (k - g.f_rows)], p, out + (u64)k * kCoefs);
}

template <class R, int M>
__global__ __launch_bounds__((kSmallThreads<M>)) void k_small_batch(
    const SmallGroup *__restrict__ groups, const SmallItem *__restrict__ items, const RegOp<R> *__restrict__ ops,
    const PhaseBits *__restrict__ phases, const SmallPass *__restrict__ passes, const int *__restrict__ slot_gate,
    const PauliWork *__restrict__ works, const PauliZ *__restrict__ zs, const int *__restrict__ pptr,
    const int *__restrict__ pgate, const double *__restrict__ obs, const R *__restrict__ coefs, double *terms,
    double *out) {
    __shared__ Cx<R> tp[1 << M];
    __shared__ Cx<R> tl[1 << M];
    __shared__ double red[kMaxSweepSlots][kSmallThreads<M> / 64];
    const SmallItem it = items[blockIdx.x];
    const SmallGroup g = groups[it.group];
    const u64 index = (u64)it.index;
    const R *fm = coefs + (g.coefs + index * (u64)(g.f_rows + g.s_rows)) * kCoefs;
    const unsigned warm = touch<kSmallThreads<M>>(ops + g.f_op, g.n_ops * (int)sizeof(RegOp<R>)) |
                          touch<kSmallThreads<M>>(fm, (g.f_rows + g.s_rows) * (int)(sizeof(R) * kCoefs));
    small_zero<R, M>(tp);
    arrived(warm);
    small_forward<R, M, true>(tp, ops + g.f_op, phases + g.f_phase, g.f_phases, fm);
    const double dot = small_pauli<R, M>(tp, works + g.work, g.n_works, zs, obs + g.obs + index * (u64)g.n_terms * 2,
                                         [&](unsigned l, const Cx<R> &a) { tl[swizzle(l)] = a; });
    const double s = block_sum_tile<kSmallThreads<M>>(dot, &red[0][0]);
    if (threadIdx.x == 0) out[g.value + index] = s;
    __syncthreads();
    double *tt = terms + g.terms + index * (u64)g.n_gates;
    small_back<R, M, true>(tp, tl, red, ops, phases, passes + g.pass, g.n_passes, slot_gate, tt,
                           fm + (u64)g.f_rows * kCoefs);
    // the last barrier of the sweep orders its terms before these reads
    double *grad = out + g.grad + index * (u64)g.n_params;
    for (int p = threadIdx.x; p < g.n_params; p += kSmallThreads<M>) {
        double sum = 0.;
        for (int j = pptr[g.param + p]; j < pptr[g.param + p + 1]; ++j) sum += tt[pgate[j]];
        grad[p] = sum;
    }
}

// ---- host ----------------------------------------------------------------------------------

// Planned passes of a whole state, appended to common tables.
template <class R>
struct SmallTables {
    std::vector<RegOp<R>> ops;
    std::vector<PhaseBits> phases;
    std::vector<SmallPass> passes;
    std::vector<int> slot_gate;
};

template <class R>
void plan_small(SmallTables<R> &t, const std::vector<RegGate> &gates, int m, GlobalPhases keep) {
    constexpr int RB = Log2<kSmallAmps>::v;
    for (const BuiltPass<R> &bp :
         build_passes<R>(gates, m, m, TileCfg<R>::Low, RB, m - RB - 6, 1 << 30, 1 << 30, 1 << 30, keep)) {
        SmallPass ps;
        ps.op_begin = (int)t.ops.size();
        ps.phase_begin = (int)t.phases.size();
        ps.n_phases = (int)bp.phases.size();
        ps.n_slots = (int)bp.slot_gate.size();
        ps.slot_begin = (int)t.slot_gate.size();
        t.ops.insert(t.ops.end(), bp.ops.begin(), bp.ops.end());
        t.phases.insert(t.phases.end(), bp.phases.begin(), bp.phases.end());
        for (int gi : bp.slot_gate) t.slot_gate.push_back(gates[gi].source);
        t.passes.push_back(ps);
    }
}

// The forward passes as one: phases whose ops count from the first one's.
template <class R>
void plan_small_forward(SmallTables<R> &t, const std::vector<RegGate> &gates, int m, GlobalPhases keep) {
    const size_t pass0 = t.passes.size(), op0 = t.ops.size();
    plan_small(t, gates, m, keep);
    for (size_t p = pass0; p < t.passes.size(); ++p)
        for (int k = 0; k < t.passes[p].n_phases; ++k)
            t.phases[t.passes[p].phase_begin + k].op_begin += t.passes[p].op_begin - (int)op0;
    t.passes.resize(pass0);
}

template <class R>
void plan_small_pauli(const std::vector<PauliGroup> &groups_in, const std::vector<u64> &xmask,
                      const std::vector<u64> &zmask, int m, std::vector<PauliWork> &works, std::vector<PauliZ> &zs) {
    std::vector<PauliGroup> groups(groups_in);
    for (PauliGroup &g : groups) g.xlocal = (unsigned)g.xmask;
    std::vector<int> bits;
    for (int b = 0; b < m; ++b) bits.push_back(b);
    plan_pauli_pass<R>(groups, 0, (int)groups.size(), zmask,
                       [&](int k) { return __builtin_popcountll(xmask[k] & zmask[k]); }, bits, (1 << m) / kSmallAmps,
                       works, zs);
}

// f(integral_constant M) for a workgroup of 2^m amplitudes.
template <class R, class F>
void for_bits(int m, F &&f) {
    switch (m) {
        case 9: f(std::integral_constant<int, 9>()); break;
        case 11: f(std::integral_constant<int, 11>()); break;
        case 12: f(std::integral_constant<int, 12>()); break;
        case 13:
            if constexpr (sizeof(R) == 4) f(std::integral_constant<int, 13>());
            break;
        default: raise_error("no workgroup of 2^%d amplitudes", m);
    }
}

}  // namespace

// Widths of 2^9 (one wave) and 2^11 (a wave on every SIMD), then one per lane: a wave more per
// workgroup costs no time while SIMDs of the compute unit are idle, padding on a busy chip does.
template <class R>
int small_bits(int n_lanes) {
    return n_lanes <= 9 ? 9 : n_lanes <= 11 ? 11 : n_lanes;
}
template int small_bits<float>(int);
template int small_bits<double>(int);

template <class R>
bool fits_workgroup(int n_lanes) {
    return use_register_tiles() && n_lanes <= kSmallMaxBits<R>;
}
template bool fits_workgroup<float>(int);
template bool fits_workgroup<double>(int);

template <class R>
bool fits_workgroup(int n_lanes, const std::vector<PauliGroup> &groups) {
    const u64 always = Unit<R>::W == 2 ? 1 : 0;   // as the general path counts them
    for (const PauliGroup &g : groups)
        if (__builtin_popcountll(g.xmask | always) > kPauliTileBits<R>) return false;
    return fits_workgroup<R>(n_lanes);
}
template bool fits_workgroup<float>(int, const std::vector<PauliGroup> &);
template bool fits_workgroup<double>(int, const std::vector<PauliGroup> &);

int small_max_gates() { return kResultDoubles; }

template <class R>
double small_expectation(Cx<R> *psi, Cx<R> *lam, int n_lanes, const std::vector<QueuedGate> &gates,
                         const std::vector<PauliGroup> &groups, const std::vector<PauliTerm> &terms) {
    const int m = small_bits<R>(n_lanes);
    SmallTables<R> t;
    plan_small_forward(
        t, merged_gates<R>((int)gates.size(), n_lanes, [&](int i) -> const QueuedGate & { return gates[i]; }), m,
        kGlobalPhase);
    t.ops.push_back(RegOp<R>());   // one more is read than there are
    std::vector<u64> xmask, zmask;
    std::vector<double> coefs;
    for (const PauliGroup &g : groups)
        for (int k = g.first; k < g.first + g.count; ++k) {
            QG_REQUIRE(k == (int)zmask.size(), "Pauli groups out of order");
            xmask.push_back(g.xmask);
            zmask.push_back(terms[k].zmask);
            coefs.push_back(terms[k].cre);
            coefs.push_back(terms[k].cim);
        }
    std::vector<PauliWork> works;
    std::vector<PauliZ> zs;
    plan_small_pauli<R>(groups, xmask, zmask, m, works, zs);
    TableLayout tab;
    const size_t o_ops = tab.add(t.ops), o_ph = tab.add(t.phases), o_w = tab.add(works), o_z = tab.add(zs),
                 o_c = tab.add(coefs);
    char *buf = static_cast<char *>(dev_alloc(tab.bytes()));
    double *value = result_buffer();
    hipStream_t s = stream();
    hipError_t e = hipSuccess;
    try {
        tab.upload(buf);
        for_bits<R>(m, [&](auto mc) {
            constexpr int M = decltype(mc)::value;
            hipLaunchKernelGGL((k_small_expect<R, M>), 1, kSmallThreads<M>, 0, s, psi, lam, n_lanes,
                               reinterpret_cast<const RegOp<R> *>(buf + o_ops), (int)t.ops.size(),
                               reinterpret_cast<const PhaseBits *>(buf + o_ph), (int)t.phases.size(),
                               reinterpret_cast<const PauliWork *>(buf + o_w), (int)works.size(),
                               reinterpret_cast<const PauliZ *>(buf + o_z),
                               reinterpret_cast<const double *>(buf + o_c), value);
        });
        QG_HIP(hipGetLastError());
        e = hipStreamSynchronize(s);
    } catch (...) {
        dev_free(buf, tab.bytes());
        throw;
    }
    dev_free(buf, tab.bytes());
    QG_HIP(e);
    table_buffer_done();
    return value[0];
}
template double small_expectation<float>(Cx<float> *, Cx<float> *, int, const std::vector<QueuedGate> &,
                                         const std::vector<PauliGroup> &, const std::vector<PauliTerm> &);
template double small_expectation<double>(Cx<double> *, Cx<double> *, int, const std::vector<QueuedGate> &,
                                          const std::vector<PauliGroup> &, const std::vector<PauliTerm> &);

template <class R>
void small_sweep(const Cx<R> *phi, const Cx<R> *lam, int n_lanes, const std::vector<SweepGate> &gates, double *out) {
    const int m = small_bits<R>(n_lanes);
    QG_REQUIRE((int)gates.size() <= small_max_gates(), "sweep in one workgroup: %d gates", (int)gates.size());
    for (size_t i = 0; i < gates.size(); ++i) out[i] = 0.;
    SmallTables<R> t;
    plan_small(t, sweep_gates(gates, n_lanes), m, kNoGlobalPhase);
    if (t.passes.empty()) return;
    t.ops.push_back(RegOp<R>());   // one more is read than there are
    TableLayout tab;
    const size_t o_ops = tab.add(t.ops), o_ph = tab.add(t.phases), o_ps = tab.add(t.passes), o_sg = tab.add(t.slot_gate);
    char *buf = static_cast<char *>(dev_alloc(tab.bytes()));
    double *terms = result_buffer();
    hipStream_t s = stream();
    hipError_t e = hipSuccess;
    try {
        tab.upload(buf);
        for_bits<R>(m, [&](auto mc) {
            constexpr int M = decltype(mc)::value;
            hipLaunchKernelGGL((k_small_sweep<R, M>), 1, kSmallThreads<M>, 0, s, phi, lam, n_lanes,
                               reinterpret_cast<const RegOp<R> *>(buf + o_ops), (int)t.ops.size(),
                               reinterpret_cast<const PhaseBits *>(buf + o_ph), (int)t.phases.size(),
                               reinterpret_cast<const SmallPass *>(buf + o_ps), (int)t.passes.size(),
                               reinterpret_cast<const int *>(buf + o_sg), terms);
        });
        QG_HIP(hipGetLastError());
        e = hipStreamSynchronize(s);
    } catch (...) {
        dev_free(buf, tab.bytes());
        throw;
    }
    dev_free(buf, tab.bytes());
    QG_HIP(e);
    table_buffer_done();
    for (int g : t.slot_gate) out[g] = terms[g];
}
template void small_sweep<float>(const Cx<float> *, const Cx<float> *, int, const std::vector<SweepGate> &, double *);
template void small_sweep<double>(const Cx<double> *, const Cx<double> *, int, const std::vector<SweepGate> &,
                                  double *);

// ---- batch ---------------------------------------------------------------------------------

SmallBatch::~SmallBatch() { dev_free_quiet(block_, bytes_); }

void SmallBatch::clear() {
    if (block_ != nullptr) dev_free(block_, bytes_);
    block_ = nullptr;
    launches_.clear();
    value_at_.clear();
    grad_at_.clear();
    passes_.clear();
    host_.clear();
}

template <class R>
void SmallBatch::build(const std::vector<SmallGroupIn> &in) {
    clear();
    if (in.empty()) return;
    SmallTables<R> t;
    std::vector<BRow<R>> rows;
    std::vector<SmallGroup> groups;
    std::vector<PauliWork> works;
    std::vector<PauliZ> zs;
    std::vector<int> pptr, pgate;
    std::vector<double> obs;
    size_t n_coefs = 0, n_terms = 0;
    n_params_ = n_out_ = n_items_ = 0;
    for (const SmallGroupIn &gi : in) {
        const int m = small_bits<R>(gi.n), n_gates = (int)gi.ops->size();
        SmallGroup g;
        g.n_params = gi.n_params;
        g.n_gates = n_gates;
        g.n_terms = (int)gi.zmask->size();
        std::vector<BRow<R>> fr, sr;
        g.f_op = (int)t.ops.size();
        g.f_phase = (int)t.phases.size();
        plan_small_forward(t, row_gates<R>(*gi.ops, gi.n, false, fr), m, kNoGlobalPhase);
        g.f_phases = (int)t.phases.size() - g.f_phase;
        g.pass = (int)t.passes.size();
        plan_small(t, row_gates<R>(*gi.ops, gi.n, true, sr), m, kNoGlobalPhase);
        g.n_passes = (int)t.passes.size() - g.pass;
        g.n_ops = (int)t.ops.size() - g.f_op;
        passes_.push_back(g.n_passes);
        g.f_rows = (int)fr.size();
        g.s_rows = (int)sr.size();
        g.f_row = (int)rows.size();
        rows.insert(rows.end(), fr.begin(), fr.end());
        g.s_row = (int)rows.size();
        rows.insert(rows.end(), sr.begin(), sr.end());
        g.work = (int)works.size();
        plan_small_pauli<R>(*gi.pgroups, *gi.xmask, *gi.zmask, m, works, zs);
        g.n_works = (int)works.size() - g.work;
        // parameter -> rotations (sweep order)
        g.param = (int)pptr.size();
        std::vector<std::vector<int>> of(gi.n_params);
        for (int i = n_gates - 1; i >= 0; --i)
            if ((*gi.ops)[i].kind == 1) of[(*gi.ops)[i].param].push_back(i);
        for (int p = 0; p < gi.n_params; ++p) {
            pptr.push_back((int)pgate.size());
            pgate.insert(pgate.end(), of[p].begin(), of[p].end());
        }
        pptr.push_back((int)pgate.size());
        const size_t ni = (size_t)gi.n_items;
        g.params = n_params_;
        n_params_ += ni * (size_t)gi.n_params;
        g.obs = obs.size();
        obs.insert(obs.end(), gi.coefs->begin(), gi.coefs->end());
        g.coefs = n_coefs;
        n_coefs += ni * (size_t)(g.f_rows + g.s_rows);
        g.terms = n_terms;
        n_terms += ni * (size_t)n_gates;
        g.value = n_out_;
        value_at_.push_back(n_out_);
        n_out_ += ni;
        g.grad = n_out_;
        grad_at_.push_back(n_out_);
        n_out_ += ni * (size_t)gi.n_params;
        n_items_ += ni;
        groups.push_back(g);
    }
    t.ops.push_back(RegOp<R>());   // one more is read than there are
    // items by workgroup width, the widest first, the longest circuits of a width first
    std::vector<int> order(in.size());
    for (size_t k = 0; k < order.size(); ++k) order[k] = (int)k;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
        const int ma = small_bits<R>(in[a].n), mb = small_bits<R>(in[b].n);
        return ma != mb ? ma > mb : in[a].ops->size() > in[b].ops->size();
    });
    std::vector<SmallItem> items;
    for (int k : order) {
        const int m = small_bits<R>(in[k].n);
        if (launches_.empty() || launches_.back().bits != m) launches_.push_back(Launch{m, items.size(), 0});
        launches_.back().count += (u64)in[k].n_items;
        for (int i = 0; i < in[k].n_items; ++i) items.push_back(SmallItem{k, i});
    }
    TableLayout tab;
    o_groups_ = tab.add(groups);
    o_items_ = tab.add(items);
    o_rows_ = tab.add(rows);
    o_ops_ = tab.add(t.ops);
    o_phases_ = tab.add(t.phases);
    o_passes_ = tab.add(t.passes);
    o_slots_ = tab.add(t.slot_gate);
    o_works_ = tab.add(works);
    o_zs_ = tab.add(zs);
    o_pptr_ = tab.add(pptr);
    o_pgate_ = tab.add(pgate);
    o_obs_ = tab.add(obs);
    size_t off = tab.bytes();
    auto carve = [&](size_t bytes) {
        off = (off + 255) & ~size_t(255);
        const size_t at = off;
        off += std::max<size_t>(bytes, 8);
        return at;
    };
    o_params_ = carve(sizeof(double) * n_params_);
    o_coefs_ = carve(sizeof(R) * kCoefs * n_coefs);
    o_terms_ = carve(sizeof(double) * n_terms);
    o_out_ = carve(sizeof(double) * n_out_);
    bytes_ = off;
    block_ = static_cast<char *>(dev_alloc(bytes_));
    host_.resize(n_out_);
    tab.upload(block_);
    QG_HIP(hipStreamSynchronize(stream()));   // the tables are host temporaries
    table_buffer_done();
}
template void SmallBatch::build<float>(const std::vector<SmallGroupIn> &);
template void SmallBatch::build<double>(const std::vector<SmallGroupIn> &);

void SmallBatch::upload(const std::vector<const std::vector<double> *> &params) {
    TableLayout tab;   // 256-byte alignment would leave gaps: one table
    std::vector<double> all;
    all.reserve(n_params_);
    for (const std::vector<double> *p : params) all.insert(all.end(), p->begin(), p->end());
    tab.add(all);
    tab.upload(block_ + o_params_);
    if (tab.bytes() > kTableBytes) QG_HIP(hipStreamSynchronize(stream()));   // `all` is a temporary
}

template <class R>
void SmallBatch::launch(hipStream_t s) const {
    const SmallGroup *groups = reinterpret_cast<const SmallGroup *>(block_ + o_groups_);
    const SmallItem *items = reinterpret_cast<const SmallItem *>(block_ + o_items_);
    R *coefs = reinterpret_cast<R *>(block_ + o_coefs_);
    hipLaunchKernelGGL((k_small_rows<R>), (unsigned)n_items_, 256, 0, s, groups, items,
                       reinterpret_cast<const BRow<R> *>(block_ + o_rows_),
                       reinterpret_cast<const double *>(block_ + o_params_), coefs);
    for (const Launch &l : launches_)
        for_bits<R>(l.bits, [&](auto mc) {
            constexpr int M = decltype(mc)::value;
            const u64 piece = launch_piece_items() / (u64)kSmallThreads<M>;
            for (u64 first = 0; first < l.count; first += piece)
                hipLaunchKernelGGL((k_small_batch<R, M>), (unsigned)std::min(piece, l.count - first), kSmallThreads<M>,
                                   0, s, groups, items + l.first + first,
                                   reinterpret_cast<const RegOp<R> *>(block_ + o_ops_),
                                   reinterpret_cast<const PhaseBits *>(block_ + o_phases_),
                                   reinterpret_cast<const SmallPass *>(block_ + o_passes_),
                                   reinterpret_cast<const int *>(block_ + o_slots_),
                                   reinterpret_cast<const PauliWork *>(block_ + o_works_),
                                   reinterpret_cast<const PauliZ *>(block_ + o_zs_),
                                   reinterpret_cast<const int *>(block_ + o_pptr_),
                                   reinterpret_cast<const int *>(block_ + o_pgate_),
                                   reinterpret_cast<const double *>(block_ + o_obs_), coefs,
                                   reinterpret_cast<double *>(block_ + o_terms_),
                                   reinterpret_cast<double *>(block_ + o_out_));
        });
    QG_HIP(hipGetLastError());
}
template void SmallBatch::launch<float>(hipStream_t) const;
template void SmallBatch::launch<double>(hipStream_t) const;

void SmallBatch::download() {
    QG_HIP(hipMemcpyAsync(host_.data(), block_ + o_out_, sizeof(double) * n_out_, hipMemcpyDeviceToHost, stream()));
}

}  // namespace qg
