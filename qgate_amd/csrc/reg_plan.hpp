// Planning of register-resident tile passes (tile_reg.hpp), on the host: how a gate list
// becomes the ops, phases and passes that the kernels run. Shared by the single-circuit passes
// (k_tile.hip) and the batched ones (k_batch.hip).
#pragma once

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <type_traits>
#include <utility>
#include <vector>

#include "gate_matrix.hpp"
#include "qg_common.hpp"

namespace qg {

// ---- gates as the register passes apply them ----------------------------------------------
//
// Any 2x2 unitary is diag . RY . diag, and a diagonal factor is nearly free in a register pass
// wherever its lane is no register bit (one factor per thread), so an uncontrolled general gate
// becomes one real rotation, which takes a quarter of its multiplications.
enum : int {
    kGateDiag = 0,   // diag(m00, m11), controls allowed
    kGateY = 1,      // [[c, -s], [s, c]], no controls
    kGateX = 2,      // [[c, -i s], [-i s, c]], no controls
    kGateSwap = 3,   // X, with or without controls
    kGateAny = 4     // any other 2x2, controls allowed
};

struct RegGate {
    int kind = kGateAny;
    int target = 0;
    int pauli = 0;      // gradient generator (1 X, 2 Y, 3 Z) of a sweep's rotation, 0: none
    int source = 0;     // the gate of the caller's list that it came from
    int parity = -1;    // diagonal gates: it acts by target ^ this lane (no controls), -1: by the target
    std::vector<int> ctrl;
    GateMatrix m;
};

inline bool is_x(const GateMatrix &g) {
    return g.m[0][0] == 0. && g.m[1][1] == 0. && g.m[0][1] == 1. && g.m[1][0] == 1.;
}

inline bool diag2(const GateMatrix &g) { return g.m[0][1] == 0. && g.m[1][0] == 0.; }

// Far from a unitary matrix's entries, quotients of entries and squares of them can leave the range of a
// state's numbers where the entries themselves are within it: such gates take the general update.
inline bool moderate(double a) { return a > 1e-6 && a < 1e6; }

// [[c, -s], [s, c]] with real entries, exactly
inline bool is_y_rotation(const GateMatrix &g) {
    for (int r = 0; r < 2; ++r)
        for (int c = 0; c < 2; ++c)
            if (g.m[r][c].imag() != 0.) return false;
    return g.m[0][0] == g.m[1][1] && g.m[0][1] == -g.m[1][0] &&
           moderate(std::max(std::abs(g.m[0][0].real()), std::abs(g.m[0][1].real())));
}

// [[c, -i s], [-i s, c]], exactly
inline bool is_x_rotation(const GateMatrix &g) {
    return g.m[0][0].imag() == 0. && g.m[1][1].imag() == 0. && g.m[0][1].real() == 0. && g.m[1][0].real() == 0. &&
           g.m[0][0] == g.m[1][1] && g.m[0][1] == g.m[1][0] &&
           moderate(std::max(std::abs(g.m[0][0].real()), std::abs(g.m[0][1].imag())));
}

// A product of gates, rounded to FP64 where a register gate is made of it: T is long double for
// complex128 states (rounded at every product, a run of 4000 gates was off by 13 2^-53, now 0.4), double
// for complex64 ones.
template <class T>
struct Product {
    std::complex<T> m[2][2];
};
template <class R>
using ProductOf = typename std::conditional<sizeof(R) == 8, long double, double>::type;

template <class A, class T>
std::complex<T> times(const std::complex<A> &a, const std::complex<T> &b) {   // (no check for infinities)
    return std::complex<T>(a.real() * b.real() - a.imag() * b.imag(), a.real() * b.imag() + a.imag() * b.real());
}
template <class T>
std::complex<double> rounded(const std::complex<T> &v) {
    return std::complex<double>((double)v.real(), (double)v.imag());
}
template <class T>
GateMatrix rounded(const Product<T> &w) {
    GateMatrix g;
    for (int r = 0; r < 2; ++r)
        for (int c = 0; c < 2; ++c) g.m[r][c] = rounded(w.m[r][c]);
    return g;
}
template <class T>
void widen(const GateMatrix &g, Product<T> &w) {
    for (int r = 0; r < 2; ++r)
        for (int c = 0; c < 2; ++c) w.m[r][c] = std::complex<T>(g.m[r][c]);
}
template <class T>
bool diag2(const Product<T> &w) {
    return w.m[0][1] == T(0) && w.m[1][0] == T(0);
}
// a <- b a, in place: copies of extended values cost more than their products
template <class T>
void multiply(const GateMatrix &b, Product<T> &a) {
    typedef std::complex<T> C;
    if (diag2(a)) {   // what a split has left
        const C d0 = a.m[0][0], d1 = a.m[1][1];
        for (int r = 0; r < 2; ++r) {
            a.m[r][0] = times(b.m[r][0], d0);
            a.m[r][1] = times(b.m[r][1], d1);
        }
        return;
    }
    const bool db = diag2(b);
    for (int c = 0; c < 2; ++c) {
        const C x = a.m[0][c], y = a.m[1][c];
        a.m[0][c] = times(b.m[0][0], x);
        a.m[1][c] = times(b.m[1][1], y);
        if (db) continue;
        a.m[0][c] += times(b.m[0][1], y);
        a.m[1][c] += times(b.m[1][0], x);
    }
}

// U = diag(a0, a1) RY diag(1, b) for a unitary U (to FP64 rounding); false for any other. In
// extended precision and rounded once, so that the factors' moduli are as close to 1 as those of
// rounded sines and cosines.
template <class T>
bool split_unitary(const Product<T> &u, std::complex<T> &a0, std::complex<T> &a1, std::complex<T> &b,
                   GateMatrix &ry) {
    typedef std::complex<long double> cl;
    const cl m00 = cl(u.m[0][0]), m01 = cl(u.m[0][1]), m10 = cl(u.m[1][0]), m11 = cl(u.m[1][1]);
    const long double tol = 4e-15L;
    if (!(std::abs(std::norm(m00) + std::norm(m01) - 1.L) < tol &&
          std::abs(std::norm(m10) + std::norm(m11) - 1.L) < tol &&
          std::norm(m00 * std::conj(m10) + m01 * std::conj(m11)) < tol * tol))
        return false;
    // (moduli at most 1 and squared without harm: no std::abs, whose hypot guards against more)
    auto modulus = [](const cl &v) { return std::sqrt(std::norm(v)); };
    const long double r0 = modulus(m00), r1 = modulus(m10), r = std::sqrt(r0 * r0 + r1 * r1);
    auto phase = [&](const cl &v) {
        const long double n = modulus(v);
        return n > 0.L ? v / n : cl(1.L);
    };
    const cl p0 = phase(m00), p1 = phase(m10);
    const cl pb = r0 >= r1 ? phase(m11) * std::conj(p1) : -phase(m01) * std::conj(p0);
    a0 = std::complex<T>((T)p0.real(), (T)p0.imag());
    a1 = std::complex<T>((T)p1.real(), (T)p1.imag());
    b = std::complex<T>((T)pb.real(), (T)pb.imag());
    const double c = (double)(r0 / r), s = (double)(r1 / r);
    ry.m[0][0] = c;
    ry.m[0][1] = -s;
    ry.m[1][0] = s;
    ry.m[1][1] = c;
    return true;
}

// Whether a diagonal gate can be applied as m00 and the ratio m11 / m00.
inline bool has_ratio(const GateMatrix &g) {
    const double b = std::abs(g.m[1][1]);
    return moderate(std::abs(g.m[0][0])) && (b == 0. || moderate(b));
}

inline bool trivial_diag(std::complex<double> d0, std::complex<double> d1) { return d0 == 1. && d1 == 1.; }

inline void append_diag(std::vector<RegGate> &out, std::complex<double> d0, std::complex<double> d1, int target,
                        int source) {
    if (trivial_diag(d0, d1)) return;
    RegGate g;
    g.kind = kGateDiag;
    g.target = target;
    g.source = source;
    g.m.m[0][0] = d0;
    g.m.m[0][1] = g.m.m[1][0] = 0.;
    g.m.m[1][1] = d1;
    out.push_back(std::move(g));
}

// CX . D . CX with D diagonal on the target (an exp(-i a Z Z / 2), for instance) is D by the parity of
// control and target: one diagonal gate and no register moves. role[i] is then kDropped for the CX
// gates and the control's lane for D, kKept for all other gates. A triple is taken if no other gate on
// its two lanes lies between. gate(i): ctrl, target; is_cx(i): X with one control; is_diag(i): a
// diagonal gate without controls (for every parameter). (13 qubits, 6 layers of ZZ and X rotations: 307 gates become 163.)
constexpr int kKept = -1, kDropped = -2;
template <class GateAt, class IsCx, class IsDiag>
std::vector<int> parity_roles(int n_gates, int n_lanes, GateAt gate, IsCx is_cx, IsDiag is_diag) {
    std::vector<int> role(n_gates, kKept), last(n_lanes, -1), before(n_gates, -1);   // before: on the target
    for (int i = 0; i < n_gates; ++i) {
        const int t = gate(i).target;
        const std::vector<int> &ctrl = gate(i).ctrl;
        if (is_cx(i)) {
            const int c = ctrl[0], d = last[t], x = d >= 0 ? before[d] : -1;
            if (x >= 0 && role[d] == kKept && role[x] == kKept && is_diag(d) && is_cx(x) && last[c] == x &&
                gate(x).target == t && gate(x).ctrl[0] == c) {
                role[x] = role[i] = kDropped;
                role[d] = c;
                last[c] = d;
                continue;
            }
        }
        before[i] = last[t];
        last[t] = i;
        for (int c : ctrl) last[c] = i;
    }
    return role;
}

// Appends the register gates of one fixed gate (no parameter), in the order they apply. exact: m before
// it was rounded, if it is a product.
template <class T = double>
void append_fixed(std::vector<RegGate> &out, const GateMatrix &m, const std::vector<int> &ctrl, int target,
                  int source, const Product<T> *exact = nullptr) {
    RegGate g;
    g.target = target;
    g.source = source;
    g.ctrl = ctrl;
    g.m = m;
    if (diag2(m) && has_ratio(m)) {
        g.kind = kGateDiag;
        if (!trivial_diag(m.m[0][0], m.m[1][1])) out.push_back(std::move(g));
        return;
    }
    if (is_x(m)) {
        g.kind = kGateSwap;
        out.push_back(std::move(g));
        return;
    }
    if (ctrl.empty()) {
        if (is_y_rotation(m) || is_x_rotation(m)) {
            g.kind = is_y_rotation(m) ? kGateY : kGateX;
            out.push_back(g);
            return;
        }
        Product<T> u;
        if (exact == nullptr) {
            widen(m, u);
            exact = &u;
        }
        std::complex<T> a0, a1, b;
        if (split_unitary(*exact, a0, a1, b, g.m)) {
            append_diag(out, 1., rounded(b), target, source);
            g.kind = kGateY;
            out.push_back(g);
            append_diag(out, rounded(a0), rounded(a1), target, source);
            return;
        }
    }
    g.kind = kGateAny;
    out.push_back(std::move(g));
}

// The register gates of a gate list whose matrices are all known. The uncontrolled gates of a lane
// between controlled ones multiply into one; of its split diag . RY . diag the last diagonal waits for
// the lane's next gate where what comes between acts diagonally on the lane.
// gate(i) has m, ctrl and target; R: the precision of the state.
template <class R, class GateAt>
std::vector<RegGate> merged_gates(int n_gates, int n_lanes, GateAt gate) {
    std::vector<RegGate> out;
    out.reserve((size_t)n_gates * 2);
    typedef ProductOf<R> T;
    std::vector<Product<T>> run(n_lanes);
    std::vector<int> last(n_lanes, -1);   // source of the lane's run, -1: none
    const std::vector<int> role = parity_roles(
        n_gates, n_lanes, gate, [&](int i) { return gate(i).ctrl.size() == 1 && is_x(gate(i).m); },
        [&](int i) { return gate(i).ctrl.empty() && diag2(gate(i).m) && has_ratio(gate(i).m); });
    auto emit = [&](int lane, bool keep_diagonal) {
        if (last[lane] < 0) return;
        Product<T> &w = run[lane];
        if (keep_diagonal && diag2(w)) return;
        const GateMatrix m = rounded(w);
        std::complex<T> a0, a1, b;
        GateMatrix ry;
        if (keep_diagonal && !is_x(m) && !is_y_rotation(m) && !is_x_rotation(m) && split_unitary(w, a0, a1, b, ry)) {
            append_diag(out, 1., rounded(b), lane, last[lane]);
            append_fixed(out, ry, {}, lane, last[lane]);
            w.m[0][0] = a0;
            w.m[0][1] = w.m[1][0] = T(0);
            w.m[1][1] = a1;
            return;
        }
        append_fixed(out, m, {}, lane, last[lane], &w);
        last[lane] = -1;
    };
    for (int i = 0; i < n_gates; ++i) {
        const auto &g = gate(i);
        if (role[i] == kDropped) continue;
        if (role[i] != kKept) {
            emit(role[i], true);
            emit(g.target, true);
            const size_t at = out.size();
            append_fixed(out, g.m, {}, g.target, i);
            if (out.size() > at) out.back().parity = role[i];
            continue;
        }
        if (g.ctrl.empty()) {
            if (last[g.target] < 0)
                widen(g.m, run[g.target]);
            else
                multiply(g.m, run[g.target]);
            last[g.target] = i;
            continue;
        }
        for (int c : g.ctrl) emit(c, true);
        emit(g.target, diag2(g.m));
        append_fixed(out, g.m, g.ctrl, g.target, i);
    }
    for (int l = 0; l < n_lanes; ++l) emit(l, false);
    return out;
}

// ---- passes and phases ----------------------------------------------------------------------

// Bit layout of one phase: local tile bits that are register, lane and wave bits.
struct PhasePlan {
    std::vector<int> regs, lanes, waves;
    std::vector<int> order;    // gates, in the order they apply
};

struct PassBits {
    std::vector<int> bits;     // state bits of the tile, ascending
    int low = 0;               // bits[j] == j for j < low
    std::vector<int> gates;    // gates, in an order they may apply in
};

// What the planner needs of a gate: its lanes, whether it acts diagonally on the target.
struct PlanGate {
    int target;
    const std::vector<int> *ctrl;
    bool diag;
    int weight;    // ops it may take
    int slots;     // gradient slots
    int parity;    // second lane of a parity gate, -1: none
};

// Lanes held by the gates left out of a scan: two gates commute when on every lane they share
// both act diagonally there (a control, or the target of a diagonal gate).
class HeldLanes {
  public:
    explicit HeldLanes(int n) : held_(n, 0) {}
    bool conflicts(const PlanGate &g) const {
        if (g.diag ? held_[g.target] == 2 : held_[g.target] != 0) return true;
        for (int c : *g.ctrl)
            if (held_[c] == 2) return true;
        return g.parity >= 0 && held_[g.parity] == 2;
    }
    void hold(const PlanGate &g) {
        put(g.target, g.diag ? 1 : 2);
        for (int c : *g.ctrl) put(c, 1);
        if (g.parity >= 0) put(g.parity, 1);
    }
    bool all() const { return full_ == (int)held_.size(); }

  private:
    void put(int lane, char v) {
        if (held_[lane] < 2 && v == 2) ++full_;
        held_[lane] = std::max(held_[lane], v);
    }
    std::vector<char> held_;
    int full_ = 0;
};

constexpr int kLookahead = 256;   // gates a scan may leave out

// The next pass over the gates not yet done: every gate that commutes with the ones left out
// before it and whose target is a tile bit, can become one, or needs none (diagonal), up to
// max_weight and max_slots. Marks them done. (A pass of consecutive gates only: a 2000-gate
// random circuit on 30 qubits took 120 passes instead of 75.)
inline PassBits next_pass(const std::vector<PlanGate> &g, std::vector<char> &done, int first, int n, int m, int low,
                          int max_weight, int max_slots) {
    PassBits p;
    std::vector<char> in(n, 0);
    int n_bits = 0, weight = 0, slots = 0, left = 0;
    for (int b = 0; b < low; ++b) in[b] = 1, ++n_bits;
    HeldLanes held(n);
    for (int i = first; i < (int)g.size(); ++i) {
        if (done[i]) continue;
        const PlanGate &q = g[i];
        const bool fits = q.diag || in[q.target] || n_bits < m;
        if (fits && weight + q.weight <= max_weight && slots + q.slots <= max_slots && !held.conflicts(q)) {
            if (!q.diag && !in[q.target]) in[q.target] = 1, ++n_bits;
            weight += q.weight;
            slots += q.slots;
            done[i] = 1;
            p.gates.push_back(i);
            continue;
        }
        held.hold(q);
        if (++left >= kLookahead || held.all()) break;
    }
    for (int b = 0; b < n && n_bits < m; ++b)   // a full tile: the lowest free bits
        if (!in[b]) in[b] = 1, ++n_bits;
    for (int b = 0; b < n; ++b)
        if (in[b]) p.bits.push_back(b);
    while (p.low < (int)p.bits.size() && p.bits[p.low] == p.low) ++p.low;
    return p;
}

// Rotations are applied up to a factor of at most sqrt(2), collected per phase; a phase takes
// at most this many of them (2^8 in the amplitudes, 2^16 in a gradient term).
constexpr int kMaxScaled = 16;

// The phases of a pass: each takes every gate that commutes with the ones it leaves out and
// whose non-diagonal target is one of its rb register bits or can become one; then each diagonal
// gate moves, between the pair gates on its lanes before and after it, to a phase where none of
// its lanes is a register bit (there it is one factor per thread instead of an update of the
// registers), if possible one that already has such factors. A parity gate stays in a phase where
// neither of its lanes becomes a register bit, so that it is always such a factor.
inline std::vector<PhasePlan> plan_phases(const std::vector<PlanGate> &g, const std::vector<int> &gates,
                                          const int *local, int n, int m, int rb, int wb) {
    std::vector<PhasePlan> out;
    std::vector<unsigned> regs;              // register bits of each phase
    std::vector<char> done(gates.size(), 0);
    size_t first = 0;
    while (first < gates.size()) {
        PhasePlan P;
        unsigned in = 0, out_of = 0;   // register bits, and bits that may not become ones
        HeldLanes held(n);
        int pairs = 0, free_regs = rb;
        for (size_t k = first; k < gates.size(); ++k) {
            if (done[k]) continue;
            const PlanGate &q = g[gates[k]];
            const unsigned bit = q.diag ? 0u : 1u << local[q.target];
            bool fits = q.diag || (pairs < kMaxScaled && ((in & bit) || (free_regs > 0 && !(out_of & bit))));
            unsigned lanes = 0;
            if (q.parity >= 0) {
                for (int l : {q.target, q.parity}) lanes |= local[l] >= 0 ? 1u << local[l] : 0u;
                fits = !(in & lanes) && m - __builtin_popcount(in | out_of | lanes) >= free_regs;
            }
            if (fits && !held.conflicts(q)) {
                out_of |= lanes;
                if (!q.diag) {
                    if (!(in & bit)) --free_regs;
                    in |= bit;
                    ++pairs;
                }
                P.order.push_back(gates[k]);
                done[k] = 1;
                continue;
            }
            held.hold(q);
            if (held.all()) break;
        }
        while (first < gates.size() && done[first]) ++first;
        // pad with the highest free bits, so that the lane bits are the lowest ones
        for (int b = m - 1; free_regs > 0 && b >= 0; --b)
            if (!(((in | out_of) >> b) & 1)) in |= 1u << b, --free_regs;
        for (int b = 0; b < m; ++b)
            ((in >> b) & 1 ? P.regs : (int)P.lanes.size() < 6 ? P.lanes : P.waves).push_back(b);
        if ((int)P.waves.size() != wb) raise_error("tile layout does not match the workgroup");
        regs.push_back(in);
        out.push_back(std::move(P));
    }
    // diagonal gates: position gp is before pair gate gp (np: after the last); lo and hi: right
    // after the last pair gate on one of its lanes before it, right before the first one after it
    struct Diag {
        int gate, lo, hi, at, phase;
    };
    std::vector<int> pairs, phase_of;
    std::vector<Diag> diags;
    std::vector<int> seen(n, 0);   // position after the last pair gate on a lane
    for (size_t ph = 0; ph < out.size(); ++ph)
        for (int gi : out[ph].order) {
            if (g[gi].diag) {
                int lo = seen[g[gi].target];
                for (int c : *g[gi].ctrl) lo = std::max(lo, seen[c]);
                diags.push_back(Diag{gi, lo, (int)pairs.size(), 0, (int)ph});
            } else {
                pairs.push_back(gi);
                phase_of.push_back((int)ph);
                seen[g[gi].target] = (int)pairs.size();
            }
        }
    const int np = (int)pairs.size(), n_ph = (int)out.size();
    if (np == 0 || diags.empty()) return out;
    std::fill(seen.begin(), seen.end(), np);   // position of the next pair gate on a lane
    for (int d = (int)diags.size() - 1, k = np; d >= 0; --d) {
        Diag &q = diags[d];
        for (; k > q.hi; --k) seen[g[pairs[k - 1]].target] = k - 1;
        if (g[q.gate].parity >= 0) {   // stays where it is
            q.at = q.hi;
            continue;
        }
        q.hi = seen[g[q.gate].target];
        for (int c : *g[q.gate].ctrl) q.hi = std::min(q.hi, seen[c]);
    }
    std::vector<char> has_factor(n_ph, 0);
    std::vector<int> count(np + 2, 0);
    for (Diag &d : diags) {
        const PlanGate &q = g[d.gate];
        if (q.parity >= 0) {
            has_factor[d.phase] = 1;
            ++count[d.at + 1];
            continue;
        }
        const auto bit = [&](int lane) { return local[lane] >= 0 ? 1u << local[lane] : 0u; };
        unsigned mask = bit(q.target);
        for (int c : *q.ctrl) mask |= bit(c);
        // phases it may run in: any from that of the pair gate before position lo to that of the
        // one after position hi
        const int ph_lo = d.lo == 0 ? 0 : phase_of[d.lo - 1], ph_hi = d.hi == np ? n_ph - 1 : phase_of[d.hi];
        auto cost = [&](int ph) {
            const unsigned on = mask & regs[ph];
            return on != 0 ? 4 - ((on & (on - 1)) != 0) : has_factor[ph] ? 0 : 1;
        };
        d.phase = ph_lo;
        for (int ph = ph_lo + 1; ph <= ph_hi; ++ph)
            if (cost(ph) < cost(d.phase)) d.phase = ph;
        if (cost(d.phase) <= 1) has_factor[d.phase] = 1;
        // the last position within [lo, hi] that still belongs to that phase
        d.at = (int)(std::upper_bound(phase_of.begin() + d.lo, phase_of.begin() + d.hi, d.phase) - phase_of.begin());
        ++count[d.at + 1];
    }
    for (int gp = 0; gp <= np; ++gp) count[gp + 1] += count[gp];
    std::vector<int> by(diags.size()), next(count);   // diagonal gates by position
    for (size_t d = 0; d < diags.size(); ++d) by[next[diags[d].at]++] = (int)d;
    for (PhasePlan &P : out) P.order.clear();
    for (int gp = 0; gp <= np; ++gp) {
        for (int k = count[gp]; k < count[gp + 1]; ++k) out[diags[by[k]].phase].order.push_back(diags[by[k]].gate);
        if (gp < np) out[phase_of[gp]].order.push_back(pairs[gp]);
    }
    return out;
}

}  // namespace qg
