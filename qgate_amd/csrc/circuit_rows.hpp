// Coefficient rows of a parameterised circuit's register gates: one row of kCoefs numbers per gate
// and item, computed on the device from each item's parameters. Shared by the batched tile passes
// (k_batch.hip) and the one-workgroup circuits (k_small.hip).
#pragma once

#include <cmath>
#include <cstring>
#include <vector>

#include "circuit.hpp"
#include "tile_reg.hpp"

namespace qg {

namespace {

template <class R>
struct BRow {           // one row of the table
    R c[8];             // fixed gates: the coefficients
    int kind;           // RegGate kind
    int pauli;          // rotations: 1 X, 2 Y, 3 Z; 0: fixed
    int param;
    int back;           // the inverse (sweep)
};

// Row `row` for an item with parameters `params`, in FP64 and rounded once, to out[0 .. kCoefs).
template <class R>
__device__ __forceinline__ void row_coefs(const BRow<R> &row, const double *__restrict__ params, R *out) {
    R c[kCoefs];
    for (int k = 0; k < kCoefs; ++k) c[k] = row.c[k];
    if (row.pauli != 0) {
        const double th = params[row.param];
        const double co = cos(0.5 * th), si = row.back ? -sin(0.5 * th) : sin(0.5 * th);
        if (row.kind == kGateY) {          // m00 = co, m01 = -si
            rotation_coefs(c, co, -si);
        } else if (row.kind == kGateX) {   // m00 = co, m01 = -i si
            rotation_coefs(c, co, si);
        } else if (row.kind == kGateDiag) {   // co - i si, co + i si and their ratio
            c[0] = (R)co;  c[1] = (R)-si;
            c[2] = (R)co;  c[3] = (R)si;
            c[4] = (R)cos(th);  c[5] = (R)(row.back ? -sin(th) : sin(th));
        } else {                           // controlled RX, RY: the whole matrix
            const double isx = row.pauli == 1 ? 1. : 0., isy = row.pauli == 2 ? 1. : 0.;
            c[0] = (R)co;  c[1] = R(0);
            c[2] = (R)(-si * isy);  c[3] = (R)(-si * isx);
            c[4] = (R)(si * isy);   c[5] = (R)(-si * isx);
            c[6] = (R)co;  c[7] = R(0);
        }
    }
    for (int k = 0; k < kCoefs; ++k) out[k] = c[k];
}

// The register gates of a circuit's structure, forward or (back) inverted in sweep order, and the
// row of each in the coefficient table. Rotations keep their form at every angle; fixed gates
// are split as in the single-circuit passes. RegGate::source is the gate of the structure.
template <class R>
std::vector<RegGate> row_gates(const std::vector<CircuitOp> &ops, int n_lanes, bool back,
                               std::vector<BRow<R>> &rows) {
    std::vector<RegGate> out;
    const int n = (int)ops.size();
    const std::vector<int> role = parity_roles(
        n, n_lanes, [&](int i) -> const CircuitOp & { return ops[i]; },
        [&](int i) { return ops[i].kind == 0 && ops[i].ctrl.size() == 1 && is_x(ops[i].mat); },
        [&](int i) {
            const CircuitOp &op = ops[i];
            return op.ctrl.empty() && (op.kind == 1 ? op.pauli == 3 : diag2(op.mat) && has_ratio(op.mat));
        });
    for (int k = 0; k < n; ++k) {
        const int i = back ? n - 1 - k : k;
        const CircuitOp &op = ops[i];
        if (role[i] == kDropped) continue;
        const size_t at = out.size();
        if (op.kind == 0) {
            append_fixed(out, back ? dagger(op.mat) : op.mat, op.ctrl, op.target, i);
            if (role[i] != kKept && out.size() > at) out.back().parity = role[i];
            continue;
        }
        RegGate g;
        g.kind = op.pauli == 3 ? kGateDiag : !op.ctrl.empty() ? kGateAny : op.pauli == 1 ? kGateX : kGateY;
        g.target = op.target;
        g.pauli = back ? op.pauli : 0;
        g.source = i;
        g.ctrl = op.ctrl;
        g.m = rotation(op.pauli, back ? -1. : 1.);   // its form; the angle is each item's own
        if (role[i] != kKept) g.parity = role[i];
        out.push_back(g);
    }
    rows.clear();
    for (const RegGate &g : out) {
        BRow<R> r;
        std::memset(&r, 0, sizeof(r));
        gate_coefs<R>(g, r.c);
        r.kind = g.kind;
        if (ops[g.source].kind == 1) {
            r.pauli = ops[g.source].pauli;
            r.param = ops[g.source].param;
        }
        r.back = back ? 1 : 0;
        rows.push_back(r);
    }
    return out;
}

}  // namespace

}  // namespace qg
