// Circuits whose whole state fits one workgroup (k_small.hip).
#pragma once

#include <vector>

#include "circuit.hpp"
#include "kernels.hpp"

namespace qg {

// Whether a circuit of n lanes with these X masks goes to one workgroup. n: up to 13 lanes in
// complex64, 12 in complex128 (two states in LDS); a Pauli term with more X and Y factors than a
// tile of the general path has bits stays there, which refuses it.
template <class R>
bool fits_workgroup(int n_lanes);
template <class R>
bool fits_workgroup(int n_lanes, const std::vector<PauliGroup> &groups);

// psi = the gates on |0...0>, lam = H psi; returns Re<psi|lam>. Synchronises.
template <class R>
double small_expectation(Cx<R> *psi, Cx<R> *lam, int n_lanes, const std::vector<QueuedGate> &gates,
                         const std::vector<PauliGroup> &groups, const std::vector<PauliTerm> &terms);
// The adjoint sweep over phi and lam, which it leaves as they are: out[i] is the gradient term of
// gates[i] (rotations). Synchronises. At most small_max_gates() gates.
template <class R>
void small_sweep(const Cx<R> *phi, const Cx<R> *lam, int n_lanes, const std::vector<SweepGate> &gates, double *out);
int small_max_gates();

// The groups of a batch whose circuits each take one workgroup: values and gradients of all of
// their items in three launches.
struct SmallGroupIn {
    int n, n_params, n_items;
    const std::vector<CircuitOp> *ops;
    const std::vector<PauliGroup> *pgroups;
    const std::vector<u64> *xmask, *zmask;
    const std::vector<double> *coefs;        // per item: (re, im) per term
};
class SmallBatch {
  public:
    SmallBatch() = default;
    SmallBatch(const SmallBatch &) = delete;
    SmallBatch &operator=(const SmallBatch &) = delete;
    ~SmallBatch();
    void clear();
    template <class R>
    void build(const std::vector<SmallGroupIn> &groups);
    bool empty() const { return block_ == nullptr; }
    void upload(const std::vector<const std::vector<double> *> &params);   // one per group
    template <class R>
    void launch(hipStream_t s) const;
    // Results of group k, after finish(): value of item i, its gradient.
    void download();
    const double *values(int k) const { return host_.data() + value_at_[k]; }
    const double *grads(int k) const { return host_.data() + grad_at_[k]; }
    int sweep_passes(int k) const { return k < (int)passes_.size() ? passes_[k] : 0; }   // 0: not built

  private:
    struct Launch {          // one width of workgroup
        int bits;
        u64 first, count;    // items
    };
    std::vector<Launch> launches_;
    std::vector<size_t> value_at_, grad_at_;   // in the output array, per group
    std::vector<int> passes_;
    std::vector<double> host_;
    size_t n_items_ = 0, n_params_ = 0, n_out_ = 0;
    char *block_ = nullptr;
    size_t bytes_ = 0;
    size_t o_groups_ = 0, o_items_ = 0, o_rows_ = 0, o_ops_ = 0, o_phases_ = 0, o_passes_ = 0, o_slots_ = 0,
           o_works_ = 0, o_zs_ = 0, o_pptr_ = 0, o_pgate_ = 0, o_params_ = 0, o_obs_ = 0, o_coefs_ = 0, o_terms_ = 0,
           o_out_ = 0;
};
// Tile bits of the workgroup that a circuit of n lanes takes in a batch.
template <class R>
int small_bits(int n_lanes);

}  // namespace qg
