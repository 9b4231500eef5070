// dense_scan product-tree plans: one circuit (an engine) or many (a batch).
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "rie_kernels.hpp"

namespace rie {

// One dense_scan circuit of several chunks as the kernels see it.  Chunk k
// holds layers [k q, min(k q + q, L)) of the circuit, T_k their product.  Node
// k of the product tree is tree + k * node_doubles: a re plane of D * D
// doubles, then the im plane, both of the TRANSPOSED matrix (row c of the
// plane is column c of T).  Level j starts at node 2P - 2 (P >> j), the root is
// node 2P - 2.
struct DenseJob {
    const double *rec;     // records of the circuit's layers
    double *tree;          // (2P - 1) nodes
    double2 *vec_a;        // P * 2D: down-sweep vectors (ping); root seed [e0 | eta]
    double2 *vec_b;        // (pong)
    double2 *head;         // psi, lambda: 2D
    double *energy;
    double *grad;          // 2 n L values
    const double *scale;   // chain-rule factor for grad, or nullptr
    size_t node_doubles;   // 2 * D * D
    double field;
    int n;
    int L;
    int D;       // max(2^n, 16)
    int log_d;   // log2(D)
    int P;       // chunks: a power of two, at least 2
    int levels;  // log2(P)
    int q;       // layers per chunk
    int reserved;
};

struct DenseSpec {
    int n;
    int L;
    double field;
    const double *params;  // 2 n L values
    double *energy;
    double *grad;
    const double *scale;
};

// Device buffers, job tables and per-launch work tables of a set of dense
// circuits.  Kernels of one launch find their job by binary search over the
// launch's (job, first block) table.
class DensePlan {
  public:
    DensePlan() = default;
    ~DensePlan();
    DensePlan(const DensePlan &) = delete;
    DensePlan &operator=(const DensePlan &) = delete;

    // sharing: dense circuits evaluated together (a circuit's chunks depend on
    // it, see chunks_for), at least specs.size().
    void build(const std::vector<DenseSpec> &specs, size_t sharing);
    // Issue every launch on s.  The overrides (single-circuit plans only)
    // redirect the parameter / energy / gradient / scale pointers of the job.
    void run(hipStream_t s, bool want_grad, const double *params_override = nullptr,
             double *energy_override = nullptr, double *grad_override = nullptr,
             const double *scale_override = nullptr) const;
    size_t size() const { return specs_.size(); }
    size_t device_bytes() const { return arena_bytes_; }
    // Chunks of a circuit (1: the whole circuit is one chunk).
    static int chunks_for(int n, int L, size_t sharing);

  private:
    struct Launch {
        int level = 0;
        int blocks = 0;  // total blocks
        int count = 0;   // circuits in the launch
        size_t tab_off = 0;
    };
    struct Group {  // circuits of one qubit count
        int n;
        int first;
        int count;
    };
    std::vector<DenseSpec> specs_;
    std::vector<DenseJob> jobs_;       // several chunks, by qubit count
    std::vector<RegJob> flat_;         // one chunk, by qubit count, deepest first
    std::vector<Group> flat_groups_;
    std::vector<RecordJob> records_;   // every circuit
    int layers_ = 0;                   // records of one evaluation
    DenseJob *d_jobs_ = nullptr;
    RegJob *d_flat_ = nullptr;
    RegJob *d_flat_energy_ = nullptr;  // without gradients
    RecordJob *d_records_ = nullptr;
    int *d_layer_job_ = nullptr;
    int2 *d_tab_ = nullptr;
    void *arena_ = nullptr;
    size_t arena_bytes_ = 0;
    std::vector<std::pair<int, Launch>> leaves_;  // per qubit count
    std::vector<Launch> gemm_;
    Launch head_;
    std::vector<Launch> down_;
    std::vector<std::pair<int, Launch>> walks_;   // per qubit count
    void release();
};

}  // namespace rie
