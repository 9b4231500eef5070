// Batched evaluation of many independent ring-Ising circuits of uneven qubit
// and layer counts, with an autotuner and HIP-graph-captured optimizer steps.
//
// Circuits with n <= dense_max_qubits take the dense_scan product tree
// (rie_dense.hip, one grouped FP64-MFMA GEMM launch per tree level and tile
// class for all of them).  The others take the whole-circuit kernels: up to
// 13 qubits one launch per qubit count with every state in registers
// (rie_regcircuit.hip), one workgroup per circuit, deepest first; 14 qubits a
// forward launch of the same kind and a persistent adjoint launch whose
// workgroups take circuits from a longest-first (LPT) schedule built on the
// host.  The launches are spread over
// four streams (branches of one graph when captured), so the tail of one
// qubit count's deep circuits overlaps the others' work.  Parameters, energies
// and gradients of all circuits are packed in device arrays owned by the
// batch: circuit i's 2 n_i L_i parameters start at offset[i], in the
// reference's per-circuit layout (l n + w) 2 + {0, 1}
// (cpp/ising_cuda_structured_adjoint_modes.inc:73-77).
//
// The reference evaluates one circuit per call (RingIsingCudaBackend::
// energy_and_grad, cpp/ising_cuda_backend.cu:429-442) and picks its kernel
// shapes from fixed qubit-count thresholds (structured_register_threads_per_
// block, cpp/ising_cuda_rotation_kernels.cu:562-575; the chunk planner,
// cpp/ising_cuda_structured_adjoint_modes.inc:18-71).  Here the autotuner
// measures the candidates on the batch itself.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <functional>
#include <memory>
#include <queue>
#include <sstream>
#include <string>
#include <vector>

#include "rie.h"
#include "rie_dense.hpp"
#include "rie_engine_internal.hpp"
#include "rie_kernels.hpp"

namespace rie {

namespace {

constexpr int kMaxN = kBatchMaxQubits;
constexpr size_t kStateAmps = (size_t)1 << kMaxN;  // of a 14-qubit circuit

// An evaluation holds the layers' records (up to 1 KB each) and 256 KB for every
// 14-qubit circuit.  Large batches run in slices that use that memory in turn.  A
// slice ends at a gigabyte once it has sixteen circuits for each CU, enough
// for the tail between two slices not to count (8192 circuits of 14 qubits x 2
// layers in three slices 12.1 ms, in one 11.9; 260 circuits of 4 qubits x 8192
// layers, cut at a gigabyte too, would take 18.6 ms instead of 11.3), and in
// any case at a quarter of the free device memory (at least a quarter gigabyte).
constexpr size_t kSliceBytes = (size_t)1 << 30;
constexpr int kSliceCircuitsPerCu = 16;

}  // namespace

struct Batch {
    Batch(size_t count, const int *nq, const int *nl, const double *fields, int dense_max_qubits);
    ~Batch();
    Batch(const Batch &) = delete;
    Batch &operator=(const Batch &) = delete;

    // problem
    size_t count = 0;
    std::vector<int> n;
    std::vector<int> L;
    std::vector<double> h;
    std::vector<char> dense_flag;
    std::vector<size_t> poff;  // count + 1 parameter offsets
    size_t total = 0;
    int dense_max = 8;    // the caller's bound: n <= dense_max may take dense_scan
    int dense_split = 8;  // the split in force: n <= dense_split takes dense_scan
    bool tune_split = true;  // the autotuner chooses dense_split in [0, dense_max]

    // device
    int device = 0;
    int num_cus = 0;
    hipStream_t s_own = nullptr;
    static constexpr int kAux = 3;  // streams beside the caller's
    hipStream_t s_aux[kAux] = {};
    hipEvent_t ev_fork = nullptr;
    hipEvent_t ev_join[kAux] = {};
    hipEvent_t ev_t0 = nullptr;
    hipEvent_t ev_t1 = nullptr;
    double *d_params = nullptr;
    double *d_grad = nullptr;
    double *d_energy = nullptr;
    double *d_m = nullptr;
    double *d_v = nullptr;
    int *d_step = nullptr;
    double *d_history = nullptr;
    size_t history_cap = 0;

    // structured part
    std::vector<int> sids;
    // up to kRegMaxQubits: one launch per qubit count, states in registers
    struct RegGroup {
        int n;
        int first;  // in d_reg_g / d_reg_e
        int count;
    };
    // circuits evaluated together: their records and states share d_rec and
    // d_psi with the other slices'
    struct Slice {
        int first_layer = 0;  // in d_layer_job
        int layers = 0;
        int g_first = 0;      // in d_jobs_g / d_jobs_e
        int g_count = 0;
        int grid = 0;         // workgroups of the 14-qubit adjoint launch
        int begin_off = 0;    // its schedule in d_wg_begin
        std::vector<RegGroup> groups;  // largest n first
    };
    std::vector<Slice> slices;
    std::vector<RegJob> reg_jobs;       // with gradients, grouped, deepest first
    std::vector<RecordJob> reg_rec;     // indexed like reg_jobs
    std::vector<RecordJob> rec_jobs;    // every structured circuit
    std::vector<int> reg_of;            // circuit -> reg_jobs index, or -1
    RegJob *d_reg_g = nullptr;
    RegJob *d_reg_e = nullptr;
    RecordJob *d_rec_jobs = nullptr;
    int *d_layer_job = nullptr;
    double *d_rec = nullptr;
    // 14 qubits
    std::vector<int> gid_of;         // circuit -> jobs_g index, or -1
    std::vector<Reg14Job> jobs_g;    // with gradients
    std::vector<RecordJob> jobs_rec; // indexed like jobs_g
    Reg14Job *d_jobs_g = nullptr;
    Reg14Job *d_jobs_e = nullptr;  // energy only
    double2 *d_psi = nullptr;      // forward results of the 14-qubit circuits
    int *d_order = nullptr;
    int *d_wg_begin = nullptr;
    double2 *d_scratch = nullptr;
    int grid = 0;  // the slices' largest
    int threads = 512;  // reported only, like chunk_by_n and dense_tile below:
                        // the kernels have one shape per qubit count
    int grid_limit = 0;  // 0: every CU
    int chunk_by_n[kMaxN + 1];
    bool measured = false;

    // dense part
    std::vector<int> dids;
    DensePlan dense;
    int dense_tile = 64;
    std::vector<std::unique_ptr<DensePlan>> dense_single;

    // graphs
    hipGraphExec_t graph_exec = nullptr;
    int graph_kind = -1;  // 0 energy, 1 energy+grad, 2 GD step, 3 Adam step
    double graph_lr = 0.0;
    int graph_capacity = 0;
    bool use_graph = false;

    std::string report = "{}";

    void build_structured();
    void build_register_jobs();
    void build_dense();
    void repartition(int split);
    void release_structured();
    void invalidate_graph();
    void issue_eval(hipStream_t s, bool want_grad);
    void issue_slice(hipStream_t s, bool want_grad, const Slice &sl, bool with_dense);
    void issue_step(hipStream_t s, int optimizer, double lr, int capacity);
    void launch_graph(int kind, double lr, int capacity, hipStream_t s);
    void run(hipStream_t s, bool want_grad);
    void run_per_circuit(hipStream_t s, bool want_grad);
    void optimize(int optimizer, double lr, size_t steps, bool graph, double *history_out,
                  hipStream_t s);
    void autotune(size_t repeats);
    double time_ms(size_t repeats, const std::function<void(hipStream_t)> &fn);
    void ensure_history(size_t entries);
    void ensure_adam();
    std::string config_json() const;
    // whether anything runs beside the persistent launch
    bool parts_beside() const { return !dids.empty() || !reg_jobs.empty(); }
};

Batch::Batch(size_t count_, const int *nq, const int *nl, const double *fields, int dense_max_qubits)
    : count(count_), dense_max(dense_max_qubits), dense_split(dense_max_qubits) {
    if (count == 0) {
        fail(RIE_INVALID_ARGUMENT, "a batch needs at least one circuit.");
    }
    if (nq == nullptr || nl == nullptr || fields == nullptr) {
        fail(RIE_INVALID_ARGUMENT, "null pointer argument.");
    }
    if (dense_max_qubits < 0 || dense_max_qubits > 8) {
        fail(RIE_INVALID_ARGUMENT, "dense_max_qubits must be in [0, 8].");
    }
    poff.assign(count + 1, 0);
    for (size_t i = 0; i < count; ++i) {
        if (nq[i] < 2 || nq[i] > kMaxN) {
            fail(RIE_INVALID_ARGUMENT, "batched circuits need 2 <= num_qubits <= 14.");
        }
        if (nl[i] < 1 || nl[i] > 65536) {
            fail(RIE_INVALID_ARGUMENT, "batched circuits need 1 <= layers <= 65536.");
        }
        if (!std::isfinite(fields[i])) {
            fail(RIE_INVALID_ARGUMENT, "field must be finite.");
        }
        n.push_back(nq[i]);
        L.push_back(nl[i]);
        h.push_back(fields[i]);
        dense_flag.push_back(nq[i] <= dense_max_qubits ? 1 : 0);
        poff[i + 1] = poff[i] + (size_t)2 * nq[i] * nl[i];
    }
    total = poff[count];
    if (total / 2 > 0x7fffffffULL) {
        fail(RIE_INVALID_ARGUMENT, "batch has too many parameters.");
    }
    for (int q = 0; q <= kMaxN; ++q) {
        chunk_by_n[q] = 3;
    }
    check(hipGetDevice(&device), "hipGetDevice");
    hipDeviceProp_t prop;
    check(hipGetDeviceProperties(&prop, device), "hipGetDeviceProperties");
    num_cus = prop.multiProcessorCount;
    check(hipStreamCreateWithFlags(&s_own, hipStreamNonBlocking), "hipStreamCreate");
    check(hipEventCreateWithFlags(&ev_fork, hipEventDisableTiming), "hipEventCreate");
    for (int a = 0; a < kAux; ++a) {
        check(hipStreamCreateWithFlags(&s_aux[a], hipStreamNonBlocking), "hipStreamCreate");
        check(hipEventCreateWithFlags(&ev_join[a], hipEventDisableTiming), "hipEventCreate");
    }
    check(hipEventCreate(&ev_t0), "hipEventCreate");
    check(hipEventCreate(&ev_t1), "hipEventCreate");
    d_params = (double *)device_alloc(sizeof(double) * total, "alloc batch params");
    d_grad = (double *)device_alloc(sizeof(double) * total, "alloc batch gradient");
    d_energy = (double *)device_alloc(sizeof(double) * count, "alloc batch energies");
    d_step = (int *)device_alloc(sizeof(int), "alloc step counter");
    check(hipMemset(d_params, 0, sizeof(double) * total), "clear params");
    check(hipMemset(d_grad, 0, sizeof(double) * total), "clear gradient");
    check(hipMemset(d_energy, 0, sizeof(double) * count), "clear energies");
    check(hipMemset(d_step, 0, sizeof(int)), "clear step");
    for (size_t i = 0; i < count; ++i) {
        (dense_flag[i] ? dids : sids).push_back((int)i);
    }
    build_structured();
    build_dense();
}

// Circuits with n <= split on dense_scan, the others on the whole-circuit
// kernel; both parts rebuilt (the per-circuit comparison plans as well).
void Batch::repartition(int split) {
    dense_split = split;
    dids.clear();
    sids.clear();
    for (size_t i = 0; i < count; ++i) {
        dense_flag[i] = n[i] <= split ? 1 : 0;
        (dense_flag[i] ? dids : sids).push_back((int)i);
    }
    dense_single.clear();
    build_structured();
    build_dense();
}

Batch::~Batch() {
    if (s_own != nullptr) {
        (void)hipStreamSynchronize(s_own);
    }
    for (hipStream_t s : s_aux) {
        if (s != nullptr) {
            (void)hipStreamSynchronize(s);
        }
    }
    invalidate_graph();
    release_structured();
    device_free(d_params);
    device_free(d_grad);
    device_free(d_energy);
    device_free(d_m);
    device_free(d_v);
    device_free(d_step);
    device_free(d_history);
    for (hipEvent_t ev : {ev_fork, ev_join[0], ev_join[1], ev_join[2], ev_t0, ev_t1}) {
        if (ev != nullptr) {
            (void)hipEventDestroy(ev);
        }
    }
    if (s_own != nullptr) {
        (void)hipStreamDestroy(s_own);
    }
    for (hipStream_t s : s_aux) {
        if (s != nullptr) {
            (void)hipStreamDestroy(s);
        }
    }
}

void Batch::invalidate_graph() {
    if (graph_exec != nullptr) {
        (void)hipGraphExecDestroy(graph_exec);
        graph_exec = nullptr;
    }
    graph_kind = -1;
}

void Batch::release_structured() {
    device_free(d_jobs_g);
    device_free(d_jobs_e);
    device_free(d_order);
    device_free(d_wg_begin);
    device_free(d_scratch);
    device_free(d_psi);
    d_psi = nullptr;
    device_free(d_reg_g);
    device_free(d_reg_e);
    device_free(d_rec_jobs);
    device_free(d_layer_job);
    device_free(d_rec);
    d_reg_g = d_reg_e = nullptr;
    d_rec_jobs = nullptr;
    d_layer_job = nullptr;
    d_rec = nullptr;
    slices.clear();
    reg_jobs.clear();
    rec_jobs.clear();
    reg_rec.clear();
    d_jobs_g = d_jobs_e = nullptr;
    d_order = d_wg_begin = nullptr;
    d_scratch = nullptr;
    grid = 0;
}

// Records of every structured circuit, jobs of those whose states fit in
// registers.
void Batch::build_register_jobs() {
    std::vector<int> ids = sids;
    reg_of.assign(count, -1);
    gid_of.assign(count, -1);
    if (ids.empty()) {
        return;
    }
    std::stable_sort(ids.begin(), ids.end(), [&](int a, int b) {
        return n[(size_t)a] != n[(size_t)b] ? n[(size_t)a] > n[(size_t)b]
                                            : L[(size_t)a] > L[(size_t)b];
    });
    std::vector<int> layer_job;
    std::vector<size_t> place;  // record offsets of rec_jobs in their slice
    size_t rec_bytes = 0;       // of the running slice
    size_t psi_bytes = 0;
    int in_slice = 0;
    size_t rec_top = 0;         // of the largest
    size_t psi_top = 0;
    size_t most = 0;  // a quarter of the free memory, asked for where it can matter
    for (int i : ids) {
        const int q = n[(size_t)i];
        const int layers = L[(size_t)i];
        const bool large = q > kRegMaxQubits;
        const size_t bytes = circuit_record_bytes(q, layers);
        const size_t state = large ? sizeof(double2) * kStateAmps : 0;
        const size_t held = rec_bytes + bytes + psi_bytes + state;
        if (held > kSliceBytes / 4 && most == 0) {
            size_t free_b = 0;
            size_t total_b = 0;
            check(hipMemGetInfo(&free_b, &total_b), "hipMemGetInfo");
            most = std::max(free_b, kSliceBytes) / 4;
        }
        if (slices.empty() || (most > 0 && held > most) ||
            (held > kSliceBytes && in_slice >= kSliceCircuitsPerCu * num_cus)) {
            Slice next;
            next.first_layer = (int)layer_job.size();
            next.g_first = (int)jobs_g.size();
            slices.push_back(next);
            rec_bytes = 0;
            psi_bytes = 0;
            in_slice = 0;
        }
        in_slice += 1;
        Slice &sl = slices.back();
        const RegJob job{nullptr, d_energy + i, d_grad + poff[(size_t)i], nullptr, nullptr,
                         h[(size_t)i], layers, 0};
        const RecordJob record{d_params + poff[(size_t)i], nullptr, q, sl.layers};
        layer_job.insert(layer_job.end(), (size_t)layers, (int)rec_jobs.size());
        rec_jobs.push_back(record);
        place.push_back(rec_bytes / sizeof(double));
        sl.layers += layers;
        rec_bytes += bytes;
        rec_top = std::max(rec_top, rec_bytes);
        if (large) {
            gid_of[(size_t)i] = (int)jobs_g.size();
            jobs_g.push_back({job, nullptr});
            jobs_rec.push_back(record);
            sl.g_count += 1;
            psi_bytes += state;
            psi_top = std::max(psi_top, psi_bytes);
            continue;
        }
        if (sl.groups.empty() || sl.groups.back().n != q) {
            sl.groups.push_back({q, (int)reg_jobs.size(), 0});
        }
        sl.groups.back().count += 1;
        reg_of[(size_t)i] = (int)reg_jobs.size();
        reg_jobs.push_back(job);
        reg_rec.push_back(record);
    }
    d_rec = (double *)device_alloc(rec_top, "alloc batch records");
    if (psi_top > 0) {
        d_psi = (double2 *)device_alloc(psi_top, "alloc batch states");
    }
    for (size_t k = 0; k < rec_jobs.size(); ++k) {
        double *rec = d_rec + place[k];
        const size_t i = (size_t)ids[k];
        rec_jobs[k].rec = rec;
        if (gid_of[i] >= 0) {
            jobs_g[(size_t)gid_of[i]].base.rec = rec;
            jobs_rec[(size_t)gid_of[i]].rec = rec;
        } else {
            reg_jobs[(size_t)reg_of[i]].rec = rec;
            reg_rec[(size_t)reg_of[i]].rec = rec;
        }
    }
    for (const Slice &sl : slices) {
        for (int k = 0; k < sl.g_count; ++k) {
            jobs_g[(size_t)(sl.g_first + k)].psi = d_psi + kStateAmps * (size_t)k;
        }
    }
    std::vector<RegJob> energy_only = reg_jobs;
    for (auto &j : energy_only) {
        j.grad = nullptr;
    }
    const size_t job_bytes = sizeof(RegJob) * reg_jobs.size();
    if (!reg_jobs.empty()) {
        d_reg_g = (RegJob *)device_alloc(job_bytes, "alloc batch jobs");
        d_reg_e = (RegJob *)device_alloc(job_bytes, "alloc batch jobs");
        check(hipMemcpy(d_reg_g, reg_jobs.data(), job_bytes, hipMemcpyHostToDevice),
              "upload batch jobs");
        check(hipMemcpy(d_reg_e, energy_only.data(), job_bytes, hipMemcpyHostToDevice),
              "upload batch jobs");
    }
    d_rec_jobs = (RecordJob *)device_alloc(sizeof(RecordJob) * rec_jobs.size(), "alloc batch jobs");
    d_layer_job = (int *)device_alloc(sizeof(int) * layer_job.size(), "alloc batch layers");
    check(hipMemcpy(d_rec_jobs, rec_jobs.data(), sizeof(RecordJob) * rec_jobs.size(),
                    hipMemcpyHostToDevice),
          "upload batch jobs");
    check(hipMemcpy(d_layer_job, layer_job.data(), sizeof(int) * layer_job.size(),
                    hipMemcpyHostToDevice),
          "upload batch layers");
}

// Jobs and records, and for each slice a longest-first schedule of its 14-qubit
// circuits' adjoint sweeps over its workgroups.
void Batch::build_structured() {
    invalidate_graph();
    release_structured();
    jobs_g.clear();
    jobs_rec.clear();
    build_register_jobs();
    if (jobs_g.empty()) {
        return;
    }
    const int cap = grid_limit > 0 ? grid_limit : num_cus;
    std::vector<int> order;  // places in the slice's jobs
    std::vector<int> begin;
    for (Slice &sl : slices) {
        if (sl.g_count == 0) {
            continue;
        }
        sl.grid = std::min(sl.g_count, std::max(1, cap));
        grid = std::max(grid, sl.grid);
        // LPT: heaviest first onto the least-loaded workgroup
        std::vector<int> idx((size_t)sl.g_count);
        for (size_t k = 0; k < idx.size(); ++k) {
            idx[k] = (int)k;
        }
        auto cost = [&](int k) { return (double)jobs_g[(size_t)(sl.g_first + k)].base.layers; };
        std::stable_sort(idx.begin(), idx.end(), [&](int a, int b) { return cost(a) > cost(b); });
        using Slot = std::pair<double, int>;
        std::priority_queue<Slot, std::vector<Slot>, std::greater<Slot>> heap;
        for (int b = 0; b < sl.grid; ++b) {
            heap.push({0.0, b});
        }
        std::vector<std::vector<int>> lists((size_t)sl.grid);
        for (int k : idx) {
            Slot top = heap.top();
            heap.pop();
            lists[(size_t)top.second].push_back(k);
            top.first += cost(k);
            heap.push(top);
        }
        sl.begin_off = (int)begin.size();
        begin.push_back((int)order.size());
        for (auto &lst : lists) {
            order.insert(order.end(), lst.begin(), lst.end());
            begin.push_back((int)order.size());
        }
    }
    std::vector<Reg14Job> jobs_e = jobs_g;
    for (auto &j : jobs_e) {
        j.base.grad = nullptr;
    }
    d_jobs_g = (Reg14Job *)device_alloc(sizeof(Reg14Job) * jobs_g.size(), "alloc batch jobs");
    d_jobs_e = (Reg14Job *)device_alloc(sizeof(Reg14Job) * jobs_g.size(), "alloc batch jobs");
    d_order = (int *)device_alloc(sizeof(int) * order.size(), "alloc batch order");
    d_wg_begin = (int *)device_alloc(sizeof(int) * begin.size(), "alloc batch schedule");
    check(hipMemcpy(d_jobs_g, jobs_g.data(), sizeof(Reg14Job) * jobs_g.size(),
                    hipMemcpyHostToDevice),
          "upload batch jobs");
    check(hipMemcpy(d_jobs_e, jobs_e.data(), sizeof(Reg14Job) * jobs_e.size(),
                    hipMemcpyHostToDevice),
          "upload batch jobs");
    check(hipMemcpy(d_order, order.data(), sizeof(int) * order.size(), hipMemcpyHostToDevice),
          "upload batch order");
    check(hipMemcpy(d_wg_begin, begin.data(), sizeof(int) * begin.size(), hipMemcpyHostToDevice),
          "upload batch schedule");
    d_scratch = (double2 *)device_alloc(sizeof(double2) * kReg14Scratch * (size_t)grid,
                                        "alloc batch scratch");
}

void Batch::build_dense() {
    invalidate_graph();
    dense_single.clear();
    std::vector<DenseSpec> specs;
    for (int i : dids) {
        specs.push_back({n[(size_t)i], L[(size_t)i], h[(size_t)i], d_params + poff[(size_t)i],
                         d_energy + i, d_grad + poff[(size_t)i], nullptr});
    }
    dense.build(specs, specs.size());
}

void Batch::issue_eval(hipStream_t s, bool want_grad) {
    for (size_t k = 0; k < std::max<size_t>(1, slices.size()); ++k) {
        issue_slice(s, want_grad, k < slices.size() ? slices[k] : Slice{}, k == 0);
    }
}

// One slice's records and circuits, the first with the dense circuits beside
// them.  Everything has joined s again at the end: the next slice writes the
// same records and states.
void Batch::issue_slice(hipStream_t s, bool want_grad, const Slice &sl, bool with_dense) {
    if (sl.layers > 0) {
        launch_circuit_records(d_rec_jobs, RecordJob{}, d_layer_job + sl.first_layer, sl.layers,
                               s);
        check_launch("batch records");
    }
    const bool dense_here = with_dense && !dids.empty();
    // part i of the evaluation runs on stream i mod 4 (0: s itself): the
    // largest circuits first, each stream's parts one after the other
    const int parts = (sl.g_count > 0 ? 1 : 0) + (dense_here ? 1 : 0) + (int)sl.groups.size();
    const int used = std::min(parts - 1, kAux);
    if (used > 0) {
        check(hipEventRecord(ev_fork, s), "record fork");
        for (int a = 0; a < used; ++a) {
            check(hipStreamWaitEvent(s_aux[a], ev_fork, 0), "wait fork");
        }
    }
    int part = 0;
    auto next_stream = [&]() {
        const int k = part++ % (kAux + 1);
        return k == 0 ? s : s_aux[k - 1];
    };
    if (sl.g_count > 0) {
        launch_reg14((want_grad ? d_jobs_g : d_jobs_e) + sl.g_first, Reg14Job{}, d_order,
                     d_wg_begin + sl.begin_off, sl.g_count, sl.grid, d_scratch, next_stream());
        check_launch("batch 14 qubits");
    }
    if (dense_here) {
        dense.run(next_stream(), want_grad);
    }
    for (const RegGroup &g : sl.groups) {
        launch_regcircuit(g.n, (want_grad ? d_reg_g : d_reg_e) + g.first, RegJob{}, g.count,
                          next_stream());
        check_launch("batch circuits");
    }
    for (int a = 0; a < used; ++a) {
        check(hipEventRecord(ev_join[a], s_aux[a]), "record join");
        check(hipStreamWaitEvent(s, ev_join[a], 0), "wait join");
    }
}

void Batch::ensure_history(size_t entries) {
    if (entries <= history_cap) {
        return;
    }
    invalidate_graph();
    device_free(d_history);
    d_history = (double *)device_alloc(sizeof(double) * entries, "alloc energy history");
    history_cap = entries;
}

void Batch::ensure_adam() {
    if (d_m == nullptr) {
        d_m = (double *)device_alloc(sizeof(double) * total, "alloc adam m");
        d_v = (double *)device_alloc(sizeof(double) * total, "alloc adam v");
    }
}

// One optimizer step: energies and gradients at the current parameters,
// energies recorded at history[step], parameters updated, step advanced.
void Batch::issue_step(hipStream_t s, int optimizer, double lr, int capacity) {
    issue_eval(s, true);
    launch_record_energies(d_energy, (int)count, d_history, d_step, capacity, s);
    check_launch("record energies");
    if (optimizer == 0) {
        launch_gd_update(d_params, d_grad, total, lr, s);
    } else {
        launch_adam_update(d_params, d_grad, d_m, d_v, total, lr, 0.9, 0.999, 1e-8, d_step, s);
    }
    check_launch("optimizer update");
    launch_step_advance(d_step, s);
    check_launch("step advance");
}

void Batch::launch_graph(int kind, double lr, int capacity, hipStream_t s) {
    if (graph_exec == nullptr || graph_kind != kind || graph_lr != lr ||
        graph_capacity != capacity) {
        invalidate_graph();
        hipGraph_t graph = nullptr;
        check(hipStreamBeginCapture(s_own, hipStreamCaptureModeThreadLocal), "begin capture");
        try {
            if (kind <= 1) {
                issue_eval(s_own, kind == 1);
            } else {
                issue_step(s_own, kind - 2, lr, capacity);
            }
        } catch (...) {
            (void)hipStreamEndCapture(s_own, &graph);
            if (graph != nullptr) {
                (void)hipGraphDestroy(graph);
            }
            throw;
        }
        check(hipStreamEndCapture(s_own, &graph), "end capture");
        const hipError_t e = hipGraphInstantiate(&graph_exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        check(e, "instantiate graph");
        graph_kind = kind;
        graph_lr = lr;
        graph_capacity = capacity;
    }
    check(hipGraphLaunch(graph_exec, s), "launch graph");
}

void Batch::run(hipStream_t s, bool want_grad) {
    if (use_graph) {
        launch_graph(want_grad ? 1 : 0, 0.0, 0, s);
    } else {
        issue_eval(s, want_grad);
    }
}

// The comparison mode: every circuit in its own launch(es), one after the
// other on one stream, with the same kernels.
void Batch::run_per_circuit(hipStream_t s, bool want_grad) {
    if (dense_single.empty() && !dids.empty()) {
        for (int i : dids) {
            auto plan = std::make_unique<DensePlan>();
            plan->build({{n[(size_t)i], L[(size_t)i], h[(size_t)i], d_params + poff[(size_t)i],
                          d_energy + i, d_grad + poff[(size_t)i], nullptr}},
                        dids.size());
            dense_single.push_back(std::move(plan));
        }
    }
    size_t di = 0;
    for (size_t i = 0; i < count; ++i) {
        if (reg_of[i] >= 0) {
            RegJob j = reg_jobs[(size_t)reg_of[i]];
            RecordJob r = reg_rec[(size_t)reg_of[i]];
            r.first_layer = 0;
            if (!want_grad) {
                j.grad = nullptr;
            }
            launch_circuit_records(nullptr, r, nullptr, j.layers, s);
            launch_regcircuit(n[i], nullptr, j, 1, s);
            continue;
        }
        if (dense_flag[i]) {
            dense_single[di++]->run(s, want_grad);
            continue;
        }
        const size_t k = (size_t)gid_of[i];
        Reg14Job j = jobs_g[k];
        RecordJob r = jobs_rec[k];
        r.first_layer = 0;
        if (!want_grad) {
            j.base.grad = nullptr;
        }
        launch_circuit_records(nullptr, r, nullptr, j.base.layers, s);
        launch_reg14(nullptr, j, nullptr, nullptr, 1, 1, d_scratch, s);
    }
    check_launch("per-circuit launches");
}

void Batch::optimize(int optimizer, double lr, size_t steps, bool graph, double *history_out,
                     hipStream_t s) {
    if (optimizer != 0 && optimizer != 1) {
        fail(RIE_INVALID_ARGUMENT, "optimizer must be 0 (gradient descent) or 1 (Adam).");
    }
    if (!std::isfinite(lr)) {
        fail(RIE_INVALID_ARGUMENT, "learning rate must be finite.");
    }
    if (steps == 0) {
        return;
    }
    if (steps > (size_t)1 << 20) {
        fail(RIE_INVALID_ARGUMENT, "at most 2^20 optimizer steps per call.");
    }
    ensure_history(steps * count);
    const int capacity = (int)steps;
    if (optimizer == 1) {
        ensure_adam();
        launch_fill(d_m, total, 0.0, s);
        launch_fill(d_v, total, 0.0, s);
    }
    launch_set_int(d_step, 0, s);
    check_launch("optimizer reset");
    if (graph) {
        // one captured step (recording into history rows [0, capacity)), replayed
        for (size_t k = 0; k < steps; ++k) {
            launch_graph(2 + optimizer, lr, capacity, s);
        }
    } else {
        for (size_t k = 0; k < steps; ++k) {
            issue_step(s, optimizer, lr, capacity);
        }
    }
    if (history_out != nullptr) {
        check(hipMemcpyAsync(history_out, d_history, sizeof(double) * steps * count,
                             hipMemcpyDeviceToHost, s),
              "download energy history");
        check(hipStreamSynchronize(s), "sync");
    }
}

double Batch::time_ms(size_t repeats, const std::function<void(hipStream_t)> &fn) {
    fn(s_own);
    check(hipStreamSynchronize(s_own), "sync");
    std::vector<float> t;
    for (size_t r = 0; r < repeats; ++r) {
        check(hipEventRecord(ev_t0, s_own), "record");
        fn(s_own);
        check(hipEventRecord(ev_t1, s_own), "record");
        check(hipEventSynchronize(ev_t1), "sync");
        float ms = 0.0f;
        check(hipEventElapsedTime(&ms, ev_t0, ev_t1), "elapsed");
        t.push_back(ms);
    }
    std::sort(t.begin(), t.end());
    return t[t.size() / 2];
}

void Batch::autotune(size_t repeats) {
    repeats = std::max<size_t>(1, std::min<size_t>(repeats, 50));
    invalidate_graph();
    // the split candidates: every qubit count <= dense_max present, and none
    std::vector<int> splits;
    if (tune_split) {
        for (int q = dense_max; q >= 1; --q) {
            if (std::find(n.begin(), n.end(), q) != n.end()) {
                splits.push_back(q);
            }
        }
        if (!splits.empty()) {
            splits.push_back(0);
        }
    }
    if (splits.empty()) {
        splits.push_back(dense_split);
    }
    std::ostringstream rep;
    rep.precision(6);
    measured = measured || !sids.empty();
    // per split: the persistent launch's grid (leaving CUs to what runs beside
    // it); the fastest whole evaluation wins
    double best_ms = -1.0;
    int best_grid = 0;
    int best_split = splits.front();
    rep << "{\"split_ms\": {";
    for (size_t si = 0; si < splits.size(); ++si) {
        const int split = splits[si];
        if (split != dense_split || si == 0) {
            repartition(split);
        }
        std::vector<int> grid_opts;
        if (!jobs_g.empty()) {
            if (parts_beside()) {
                for (int f : {1, 2, 3, 4}) {
                    grid_opts.push_back(num_cus * f / 4);
                }
            } else {
                grid_opts.push_back(num_cus);
            }
        } else {
            grid_opts.push_back(0);
        }
        rep << (si ? ", " : "") << "\"" << split << "\": {";
        for (size_t k = 0; k < grid_opts.size(); ++k) {
            grid_limit = grid_opts[k];
            build_structured();
            const double ms = time_ms(repeats, [&](hipStream_t s) { issue_eval(s, true); });
            rep << (k ? ", " : "") << "\"" << grid_limit << "\": " << ms;
            if (best_ms < 0.0 || ms < best_ms) {
                best_ms = ms;
                best_grid = grid_limit;
                best_split = split;
            }
        }
        rep << "}";
    }
    rep << "}";
    grid_limit = best_grid;
    repartition(best_split);
    rep << ", \"dense_max_qubits\": " << best_split << ", \"batch_ms\": " << best_ms << "}";
    report = rep.str();
}

std::string Batch::config_json() const {
    std::ostringstream o;
    o << "{\"threads\": " << threads << ", \"grid\": " << grid << ", \"grid_limit\": " << grid_limit
      << ", \"dense_max_qubits\": " << dense_split << ", \"tune_split\": " << (tune_split ? "true" : "false")
      << ", \"dense_tile\": " << dense_tile << ", \"measured\": " << (measured ? "true" : "false")
      << ", \"structured_circuits\": " << sids.size() << ", \"dense_circuits\": " << dids.size()
      << ", \"chunk_by_n\": {";
    const int widest = threads >= 1024 ? 2 : threads >= 512 ? 3 : 4;  // of that workgroup size
    bool first = true;
    for (int q = 2; q <= kMaxN; ++q) {
        o << (first ? "" : ", ") << "\"" << q << "\": " << std::min(chunk_by_n[q], widest);
        first = false;
    }
    o << "}, \"autotune\": " << report << "}";
    return o.str();
}

}  // namespace rie

// ===========================================================================
// C ABI
// ===========================================================================

using rie::Batch;
using rie::guard;

namespace {

Batch *as_batch(rie_batch *b) {
    if (b == nullptr) {
        rie::fail(RIE_INVALID_ARGUMENT, "null batch");
    }
    return reinterpret_cast<Batch *>(b);
}

const Batch *as_batch(const rie_batch *b) {
    if (b == nullptr) {
        rie::fail(RIE_INVALID_ARGUMENT, "null batch");
    }
    return reinterpret_cast<const Batch *>(b);
}

}  // namespace

extern "C" {

rie_status rie_batch_create(size_t count, const int *num_qubits, const int *num_layers,
                            const double *fields, int dense_max_qubits, rie_batch **batch_out) {
    return guard([&]() {
        if (batch_out == nullptr) {
            rie::fail(RIE_INVALID_ARGUMENT, "null pointer argument.");
        }
        *batch_out = nullptr;
        auto b = std::make_unique<Batch>(count, num_qubits, num_layers, fields, dense_max_qubits);
        *batch_out = reinterpret_cast<rie_batch *>(b.release());
    });
}

void rie_batch_destroy(rie_batch *batch) {
    if (batch != nullptr) {
        delete reinterpret_cast<Batch *>(batch);
    }
}

size_t rie_batch_size(const rie_batch *batch) {
    return batch == nullptr ? 0 : reinterpret_cast<const Batch *>(batch)->count;
}

size_t rie_batch_num_params(const rie_batch *batch) {
    return batch == nullptr ? 0 : reinterpret_cast<const Batch *>(batch)->total;
}

rie_status rie_batch_param_offsets(const rie_batch *batch, size_t *offsets_out, size_t len) {
    return guard([&]() {
        const Batch *b = as_batch(batch);
        if (offsets_out == nullptr || len != b->count + 1) {
            rie::fail(RIE_INVALID_ARGUMENT, "offsets_out must hold count + 1 values.");
        }
        std::copy(b->poff.begin(), b->poff.end(), offsets_out);
    });
}

rie_status rie_batch_strategies(const rie_batch *batch, int *strategy_out, size_t len) {
    return guard([&]() {
        const Batch *b = as_batch(batch);
        if (strategy_out == nullptr || len != b->count) {
            rie::fail(RIE_INVALID_ARGUMENT, "strategy_out must hold count values.");
        }
        for (size_t i = 0; i < b->count; ++i) {
            strategy_out[i] =
                b->dense_flag[i] ? RIE_STRATEGY_DENSE_SCAN : RIE_STRATEGY_STRUCTURED_ADJOINT;
        }
    });
}

rie_status rie_batch_device_buffers(rie_batch *batch, double **d_params, double **d_energies,
                                    double **d_gradient) {
    return guard([&]() {
        Batch *b = as_batch(batch);
        if (d_params != nullptr) {
            *d_params = b->d_params;
        }
        if (d_energies != nullptr) {
            *d_energies = b->d_energy;
        }
        if (d_gradient != nullptr) {
            *d_gradient = b->d_grad;
        }
    });
}

rie_status rie_batch_set_params(rie_batch *batch, const double *params, size_t num_params) {
    return guard([&]() {
        Batch *b = as_batch(batch);
        if (params == nullptr || num_params != b->total) {
            rie::fail(RIE_INVALID_ARGUMENT, "num_params does not match the batch.");
        }
        rie::check(hipMemcpyAsync(b->d_params, params, sizeof(double) * b->total,
                                  hipMemcpyHostToDevice, b->s_own),
                   "upload params");
        rie::check(hipStreamSynchronize(b->s_own), "sync");
    });
}

rie_status rie_batch_get_params(rie_batch *batch, double *params_out, size_t num_params) {
    return guard([&]() {
        Batch *b = as_batch(batch);
        if (params_out == nullptr || num_params != b->total) {
            rie::fail(RIE_INVALID_ARGUMENT, "num_params does not match the batch.");
        }
        rie::check(hipDeviceSynchronize(), "sync");
        rie::check(hipMemcpy(params_out, b->d_params, sizeof(double) * b->total,
                             hipMemcpyDeviceToHost),
                   "download params");
    });
}

rie_status rie_batch_get_results(rie_batch *batch, double *energies_out, double *gradient_out) {
    return guard([&]() {
        Batch *b = as_batch(batch);
        if (energies_out == nullptr) {
            rie::fail(RIE_INVALID_ARGUMENT, "null pointer argument.");
        }
        rie::check(hipDeviceSynchronize(), "sync");
        rie::check(hipMemcpy(energies_out, b->d_energy, sizeof(double) * b->count,
                             hipMemcpyDeviceToHost),
                   "download energies");
        if (gradient_out != nullptr) {
            rie::check(hipMemcpy(gradient_out, b->d_grad, sizeof(double) * b->total,
                                 hipMemcpyDeviceToHost),
                       "download gradient");
        }
    });
}

rie_status rie_batch_energy_and_grad(rie_batch *batch, const double *params, size_t num_params,
                                     int compute_gradient, double *energies_out,
                                     double *gradient_out) {
    return guard([&]() {
        Batch *b = as_batch(batch);
        if (params == nullptr || energies_out == nullptr ||
            (compute_gradient && gradient_out == nullptr)) {
            rie::fail(RIE_INVALID_ARGUMENT, "null pointer argument.");
        }
        if (num_params != b->total) {
            rie::fail(RIE_INVALID_ARGUMENT, "num_params does not match the batch.");
        }
        hipStream_t s = b->s_own;
        rie::check(hipMemcpyAsync(b->d_params, params, sizeof(double) * b->total,
                                  hipMemcpyHostToDevice, s),
                   "upload params");
        b->run(s, compute_gradient != 0);
        rie::check(hipMemcpyAsync(energies_out, b->d_energy, sizeof(double) * b->count,
                                  hipMemcpyDeviceToHost, s),
                   "download energies");
        if (compute_gradient) {
            rie::check(hipMemcpyAsync(gradient_out, b->d_grad, sizeof(double) * b->total,
                                      hipMemcpyDeviceToHost, s),
                       "download gradient");
        }
        rie::check(hipStreamSynchronize(s), "sync");
    });
}

rie_status rie_batch_run_device(rie_batch *batch, int compute_gradient, void *stream) {
    return guard([&]() { as_batch(batch)->run((hipStream_t)stream, compute_gradient != 0); });
}

rie_status rie_batch_run_per_circuit(rie_batch *batch, int compute_gradient, void *stream) {
    return guard(
        [&]() { as_batch(batch)->run_per_circuit((hipStream_t)stream, compute_gradient != 0); });
}

rie_status rie_batch_set_use_graph(rie_batch *batch, int use_graph) {
    return guard([&]() {
        Batch *b = as_batch(batch);
        b->use_graph = use_graph != 0;
        b->invalidate_graph();
    });
}

rie_status rie_batch_optimize(rie_batch *batch, int optimizer, double learning_rate, size_t steps,
                              int use_graph, double *energy_history_out, void *stream) {
    return guard([&]() {
        as_batch(batch)->optimize(optimizer, learning_rate, steps, use_graph != 0,
                                  energy_history_out, (hipStream_t)stream);
    });
}

rie_status rie_batch_autotune(rie_batch *batch, size_t repeats) {
    return guard([&]() {
        Batch *b = as_batch(batch);
        rie::check(hipDeviceSynchronize(), "sync");
        b->autotune(repeats);
    });
}

rie_status rie_batch_set_tune_split(rie_batch *batch, int enabled) {
    return guard([&]() { as_batch(batch)->tune_split = enabled != 0; });
}

rie_status rie_batch_set_config(rie_batch *batch, int threads, const int *chunk_by_n,
                                size_t chunk_len, int dense_tile, int structured_grid) {
    return guard([&]() {
        Batch *b = as_batch(batch);
        if (threads != 256 && threads != 512 && threads != 1024) {
            rie::fail(RIE_INVALID_ARGUMENT, "threads must be 256, 512 or 1024.");
        }
        if (dense_tile != 32 && dense_tile != 64) {
            rie::fail(RIE_INVALID_ARGUMENT, "dense_tile must be 32 or 64.");
        }
        if (structured_grid < 0) {
            rie::fail(RIE_INVALID_ARGUMENT, "structured_grid must be >= 0.");
        }
        if (chunk_by_n != nullptr) {
            if (chunk_len != (size_t)rie::kBatchMaxQubits + 1) {
                rie::fail(RIE_INVALID_ARGUMENT, "chunk_by_n must hold 15 values (index n).");
            }
            for (size_t q = 0; q < chunk_len; ++q) {
                if (chunk_by_n[q] < 1 || chunk_by_n[q] > 4) {
                    rie::fail(RIE_INVALID_ARGUMENT, "chunk widths must be in [1, 4].");
                }
            }
            std::copy(chunk_by_n, chunk_by_n + chunk_len, b->chunk_by_n);
        }
        rie::check(hipDeviceSynchronize(), "sync");
        b->threads = threads;
        b->grid_limit = structured_grid;
        b->dense_tile = dense_tile;
        b->build_structured();
    });
}

rie_status rie_batch_config(const rie_batch *batch, char *json_out, size_t len,
                            size_t *needed_out) {
    return guard([&]() {
        const std::string s = as_batch(batch)->config_json();
        if (needed_out != nullptr) {
            *needed_out = s.size() + 1;
        }
        if (json_out != nullptr && len > 0) {
            const size_t k = std::min(len - 1, s.size());
            std::copy(s.begin(), s.begin() + (long)k, json_out);
            json_out[k] = '\0';
        }
    });
}

}  // extern "C"
