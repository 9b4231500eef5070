// Energy and gradient of whole circuits of 2..13 qubits, one workgroup per
// circuit, state and adjoint in registers (rie_regstate.hpp), and the
// per-layer records those kernels read.
//
// One kernel per qubit count: every gate, permutation and reduction of a layer
// is unrolled for it.  Grid = circuits; the workgroups of a launch are
// dispatched in order, so a caller lists the deepest circuits first.
//
// Bound by the latency of one workgroup's dependent FP64 and lane moves: a
// layer of one circuit, forward and back, takes 1.1 us at 4 qubits, 2.5 at 8,
// 14 at 12 and 22 at 13 (128 layers).  Before, with psi and lambda in LDS (a
// sweep per chunk of wires, one barrier each, pair indexes computed per group)
// or at 13 qubits in L2: 8, 15, 23 and 102 us.
#include <hip/hip_runtime.h>

#include "rie_regstate.hpp"

namespace rie {

// ---------------------------------------------------------------------------
// Records: one wave per (circuit, layer).
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void circuit_records_kernel(const RecordJob *__restrict__ jobs,
                                                              RecordJob single,
                                                              const int *__restrict__ layer_job,
                                                              int total_layers) {
    __shared__ double sh_f[4][16];
    __shared__ double sh_t[4][16];
    __shared__ double2 sh_e[4][16];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int gl = blockIdx.x * 4 + wave;
    if (gl >= total_layers) {
        return;
    }
    const RecordJob job = jobs != nullptr ? jobs[layer_job[gl]] : single;
    const int n = job.n;
    const int l = gl - job.first_layer;
    const int R = reg_bits(n);
    const int W = wave_bits(n);
    const double *p = job.params + (size_t)l * 2 * n;
    bool flip = false;
    if (lane < n) {
        double c;
        double s;
        sincos(0.5 * p[2 * lane], &s, &c);
        flip = fabs(s) > fabs(c);
        sh_f[wave][lane] = flip ? s : c;
        sh_t[wave][lane] = flip ? -c / s : s / c;
        double2 e;
        sincos(p[2 * lane + 1], &e.y, &e.x);
        // phase of logical bit 1: e, or with the flip's Z (diag(e, -1), its
        // global phase taken out) -1 / e
        sh_e[wave][lane] = flip ? make_double2(-e.x, e.y) : e;
    }
    const uint64_t flips = __ballot(flip);
    wave_lds_fence();
    const double *f = sh_f[wave];
    const double2 *e = sh_e[wave];
    double *rec = job.rec + (size_t)l * record_doubles(n);
    double sigma = 1.0;
    for (int w = 0; w < n; ++w) {
        sigma *= f[w];
    }
    // phase tables: [first, first + count) wires of one entry's index bits
    int first = -1;
    int count = 0;
    int index = 0;
    int at = 0;
    if (lane < 8) {
        first = 0;
        count = 3;
        index = lane;
        at = kRecLa + 2 * lane;
    } else if (lane < 16) {
        first = 3;
        count = 3;
        index = lane - 8;
        at = kRecLb + 2 * index;
    } else if (lane < 16 + (1 << R)) {
        first = 6;
        count = R;
        index = lane - 16;
        at = kRecReg + 2 * index;
    } else if (lane >= 32 && lane < 32 + (1 << W)) {
        first = 6 + R;
        count = W;
        index = lane - 32;
        at = kRecReg + 2 * (1 << R) + 2 * index;
    }
    if (first >= 0) {
        double2 v = make_double2(lane < 8 ? sigma : 1.0, 0.0);
        for (int j = 0; j < count; ++j) {
            if (first + j < n && ((index >> j) & 1)) {
                v = cmul(v, e[first + j]);
            }
        }
        rec[at] = v.x;
        rec[at + 1] = v.y;
    }
    if (lane >= 48) {
        const int w = lane - 48;
        // when the adjoint sweep sums wire w's dtheta, both arrays still carry
        // the factors of w and of the wires after it in its order
        double g = 1.0;
        if (w < n) {
            double left = 1.0;
            for (int v = 0; v < n; ++v) {
                left *= adjoint_order(v, R) >= adjoint_order(w, R) ? f[v] : 1.0;
            }
            g = 1.0 / (left * left);
        }
        double t = w < n ? sh_t[wave][w] : 0.0;
        if (w == kRecDphi) {
            t = 1.0 / (sigma * sigma);
        } else if (w == kRecFlips) {
            t = (double)flips;
        }
        rec[w] = t;
        rec[kRecG + w] = g;
    }
}

void launch_circuit_records(const RecordJob *d_jobs, const RecordJob &single,
                            const int *d_layer_job, int total_layers, hipStream_t s) {
    circuit_records_kernel<<<(total_layers + 3) / 4, 256, 0, s>>>(d_jobs, single, d_layer_job,
                                                                  total_layers);
}

size_t circuit_record_bytes(int n, int layers) {
    return sizeof(double) * (size_t)record_doubles(n) * (size_t)layers;
}

// ---------------------------------------------------------------------------
// Whole circuit
// ---------------------------------------------------------------------------

// kDrift: the walk goes through layer 0's rotations too and reports
// || psi - |0...0> ||^2; otherwise layer 0 only gives its gradients.
template <int n, bool kDrift>
__global__ __launch_bounds__(RegState<n>::kThreads) __attribute__((
    amdgpu_waves_per_eu(2))) void regcircuit_kernel(
    const RegJob *__restrict__ jobs, RegJob single) {
    using S = RegState<n>;
    constexpr int A = S::A;
    constexpr bool kSplit = n >= 12;  // one exchange buffer (64 KB at 12 qubits, 128 KB at 13)
    extern __shared__ double2 ex[];
    __shared__ __align__(16) double slots[3][S::kRec];
    __shared__ double red[2][32 * S::kWaves];
    const RegJob job = uniform(jobs != nullptr ? jobs[blockIdx.x] : single);
    const int t = threadIdx.x;
    S st;
    st.setup((uint32_t)(t & 63), (uint32_t)__builtin_amdgcn_readfirstlane(t >> 6));
    const int L = job.layers;
    const bool want_grad = job.grad != nullptr;
    RecordRing<S::kRec> ring{slots, job.rec, L, want_grad ? 2 * L : L, st.wave == 0,
                             2 * min(t & 63, S::kRec / 2 - 1)};
    ring.start();
    S::sync();

    double2 c[A];
    uint32_t f = 0;  // label mask (logical index = storage index ^ f)
    uint32_t k;      // flips of the current layer
    {
        const double *rec = ring.advance();
        st.product_state({rec, 0u}, c);
        k = S::flips(rec);
    }
    for (int l = 1; l < L; ++l) {
        S::sync();
        st.put(ex, c);
        S::sync();
        st.template get<0>(ex, c);
        f = ring_fwd_c(f ^ k, n);
        const double *rec = ring.advance();
        st.forward_layer({rec, f}, c, ex);
        k = S::flips(rec);
    }
    S::sync();
    st.put(ex, c);
    S::sync();
    st.template get<1>(ex, c);
    f = ring_fwd_c(f ^ k, n);

    double2 lam[A];
    const double e = wave_sum(st.hamiltonian(job.field, f, c, lam, ex));
    if (st.lane == 0) {
        red[0][32 * st.wave] = e;
    }
    S::sync();
    if (t == 0) {
        double acc = 0.0;
        for (int w = 0; w < S::kWaves; ++w) {
            acc += red[0][32 * w];
        }
        *job.energy = acc;
    }
    if (!want_grad) {
        return;
    }
    const double gscale = job.scale != nullptr ? *job.scale : 1.0;

    // psi and lambda through the inverse ring CNOT
    auto inverse_ring = [&](auto kind) {
        constexpr int k = decltype(kind)::value;
        S::sync();
        st.put(ex, c);
        if constexpr (kSplit) {
            S::sync();
            st.template get<k>(ex, c);
            S::sync();
            st.put(ex, lam);
            S::sync();
            st.template get<k>(ex, lam);
        } else {
            st.put(ex + S::kBuf, lam);
            S::sync();
            st.template get<k>(ex, c);
            st.template get<k>(ex + S::kBuf, lam);
        }
    };
    auto write_gradient = [&](int l, const double *rec, const double *sums, bool all_scaled) {
        if (t < 2 * n) {
            job.grad[(size_t)l * 2 * n + t] =
                S::gradient_entry(t, rec, sums, f, k, all_scaled) * gscale;
        }
    };
    inverse_ring(std::integral_constant<int, 3>{});
    int l = L - 1;
    if (l > 0) {
        do {
            const double *rec = ring.advance();
            k = S::flips(rec);
            f = ring_inv_c(f, n) ^ k;
            double *sums = red[l & 1];
            st.template adjoint_layer<true, kSplit>({rec, f}, c, lam, ex, sums + 32 * st.wave);
            S::sync();
            write_gradient(l, rec, sums, false);
            inverse_ring(std::integral_constant<int, 2>{});
        } while (--l > 0);
    }
    const double *rec = ring.advance();
    k = S::flips(rec);
    f = ring_inv_c(f, n) ^ k;
    st.template adjoint_layer<kDrift, kSplit>({rec, f}, c, lam, ex, red[0] + 32 * st.wave);
    S::sync();
    write_gradient(0, rec, red[0], !kDrift);
    if constexpr (!kDrift) {
        return;
    }
    // |0...0> sits at storage position 0 in every layout
    double acc = 0.0;
#pragma unroll
    for (int r = 0; r < A; ++r) {
        const double re = c[r].x - ((t == 0 && r == 0) ? 1.0 : 0.0);
        acc += re * re + c[r].y * c[r].y;
    }
    acc = wave_sum(acc);
    if (st.lane == 0) {
        red[1][32 * st.wave] = acc;
    }
    S::sync();
    if (t == 0) {
        double s = 0.0;
        for (int w = 0; w < S::kWaves; ++w) {
            s += red[1][32 * w];
        }
        *job.drift = s;
    }
}

namespace {

template <int n>
void launch_one(const RegJob *d_jobs, const RegJob &single, int count, hipStream_t s) {
    using S = RegState<n>;
    const size_t bytes = sizeof(double2) * (size_t)S::kBuf * (n >= 12 ? 1 : 2);
    if constexpr (n <= kEngineWholeQubits) {
        if (single.drift != nullptr) {
            regcircuit_kernel<n, true><<<count, S::kThreads, bytes, s>>>(d_jobs, single);
            return;
        }
    }
    regcircuit_kernel<n, false><<<count, S::kThreads, bytes, s>>>(d_jobs, single);
}

}  // namespace

void launch_regcircuit(int n, const RegJob *d_jobs, const RegJob &single, int count,
                       hipStream_t s) {
    switch (n) {
        case 2: launch_one<2>(d_jobs, single, count, s); break;
        case 3: launch_one<3>(d_jobs, single, count, s); break;
        case 4: launch_one<4>(d_jobs, single, count, s); break;
        case 5: launch_one<5>(d_jobs, single, count, s); break;
        case 6: launch_one<6>(d_jobs, single, count, s); break;
        case 7: launch_one<7>(d_jobs, single, count, s); break;
        case 8: launch_one<8>(d_jobs, single, count, s); break;
        case 9: launch_one<9>(d_jobs, single, count, s); break;
        case 10: launch_one<10>(d_jobs, single, count, s); break;
        case 11: launch_one<11>(d_jobs, single, count, s); break;
        case 12: launch_one<12>(d_jobs, single, count, s); break;
        default: launch_one<13>(d_jobs, single, count, s); break;
    }
}

}  // namespace rie
