// Energy and gradient of whole circuits of 2..13 qubits, one workgroup per
// circuit, state and adjoint in registers (rie_regstate.hpp), and the
// per-layer records those kernels read.
//
// One kernel per qubit count: every gate, permutation and reduction of a layer
// is unrolled for it.  Grid = circuits; the workgroups of a launch are
// dispatched in order, so a caller lists the deepest circuits first.
//
// Bound by the latency of one workgroup's dependent FP64 and lane moves: a
// layer of one circuit, forward and back, takes 1.0 us at 4 qubits, 2.5 at 8,
// 11 at 12 and 22 at 13 (128 layers).  Before, with psi and lambda in LDS (a
// sweep per chunk of wires, one barrier each, pair indexes computed per group)
// or at 13 qubits in L2: 8, 15, 23 and 102 us.  13 qubits pay for spills too:
// with 128 of a lane's 256 VGPRs taken by psi and lambda, 105 values go through
// scratch (336 bytes a lane).
#include <hip/hip_runtime.h>

#include "rie_regstate.hpp"

namespace rie {

// ---------------------------------------------------------------------------
// Records: one wave per (circuit, layer).
// ---------------------------------------------------------------------------

// 1 / sqrt(product of 1 + t_w^2), the scale that the tangent forms of a layer
// leave out (each wire's factor is +-1 / sqrt(1 + t^2)), and that product.  In
// twice the precision and rounded once: a product of rounded factors would let
// the norm drift by a few ulp a layer.
__device__ __forceinline__ double layer_scale(const double *t, int n, double &product) {
#pragma clang fp contract(off)
    double ph = 1.0;
    double pl = 0.0;
    for (int w = 0; w < n; ++w) {
        const double t2 = t[w] * t[w];
        const double sh = 1.0 + t2;
        const double sl = (t2 - (sh - 1.0)) + fma(t[w], t[w], -t2);
        const double h = ph * sh;
        const double l = fma(ph, sh, -h) + (ph * sl + pl * sh);
        ph = h + l;
        pl = (h - ph) + l;
    }
    const double r = 1.0 / sqrt(ph);
    const double r2 = r * r;
    const double q = r2 * ph;
    const double left = ((1.0 - q) - fma(r2, ph, -q)) - (fma(r, r, -r2) * ph + r2 * pl);
    product = ph;
    return r + 0.5 * r * left;
}

__global__ __launch_bounds__(256) void circuit_records_kernel(const RecordJob *__restrict__ jobs,
                                                              RecordJob single,
                                                              const int *__restrict__ layer_job,
                                                              int total_layers) {
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
    bool negative = false;  // the factor cos or sin taken out
    if (lane < n) {
        double c;
        double s;
        sincos(0.5 * p[2 * lane], &s, &c);
        flip = fabs(s) > fabs(c);
        const double tangent = flip ? -c / s : s / c;
        sh_t[wave][lane] = tangent;
        negative = (flip ? s : c) < 0.0;
        double2 e;
        sincos(p[2 * lane + 1], &e.y, &e.x);
        // phase of logical bit 1: e, or with the flip's Z (diag(e, -1), its
        // global phase taken out) -1 / e
        sh_e[wave][lane] = flip ? make_double2(-e.x, e.y) : e;
    }
    const uint64_t flips = __ballot(flip);
    const bool odd = (__popcll(__ballot(negative)) & 1) != 0;
    wave_lds_fence();
    const double *tw = sh_t[wave];
    const double2 *e = sh_e[wave];
    double *rec = job.rec + (size_t)l * record_doubles(n);
    double ph;
    double sigma = layer_scale(tw, n, ph);
    sigma = odd ? -sigma : sigma;
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
        for (int v = 0; v < n; ++v) {
            g *= w < n && adjoint_order(v, R) >= adjoint_order(w, R) ? fma(tw[v], tw[v], 1.0)
                                                                      : 1.0;
        }
        double t = w < n ? sh_t[wave][w] : 0.0;
        if (w == kRecDphi) {
            t = ph;
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
        st.template exchange<0>(ex, c);
        f = ring_fwd_c(f ^ k, n);
        const double *rec = ring.advance();
        st.forward_layer({rec, f}, c, ex);
        k = S::flips(rec);
    }
    st.template exchange<1>(ex, c);
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

    auto write_gradient = [&](int l, const double *rec, const double *sums, bool all_scaled) {
        if (t < 2 * n) {
            job.grad[(size_t)l * 2 * n + t] =
                S::gradient_entry(t, rec, sums, f, k, all_scaled) * gscale;
        }
    };
    st.template exchange2<3, kSplit>(ex, c, lam);
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
            st.template exchange2<2, kSplit>(ex, c, lam);
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

// ---------------------------------------------------------------------------
// 14 qubits.  psi alone fits the registers of 1024 threads (64 VGPRs of 128),
// psi and lambda together fill the whole register file.  So the forward sweep
// runs in registers and leaves psi in memory; the adjoint sweep takes the two
// halves (top wire 0 and 1) of both arrays through 512 threads' registers, one
// after the other, 13 wires each, and moves them through a scratch of two copies
// (L2 / MALL) once a layer: the read applies the inverse ring CNOT and, as it
// meets both halves, un-rotates the top wire of the layer before.
//
// Bound by latency, L2 and spills: the adjoint kernel keeps 318 values of its 256
// VGPRs in scratch (1076 bytes a lane).  A layer of one circuit takes 69 us forward
// and back against 212 for sweeps of chunks of three wires over the scratch.
// ---------------------------------------------------------------------------

constexpr uint32_t kHalf14 = 1u << 13;

__global__ __launch_bounds__(1024) void reg14_forward_kernel(const Reg14Job *__restrict__ jobs,
                                                             Reg14Job single) {
    using S = RegState<14>;
    extern __shared__ double2 ex[];
    __shared__ __align__(16) double slots[3][S::kRec];
    const Reg14Job job = uniform(jobs != nullptr ? jobs[blockIdx.x] : single);
    const int t = threadIdx.x;
    S st;
    st.setup((uint32_t)(t & 63), (uint32_t)__builtin_amdgcn_readfirstlane(t >> 6));
    const int L = job.base.layers;
    RecordRing<S::kRec> ring{slots, job.base.rec, L, L, st.wave == 0,
                             2 * min(t & 63, S::kRec / 2 - 1)};
    ring.start();
    S::sync();
    double2 c[S::A];
    const double *rec = ring.advance();
    st.product_state({rec, 0u}, c);
    uint32_t f = 0;
    uint32_t k = S::flips(rec);
    for (int l = 1; l < L; ++l) {
        st.exchange<0>(ex, c);
        f = ring_fwd_c(f ^ k, 14);
        rec = ring.advance();
        st.forward_layer({rec, f}, c, ex);
        k = S::flips(rec);
    }
    st.exchange<1>(ex, c);
    f = ring_fwd_c(f ^ k, 14);
    // storage order without label flips
    const uint32_t at = st.own ^ S::frame(f);
#pragma unroll
    for (int r = 0; r < S::A; ++r) {
        job.psi[at ^ (64u * r)] = c[r];
    }
}

// Storage position (both halves: bit 13 the top wire) that position s reads
// through the inverse ring CNOT, from layout 1 or 2 of the halves.
template <bool kLayout2>
__host__ __device__ constexpr uint32_t source14(uint32_t s) {
    using S = RegState<13, 1>;
    const uint32_t i = ring_fwd_c(S::frame(s & (kHalf14 - 1u)) | (s & kHalf14), 14);
    const uint32_t low = i & (kHalf14 - 1u);
    return (kLayout2 ? S::storage2(low) : S::frame(low)) | (i & kHalf14);
}

// Workgroup b takes circuits order[wg_begin[b] .. wg_begin[b + 1]) in turn
// (without wg_begin: `single`) on scratch + b * kReg14Scratch.
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void reg14_adjoint_kernel(
    const Reg14Job *__restrict__ jobs, Reg14Job single, const int *__restrict__ order,
    const int *__restrict__ wg_begin, double2 *scratch) {
    using S = RegState<13, 1>;
    constexpr int A = S::A;
    constexpr uint32_t kAll = 2 * kHalf14;
    extern __shared__ double2 ex[];
    __shared__ __align__(16) double slots[3][S::kRec];
    __shared__ double red[3][32 * 16];  // sums of (half, wave), three layers in turn
    const int t = threadIdx.x;
    S st;
    st.setup((uint32_t)(t & 63), (uint32_t)__builtin_amdgcn_readfirstlane(t >> 6));
    const uint32_t from1 = source14<false>(st.own);
    const uint32_t from2 = source14<true>(st.own);
    double2 *slot = scratch + (size_t)blockIdx.x * kReg14Scratch;
    const int q0 = wg_begin != nullptr ? wg_begin[blockIdx.x] : 0;
    const int q1 = wg_begin != nullptr ? wg_begin[blockIdx.x + 1] : 1;
    for (int at = q0; at < q1; ++at) {
        const Reg14Job job = uniform(jobs != nullptr ? jobs[order[at]] : single);
        const int L = job.base.layers;
        double2 c[A];
        double2 lam[A];
        double2 *next = slot + 2 * kAll;  // written now; each buffer: psi, lambda
        const double2 *src_c = job.psi;
        const double2 *src_l = slot + kAll;
        double e = 0.0;
        for (uint32_t h = 0; h < 2; ++h) {
            st.outer = h;
            const double2 *half = job.psi + h * kHalf14;
#pragma unroll
            for (int r = 0; r < A; ++r) {
                c[r] = half[st.own + 64u * r];
            }
            e += st.hamiltonian_of(job.base.field, 0u, c, lam, half,
                                   job.psi + (h ^ 1u) * kHalf14);
            st.put(slot + kAll + h * kHalf14, lam);
        }
        e = wave_sum(e);
        if (st.lane == 0) {
            red[0][st.wave] = e;
        }
        S::sync();
        if (t == 0) {
            double acc = 0.0;
            for (int w = 0; w < S::kWaves; ++w) {
                acc += red[0][w];
            }
            *job.base.energy = acc;
        }
        S::sync();
        if (job.base.grad == nullptr) {
            continue;
        }
        const double gscale = job.base.scale != nullptr ? *job.base.scale : 1.0;
        RecordRing<S::kRec> ring{slots, job.base.rec, L, 2 * L, st.wave == 0,
                                 2 * min(t & 63, S::kRec / 2 - 1), L};
        ring.start();
        S::sync();
        // One half through the inverse ring CNOT: with kTop the top wire's RY of
        // the layer before (tangent tt) comes off on the way; returns this
        // lane's share of that wire's dtheta sum.
        auto load = [&](auto first, auto rotate, uint32_t h, double tt) {
            constexpr bool kFirst = decltype(first)::value;
            constexpr bool kRotate = decltype(rotate)::value;
            uint32_t base = (kFirst ? from1 : from2) ^
                            (h != 0 ? source14<!kFirst>(kHalf14) : 0u);
            asm volatile("" : "+v"(base));
            double s = 0.0;
#pragma unroll
            for (int r = 0; r < A; ++r) {
                const uint32_t o = base ^ source14<!kFirst>(64u * r);
                c[r] = src_c[o];
                lam[r] = src_l[o];
                if constexpr (!kFirst) {
                    const double sign = (o & kHalf14) ? -1.0 : 1.0;
                    double2 pc = src_c[o ^ kHalf14];
                    pc = make_double2(sign * pc.x, sign * pc.y);
                    s += lam[r].x * pc.x + lam[r].y * pc.y;
                    if constexpr (kRotate) {
                        double2 pl = src_l[o ^ kHalf14];
                        pl = make_double2(sign * pl.x, sign * pl.y);
                        c[r] = S::rot_with(c[r], pc, tt);
                        lam[r] = S::rot_with(lam[r], pl, tt);
                    }
                    if ((r & 7) == 7) {
                        hold_schedule();
                    }
                }
            }
            return s;
        };
        auto put_top = [&](double s, double *sums) {
            const double v = wave_sum(s);
            if (st.lane == 0) {
                sums[13] = v;
            }
        };
        auto write_gradient = [&](int l, const double *rec, const double *sums, uint32_t f,
                                  uint32_t k) {
            if (t < 28) {
                job.base.grad[(size_t)l * 28 + t] =
                    RegState<14>::gradient_entry(t, rec, sums, f, k, false) * gscale;
            }
        };
        const std::true_type yes;
        const std::false_type no;
        uint32_t f = 0;  // labels of the layer before (l + 1), and its flips and record
        uint32_t k = 0;
        const double *rec = nullptr;
        int parity = 0;  // sums of the layer before
        for (int l = L - 1; l >= 0; --l) {
            const double *before = rec;
            const uint32_t f_before = f;
            const uint32_t k_before = k;
            const int now = parity == 2 ? 0 : parity + 1;
            rec = ring.advance();
            k = S::flips(rec);
            f = ring_inv_c(f, 14) ^ k;
            for (uint32_t h = 0; h < 2; ++h) {
                st.outer = h;
                const uint32_t v = st.wave | (h << 3);
                if (l == L - 1) {
                    load(yes, no, h, 0.0);
                } else {
                    const typename S::Rec kb{before, f_before};
                    const double s = load(no, yes, h, kb.t(13));
                    put_top(s, red[parity] + 32 * v);
                }
                st.adjoint_layer<true, true>({rec, f}, c, lam, ex, red[now] + 32 * v);
                st.put(next + h * kHalf14, c);
                st.put(next + kAll + h * kHalf14, lam);
            }
            S::sync();
            if (l < L - 1) {
                write_gradient(l + 1, before, red[parity], f_before, k_before);
            }
            src_c = next;
            src_l = next + kAll;
            next = next == slot ? slot + 2 * kAll : slot;
            parity = now;
        }
        for (uint32_t h = 0; h < 2; ++h) {
            const uint32_t v = st.wave | (h << 3);
            put_top(load(no, no, h, 0.0), red[parity] + 32 * v);
        }
        S::sync();
        write_gradient(0, rec, red[parity], f, k);
        S::sync();
    }
}

namespace {

template <int n>
void launch_one(const RegJob *d_jobs, const RegJob &single, int count, hipStream_t s) {
    using S = RegState<n>;
    const size_t bytes = S::kExchangeBytes * (n >= 12 ? 1 : 2);
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

void launch_reg14(const Reg14Job *d_jobs, const Reg14Job &single, const int *d_order,
                  const int *d_wg_begin, int count, int grid, double2 *scratch, hipStream_t s) {
    reg14_forward_kernel<<<count, 1024, RegState<14>::kExchangeBytes, s>>>(d_jobs, single);
    reg14_adjoint_kernel<<<grid, 512, RegState<13, 1>::kExchangeBytes, s>>>(
        d_jobs, single, d_order, d_wg_begin, scratch);
}

}  // namespace rie
