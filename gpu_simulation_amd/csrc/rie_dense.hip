// dense_scan strategy (num_qubits <= 8): products of layer chunks and a
// parallel product tree of complex128 GEMMs on the FP64 matrix cores.
//
// Reference behaviour: cpp/ising_cuda_dense_modes.inc:96-369 and
// cpp/ising_cuda_dense_kernels.cu:12-305 build [R_0, C_0, R_1, C_1, ...],
// multiply them pairwise with cuBLAS ZGEMM into a product tree, derive the
// prefix states with a down-sweep, and form the gradients layer by layer.
//
// This build:
//  * cuts the circuit into P chunks of q consecutive layers.  A leaf is the
//    product of one chunk's layers, formed column by column: each wave evolves
//    one basis state through the chunk in registers (rie_regstate.hpp), which
//    costs n 2^n per column and layer where a GEMM per layer pair costs 4^n;
//  * multiplies the leaves pairwise on v_mfma_f64_16x16x4f64 (D padded to 16
//    with an identity block), split complex, four real products;
//  * obtains the states at the chunk ends from the prefix vectors
//    x = T_{k-1}..T_0 e0 and y = T_{k-1}..T_0 T^dagger H psi of the down-sweep;
//  * walks every chunk backward from its end in registers, un-rotating x and y
//    layer by layer and taking the gradients as the whole-circuit kernel does
//    with psi and lambda.
// A circuit of one chunk needs no product: it is the whole-circuit kernel.
//
// Nodes hold transposed matrices: a wave's column is then a contiguous row,
// the parent's transpose is left^T right^T, T e0 is a row, and the matrix-vector
// products of head and down-sweep read rows in order.
//
// Every kernel is driven by a job table (DenseJob) and a work table of
// (job, first block) pairs, so one launch serves one circuit or a whole
// batch of circuits of different sizes.
//
// Measured, 8 qubits x 128 layers through the host-array call: 1174 us before
// (one leaf per layer, 127 GEMMs of 256^3, a down-sweep level of 91 us in one
// workgroup per parent), 150 us now.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <utility>
#include <vector>

#include "rie_dense.hpp"
#include "rie_engine_internal.hpp"
#include "rie_regstate.hpp"

namespace rie {

typedef double double4_t __attribute__((ext_vector_type(4)));

// Entry of a launch's work table whose block range holds block b:
// tab[k].x = job index, tab[k].y = first block of that job in the launch.
__device__ __forceinline__ int find_item(const int2 *__restrict__ tab, int count, int b) {
    int lo = 0;
    int hi = count - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (tab[mid].y <= b) {
            lo = mid;
        } else {
            hi = mid - 1;
        }
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

__host__ __device__ __forceinline__ size_t level_node(int P, int level) {
    return (size_t)(2 * P - 2 * (P >> level));
}

constexpr int kLeafWaves = 4;  // waves (columns, or chunks) per workgroup

// LDS of one wave of the chunk kernels.
template <int n>
struct ChunkLds {
    double2 ex[2 * RegState<n>::kBuf];
    double slots[3][RegState<n>::kRec];
    double red[32];
};

// ---------------------------------------------------------------------------
// Leaves: wave = (chunk, column).  Row c of the node's transposed planes is
// the chunk applied to basis state c.  Padding rows (2^n <= c < D, n < 4) are
// identity.
// ---------------------------------------------------------------------------

template <int n>
__global__ __launch_bounds__(64 * kLeafWaves) void dense_leaf_kernel(
    const DenseJob *__restrict__ jobs, const int2 *__restrict__ tab, int count) {
    using S = RegState<n>;
    constexpr int A = S::A;
    __shared__ ChunkLds<n> lds[kLeafWaves];
    const int item = find_item(tab, count, blockIdx.x);
    const DenseJob &J = jobs[tab[item].x];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int D = uniform(J.D);
    const int at = ((int)blockIdx.x - tab[item].y) * kLeafWaves + wave;
    const int chunk = __builtin_amdgcn_readfirstlane(at >> J.log_d);
    const int col = __builtin_amdgcn_readfirstlane(at & (D - 1));
    const int q = uniform(J.q);
    const int l0 = chunk * q;
    const int layers = max(0, min(uniform(J.L) - l0, q));
    double *re = J.tree + (size_t)chunk * J.node_doubles + (size_t)col * D;
    double *im = re + (size_t)D * D;
    if (col >= (int)S::kAmps || layers == 0) {
        for (int i = lane; i < D; i += 64) {
            re[i] = i == col ? 1.0 : 0.0;
            im[i] = 0.0;
        }
        return;
    }
    S st;
    st.setup((uint32_t)lane, 0u);
    ChunkLds<n> &my = lds[wave];
    RecordRing<S::kRec> ring{my.slots, uniform(J.rec) + (size_t)l0 * S::kRec, layers, layers, true,
                             2 * min(lane, S::kRec / 2 - 1)};
    ring.start();
    double2 a[A];
#pragma unroll
    for (int r = 0; r < A; ++r) {
        const bool one = st.active && S::logical2(st.own ^ (uint32_t)(64 * r)) == (uint32_t)col;
        a[r] = make_double2(one ? 1.0 : 0.0, 0.0);
    }
    uint32_t f = 0;
    int l = 0;
    while (true) {
        const double *rec = ring.advance();
        st.forward_layer({rec, f}, a, my.ex);
        f = ring_fwd_c(f ^ S::flips(rec), n);
        S::sync();
        st.put(my.ex, a);
        S::sync();
        if (++l == layers) {
            break;
        }
        st.template get<0>(my.ex, a);
    }
    st.template get<1>(my.ex, a);
#pragma unroll
    for (int r = 0; r < A; ++r) {
        if (st.active) {
            const uint32_t i = (st.x | ((uint32_t)r << 6)) ^ f;
            re[i] = a[r].x;
            im[i] = a[r].y;
        } else if (lane < D) {
            re[lane] = 0.0;
            im[lane] = 0.0;
        }
    }
}

// ---------------------------------------------------------------------------
// Product-tree level on FP64 MFMA: parent q = left child (2q) * right child
// (2q + 1) of the transposed planes, one 16 x 16 output tile per workgroup, the
// sum over k split over its four waves: a level has few products (at most P / 2
// of D x D), so the tiles are small and the chain of MFMAs a wave runs is D / 16
// k-steps instead of D / 4.  Operands come straight from L2: lane (i, g) takes
// A[i][4g .. 4g+3] of a 16-wide k block with two 16-byte loads and the MFMA of
// step m pairs it with B[4g + m][j].
// v_mfma_f64_16x16x4f64 lane layout: A[i][k] in lane i + 16k, B[k][j] in
// lane j + 16k, D[i][j] in lane j + 16(i%4), element i/4 (one output row per
// 16-lane group and register, unlike the FP32 16x16 forms).
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void zgemm_level_kernel(const DenseJob *__restrict__ jobs,
                                                          const int2 *__restrict__ tab, int count,
                                                          int level) {
    __shared__ double part[3][2][4][64];  // waves 1..3: re, im
    const int item = find_item(tab, count, blockIdx.x);
    const DenseJob &J = jobs[tab[item].x];
    const int D = J.D;
    const int local = (int)blockIdx.x - tab[item].y;
    const int side = D >> 4;
    const int q = local / (side * side);
    const int bt = local % (side * side);
    const int tr = (bt / side) * 16;
    const int tc = (bt % side) * 16;
    const size_t DD = (size_t)D * D;
    const size_t nd = J.node_doubles;
    const double *ar = J.tree + (level_node(J.P, level - 1) + 2 * (size_t)q) * nd;
    const double *ai = ar + DD;
    const double *br = ar + nd;
    const double *bi = br + DD;
    double *cr = J.tree + (level_node(J.P, level) + (size_t)q) * nd;
    double *ci = cr + DD;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int i = lane & 15;
    const int g = lane >> 4;
    double4_t acc_r = {0.0, 0.0, 0.0, 0.0};
    double4_t acc_i = {0.0, 0.0, 0.0, 0.0};
    for (int k0 = 16 * wave; k0 < D; k0 += 64) {
        const double *pa = ar + (size_t)(tr + i) * D + k0 + 4 * g;
        const double *pai = ai + (size_t)(tr + i) * D + k0 + 4 * g;
        const double2 r01 = *reinterpret_cast<const double2 *>(pa);
        const double2 r23 = *reinterpret_cast<const double2 *>(pa + 2);
        const double2 i01 = *reinterpret_cast<const double2 *>(pai);
        const double2 i23 = *reinterpret_cast<const double2 *>(pai + 2);
        const double a_r[4] = {r01.x, r01.y, r23.x, r23.y};
        const double a_i[4] = {i01.x, i01.y, i23.x, i23.y};
        double b_r[4];
        double b_i[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const size_t o = (size_t)(k0 + 4 * g + m) * D + tc + i;
            b_r[m] = br[o];
            b_i[m] = bi[o];
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            acc_r = __builtin_amdgcn_mfma_f64_16x16x4f64(a_r[m], b_r[m], acc_r, 0, 0, 0);
            acc_i = __builtin_amdgcn_mfma_f64_16x16x4f64(a_r[m], b_i[m], acc_i, 0, 0, 0);
            acc_r = __builtin_amdgcn_mfma_f64_16x16x4f64(-a_i[m], b_i[m], acc_r, 0, 0, 0);
            acc_i = __builtin_amdgcn_mfma_f64_16x16x4f64(a_i[m], b_r[m], acc_i, 0, 0, 0);
        }
    }
    if (wave > 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            part[wave - 1][0][e][lane] = acc_r[e];
            part[wave - 1][1][e][lane] = acc_i[e];
        }
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const double vr = (acc_r[e] + part[0][0][e][lane]) +
                              (part[1][0][e][lane] + part[2][0][e][lane]);
            const double vi = (acc_i[e] + part[0][1][e][lane]) +
                              (part[1][1][e][lane] + part[2][1][e][lane]);
            const size_t o = (size_t)(tr + 4 * e + g) * D + tc + i;
            cr[o] = vr;
            ci[o] = vi;
        }
    }
}

// ---------------------------------------------------------------------------
// Root: psi = T e0, lambda = H psi, E = Re<psi|lambda>, eta = T^dagger lambda;
// also seeds the down-sweep with the root pair [x = e0 | y = eta] in vec_a.
// A workgroup forms psi and lambda for itself and 16 entries of eta (one row
// of the transposed root each); a circuit's first one writes the rest.
// ---------------------------------------------------------------------------

constexpr int kHeadRows = 16;

__global__ __launch_bounds__(256) void dense_head_kernel(const DenseJob *__restrict__ jobs,
                                                         const int2 *__restrict__ tab, int count,
                                                         double *energy_override) {
    __shared__ double2 psi[256];
    __shared__ double2 lam[256];
    __shared__ double red[4];
    const int item = find_item(tab, count, blockIdx.x);
    const DenseJob &J = jobs[tab[item].x];
    const int block = (int)blockIdx.x - tab[item].y;
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = t >> 6;
    const int n = J.n;
    const int D = J.D;
    const int d = 1 << n;
    const size_t DD = (size_t)D * D;
    const double *re = J.tree + (size_t)(2 * J.P - 2) * J.node_doubles;
    const double *im = re + DD;
    if (t < D) {
        psi[t] = (t < d) ? make_double2(re[t], im[t]) : make_double2(0, 0);
    }
    __syncthreads();
    double e = 0.0;
    if (t < D) {
        double2 hv = make_double2(0.0, 0.0);
        if (t < d) {
            const double dg = ham_diag((uint64_t)t, n);
            const double2 v = psi[t];
            double fx = 0.0;
            double fy = 0.0;
            for (int w = 0; w < n; ++w) {
                const double2 p = psi[t ^ (1 << w)];
                fx += p.x;
                fy += p.y;
            }
            hv = make_double2(dg * v.x - J.field * fx, dg * v.y - J.field * fy);
            e = v.x * hv.x + v.y * hv.y;
        }
        lam[t] = hv;
    }
    e = wave_sum(e);
    if (lane == 0) {
        red[wave] = e;
    }
    __syncthreads();
    if (block == 0) {
        if (t == 0) {
            double *out = energy_override != nullptr ? energy_override : J.energy;
            *out = red[0] + red[1] + red[2] + red[3];
        }
        if (t < D) {
            J.head[t] = psi[t];
            J.head[D + t] = lam[t];
            J.vec_a[t] = make_double2(t == 0 ? 1.0 : 0.0, 0.0);
        }
    }
    // eta_c = sum_r conj(T[r][c]) lambda_r
    for (int j = wave; j < kHeadRows; j += 4) {
        const int c = block * kHeadRows + j;
        double ex = 0.0;
        double ey = 0.0;
        for (int r = lane; r < D; r += 64) {
            const double tr = re[(size_t)c * D + r];
            const double ti = im[(size_t)c * D + r];
            const double2 l = lam[r];
            ex += tr * l.x + ti * l.y;
            ey += tr * l.y - ti * l.x;
        }
        ex = wave_sum(ex);
        ey = wave_sum(ey);
        if (lane == 0) {
            J.vec_a[D + c] = make_double2(ex, ey);
        }
    }
}

// One down-sweep level: parent p hands (x, y) to its left child and
// (N x, N y) to its right child, N = the left child's product.  A circuit's
// step at level j reads vec_a when (levels - j) is even, else vec_b.  A
// workgroup forms 64 entries (or all D) of both products: thread (r, s) adds
// columns s, s + S, ... of N, whose transposed rows it reads in order with the
// wave's other r, and the S partial sums meet in LDS.
constexpr int kDownRows = 64;

__global__ __launch_bounds__(256) void dense_down_kernel(const DenseJob *__restrict__ jobs,
                                                         const int2 *__restrict__ tab, int count,
                                                         int level) {
    __shared__ double2 xs[256];
    __shared__ double2 ys[256];
    __shared__ double2 px[256];
    __shared__ double2 py[256];
    const int item = find_item(tab, count, blockIdx.x);
    const DenseJob &J = jobs[tab[item].x];
    const int D = J.D;
    const int t = threadIdx.x;
    const bool even = ((J.levels - level) & 1) == 0;
    const double2 *vin = even ? J.vec_a : J.vec_b;
    double2 *vout = even ? J.vec_b : J.vec_a;
    const size_t DD = (size_t)D * D;
    const int rows = D < kDownRows ? D : kDownRows;
    const int parts = D / rows;
    const int block = (int)blockIdx.x - tab[item].y;
    const int p = block / parts;
    const int r0 = (block % parts) * rows;
    const double2 *x = vin + (size_t)p * 2 * D;
    const double2 *y = x + D;
    const double *re = J.tree + (level_node(J.P, level - 1) + 2 * (size_t)p) * J.node_doubles;
    const double *im = re + DD;
    if (t < D) {
        xs[t] = x[t];
        ys[t] = y[t];
    }
    __syncthreads();
    const int S = 256 / rows;
    const int r = r0 + t % rows;
    double2 nx = make_double2(0.0, 0.0);
    double2 ny = make_double2(0.0, 0.0);
#pragma unroll 8
    for (int c = t / rows; c < D; c += S) {
        const double mr = re[(size_t)c * D + r];
        const double mi = im[(size_t)c * D + r];
        const double2 xv = xs[c];
        const double2 yv = ys[c];
        nx.x += mr * xv.x - mi * xv.y;
        nx.y += mr * xv.y + mi * xv.x;
        ny.x += mr * yv.x - mi * yv.y;
        ny.y += mr * yv.y + mi * yv.x;
    }
    px[t] = nx;
    py[t] = ny;
    __syncthreads();
    if (t < rows) {
        for (int s = 1; s < S; ++s) {
            nx.x += px[t + s * rows].x;
            nx.y += px[t + s * rows].y;
            ny.x += py[t + s * rows].x;
            ny.y += py[t + s * rows].y;
        }
        double2 *left = vout + (size_t)(2 * p) * 2 * D;
        double2 *right = vout + (size_t)(2 * p + 1) * 2 * D;
        left[r] = xs[r];
        left[D + r] = ys[r];
        right[r] = nx;
        right[D + r] = ny;
    }
}

// ---------------------------------------------------------------------------
// Gradients: one wave walks one chunk backward from its end states (the next
// chunk's prefix pair, or psi and lambda).
// ---------------------------------------------------------------------------

template <int n>
__global__ __launch_bounds__(64 * kLeafWaves) void dense_walk_kernel(
    const DenseJob *__restrict__ jobs, const int2 *__restrict__ tab, int count,
    double *grad_override, const double *scale_override) {
    using S = RegState<n>;
    constexpr int A = S::A;
    __shared__ ChunkLds<n> lds[kLeafWaves];
    const int item = find_item(tab, count, blockIdx.x);
    const DenseJob &J = jobs[tab[item].x];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int P = uniform(J.P);
    const int D = uniform(J.D);
    const int L = uniform(J.L);
    const int q = uniform(J.q);
    const int chunk = ((int)blockIdx.x - uniform(tab[item].y)) * kLeafWaves + wave;
    const int l0 = chunk * q;
    const int layers = min(L - l0, q);
    if (chunk >= P || layers <= 0) {
        return;
    }
    const double *sp = scale_override != nullptr ? scale_override : uniform(J.scale);
    const double gscale = sp != nullptr ? *sp : 1.0;
    double *grad = grad_override != nullptr ? grad_override : uniform(J.grad);
    // the last down-sweep step (level 1) wrote vec_b when levels is odd
    const double2 *leaves = (uniform(J.levels) & 1) ? uniform(J.vec_b) : uniform(J.vec_a);
    const double2 *end = l0 + layers < L ? leaves + (size_t)(chunk + 1) * 2 * D : uniform(J.head);
    S st;
    st.setup((uint32_t)lane, 0u);
    ChunkLds<n> &my = lds[wave];
    RecordRing<S::kRec> ring{my.slots, uniform(J.rec) + (size_t)l0 * S::kRec, layers, 2 * layers,
                             true, 2 * min(lane, S::kRec / 2 - 1), layers};
    ring.start();
    double2 c[A];
    double2 l[A];
#pragma unroll
    for (int r = 0; r < A; ++r) {
        const uint32_t i = st.x | ((uint32_t)r << 6);
        c[r] = st.active ? end[i] : make_double2(0.0, 0.0);
        l[r] = st.active ? end[D + i] : make_double2(0.0, 0.0);
    }
    S::sync();
    st.put(my.ex, c);
    st.put(my.ex + S::kBuf, l);
    S::sync();
    st.template get<3>(my.ex, c);
    st.template get<3>(my.ex + S::kBuf, l);
    uint32_t f = 0;
    int left = layers;
    do {
        --left;
        const double *rec = ring.advance();
        const uint32_t k = S::flips(rec);
        f = ring_inv_c(f, n) ^ k;
        st.template adjoint_layer<true, false>({rec, f}, c, l, my.ex, my.red);
        S::sync();
        if (lane < 2 * n) {
            grad[(size_t)(l0 + left) * 2 * n + lane] =
                S::gradient_entry(lane, rec, my.red, f, k, false) * gscale;
        }
        S::sync();
        st.put(my.ex, c);
        st.put(my.ex + S::kBuf, l);
        S::sync();
        st.template get<2>(my.ex, c);
        st.template get<2>(my.ex + S::kBuf, l);
    } while (left > 0);
}

// ---------------------------------------------------------------------------
// Plans
// ---------------------------------------------------------------------------

namespace {

struct Geometry {
    int D;
    int P;
    int q;
    int levels;
    size_t nd;
    size_t tree_bytes;
    size_t vec_bytes;
    size_t head_bytes;
    size_t bytes;
};

size_t align256(size_t b) { return (b + 255) & ~size_t{255}; }

Geometry geometry(int n, int L, int P) {
    Geometry g{};
    g.D = std::max(1 << n, 16);
    g.P = P;
    g.q = (L + P - 1) / P;
    while ((1 << g.levels) < P) {
        g.levels++;
    }
    g.nd = (size_t)2 * g.D * g.D;
    g.tree_bytes = sizeof(double) * g.nd * (2 * (size_t)P - 1);
    g.vec_bytes = sizeof(double2) * (size_t)P * 2 * g.D;
    g.head_bytes = sizeof(double2) * 2 * (size_t)g.D;
    g.bytes = align256(g.tree_bytes) + 2 * align256(g.vec_bytes) + align256(g.head_bytes);
    return g;
}

template <int n>
void launch_leaf_n(const DenseJob *jobs, const int2 *tab, int count, int blocks, hipStream_t s) {
    dense_leaf_kernel<n><<<blocks, 64 * kLeafWaves, 0, s>>>(jobs, tab, count);
}

template <int n>
void launch_walk_n(const DenseJob *jobs, const int2 *tab, int count, int blocks, double *grad,
                   const double *scale, hipStream_t s) {
    dense_walk_kernel<n><<<blocks, 64 * kLeafWaves, 0, s>>>(jobs, tab, count, grad, scale);
}

#define RIE_DENSE_BY_N(fn, n, ...)             \
    switch (n) {                               \
        case 1: break;                         \
        case 2: fn<2>(__VA_ARGS__); break;     \
        case 3: fn<3>(__VA_ARGS__); break;     \
        case 4: fn<4>(__VA_ARGS__); break;     \
        case 5: fn<5>(__VA_ARGS__); break;     \
        case 6: fn<6>(__VA_ARGS__); break;     \
        case 7: fn<7>(__VA_ARGS__); break;     \
        default: fn<8>(__VA_ARGS__); break;    \
    }

}  // namespace

// The largest power of two that leaves chunks of 16 layers or more, if that is
// at least 4: the sweep through a chunk and back takes about 1.1 (4 qubits) to
// 2.5 us (8) a layer, a tree level (GEMM and down-sweep launch) about 15 us, so
// below 64 layers the tree costs more than the parallel chunks save.  The
// leaves of all circuits that run together (one wave per column and chunk)
// stay within eight waves per SIMD of the chip: beyond that the columns cost
// more than the sequential sweep they replace.
int DensePlan::chunks_for(int n, int L, size_t sharing) {
    constexpr size_t kWaveBudget = 8192;
    int P = 1;
    while (L / (2 * P) >= 16 && sharing * (size_t)(2 * P) * (size_t{1} << n) <= kWaveBudget) {
        P *= 2;
    }
    return P >= 4 ? P : 1;
}

void DensePlan::release() {
    device_free(d_jobs_);
    device_free(d_flat_);
    device_free(d_flat_energy_);
    device_free(d_records_);
    device_free(d_layer_job_);
    device_free(d_tab_);
    device_free(arena_);
    d_jobs_ = nullptr;
    d_flat_ = d_flat_energy_ = nullptr;
    d_records_ = nullptr;
    d_layer_job_ = nullptr;
    d_tab_ = nullptr;
    arena_ = nullptr;
    arena_bytes_ = 0;
    specs_.clear();
    jobs_.clear();
    flat_.clear();
    flat_groups_.clear();
    records_.clear();
    layers_ = 0;
    leaves_.clear();
    gemm_.clear();
    down_.clear();
    walks_.clear();
}

DensePlan::~DensePlan() { release(); }

void DensePlan::build(const std::vector<DenseSpec> &specs, size_t sharing) {
    release();
    if (specs.empty()) {
        return;
    }
    if (specs.size() > 65535) {
        fail(RIE_INVALID_ARGUMENT, "at most 65535 dense_scan circuits per batch");
    }
    for (const auto &sp : specs) {
        if (sp.n < 2 || sp.n > 8 || sp.L < 1) {
            fail(RIE_INVALID_ARGUMENT, "dense_scan requires 2 <= num_qubits <= 8 and layers >= 1.");
        }
    }
    specs_ = specs;
    std::stable_sort(specs_.begin(), specs_.end(), [](const DenseSpec &a, const DenseSpec &b) {
        return a.n != b.n ? a.n > b.n : a.L > b.L;
    });
    sharing = std::max(sharing, specs_.size());
    size_t total = 0;
    for (const auto &sp : specs_) {
        const int P = chunks_for(sp.n, sp.L, sharing);
        total += align256(circuit_record_bytes(sp.n, sp.L));
        total += P > 1 ? geometry(sp.n, sp.L, P).bytes : 0;
    }
    arena_ = device_alloc(total, "alloc dense_scan buffers");
    arena_bytes_ = total;
    char *cursor = (char *)arena_;
    auto take = [&](size_t bytes) {
        char *p = cursor;
        cursor += align256(bytes);
        return p;
    };
    std::vector<int> layer_job;
    int max_levels = 0;
    for (const auto &sp : specs_) {
        double *rec = (double *)take(circuit_record_bytes(sp.n, sp.L));
        layer_job.insert(layer_job.end(), (size_t)sp.L, (int)records_.size());
        records_.push_back({sp.params, rec, sp.n, layers_});
        layers_ += sp.L;
        const int P = chunks_for(sp.n, sp.L, sharing);
        if (P == 1) {
            if (flat_groups_.empty() || flat_groups_.back().n != sp.n) {
                flat_groups_.push_back({sp.n, (int)flat_.size(), 0});
            }
            flat_groups_.back().count += 1;
            flat_.push_back({rec, sp.energy, sp.grad, nullptr, sp.scale, sp.field, sp.L, 0});
            continue;
        }
        const Geometry g = geometry(sp.n, sp.L, P);
        DenseJob J{};
        J.rec = rec;
        J.tree = (double *)take(g.tree_bytes);
        J.vec_a = (double2 *)take(g.vec_bytes);
        J.vec_b = (double2 *)take(g.vec_bytes);
        J.head = (double2 *)take(g.head_bytes);
        J.energy = sp.energy;
        J.grad = sp.grad;
        J.scale = sp.scale;
        J.node_doubles = g.nd;
        J.field = sp.field;
        J.n = sp.n;
        J.L = sp.L;
        J.D = g.D;
        while ((1 << J.log_d) < g.D) {
            J.log_d++;
        }
        J.P = g.P;
        J.levels = g.levels;
        J.q = g.q;
        jobs_.push_back(J);
        max_levels = std::max(max_levels, g.levels);
    }

    std::vector<int2> tab;
    auto add_launch = [&](Launch &la, auto &&blocks_of) {
        la.tab_off = tab.size();
        for (int j = 0; j < (int)jobs_.size(); ++j) {
            const long b = blocks_of(jobs_[(size_t)j]);
            if (b <= 0) {
                continue;
            }
            if ((long)la.blocks + b > 0x7fffffffL) {
                fail(RIE_INVALID_ARGUMENT, "dense_scan batch too large for one launch");
            }
            tab.push_back(make_int2(j, la.blocks));
            la.blocks += (int)b;
            la.count += 1;
        }
        return la.count > 0;
    };
    for (int n = 8; n >= 2; --n) {
        Launch leaf;
        if (add_launch(leaf, [n](const DenseJob &J) {
                return J.n == n ? (long)J.P * J.D / kLeafWaves : 0L;
            })) {
            leaves_.push_back({n, leaf});
            Launch walk;
            add_launch(walk, [n](const DenseJob &J) {
                return J.n == n ? (long)(J.P + kLeafWaves - 1) / kLeafWaves : 0L;
            });
            walks_.push_back({n, walk});
        }
    }
    for (int level = 1; level <= max_levels; ++level) {
        Launch la;
        la.level = level;
        add_launch(la, [&](const DenseJob &J) {
            const long side = J.D / 16;
            return J.levels < level ? 0L : (long)(J.P >> level) * side * side;
        });
        gemm_.push_back(la);
    }
    head_ = Launch{};
    add_launch(head_, [](const DenseJob &J) { return (long)J.D / kHeadRows; });
    for (int level = max_levels; level >= 1; --level) {
        Launch la;
        la.level = level;
        add_launch(la, [&](const DenseJob &J) {
            return J.levels < level ? 0L : (long)(J.P >> level) * std::max(1, J.D / kDownRows);
        });
        down_.push_back(la);
    }

    auto upload = [](auto **dst, const auto &src, const char *what) {
        if (src.empty()) {
            return;
        }
        using T = std::decay_t<decltype(src[0])>;
        *dst = (T *)device_alloc(sizeof(T) * src.size(), what);
        check(hipMemcpy(*dst, src.data(), sizeof(T) * src.size(), hipMemcpyHostToDevice), what);
    };
    std::vector<RegJob> energy_only = flat_;
    for (auto &j : energy_only) {
        j.grad = nullptr;
    }
    upload(&d_jobs_, jobs_, "upload dense jobs");
    upload(&d_flat_, flat_, "upload dense jobs");
    upload(&d_flat_energy_, energy_only, "upload dense jobs");
    upload(&d_records_, records_, "upload dense jobs");
    upload(&d_layer_job_, layer_job, "upload dense layers");
    upload(&d_tab_, tab, "upload dense work tables");
}

void DensePlan::run(hipStream_t s, bool want_grad, const double *params_override,
                    double *energy_override, double *grad_override,
                    const double *scale_override) const {
    if (specs_.empty()) {
        return;
    }
    const bool overridden = params_override != nullptr || energy_override != nullptr ||
                            grad_override != nullptr || scale_override != nullptr;
    if (overridden && specs_.size() != 1) {
        fail(RIE_DEVICE_ERROR, "internal: dense overrides need a single-circuit plan");
    }
    RecordJob record = records_[0];
    if (params_override != nullptr) {
        record.params = params_override;
    }
    launch_circuit_records(overridden ? nullptr : d_records_, record, d_layer_job_, layers_, s);
    check_launch("dense records");
    for (const Group &g : flat_groups_) {
        RegJob j = flat_[(size_t)g.first];
        j.energy = energy_override != nullptr ? energy_override : j.energy;
        j.grad = !want_grad ? nullptr : grad_override != nullptr ? grad_override : j.grad;
        j.scale = scale_override != nullptr ? scale_override : j.scale;
        const RegJob *table = (want_grad ? d_flat_ : d_flat_energy_) + g.first;
        launch_regcircuit(g.n, overridden ? nullptr : table, j, g.count, s);
        check_launch("dense whole circuits");
    }
    if (jobs_.empty()) {
        return;
    }
    for (const auto &[n, la] : leaves_) {
        RIE_DENSE_BY_N(launch_leaf_n, n, d_jobs_, d_tab_ + la.tab_off, la.count, la.blocks, s)
        check_launch("dense_leaf");
    }
    for (const Launch &la : gemm_) {
        zgemm_level_kernel<<<la.blocks, 256, 0, s>>>(d_jobs_, d_tab_ + la.tab_off, la.count,
                                                     la.level);
        check_launch("zgemm_level");
    }
    dense_head_kernel<<<head_.blocks, 256, 0, s>>>(d_jobs_, d_tab_ + head_.tab_off, head_.count,
                                                   energy_override);
    check_launch("dense_head");
    if (!want_grad) {
        return;
    }
    for (const Launch &la : down_) {
        dense_down_kernel<<<la.blocks, 256, 0, s>>>(d_jobs_, d_tab_ + la.tab_off, la.count,
                                                    la.level);
        check_launch("dense_down");
    }
    for (const auto &[n, la] : walks_) {
        RIE_DENSE_BY_N(launch_walk_n, n, d_jobs_, d_tab_ + la.tab_off, la.count, la.blocks,
                       grad_override, scale_override, s)
        check_launch("dense_walk");
    }
}

// ---------------------------------------------------------------------------
// Engine glue (one circuit)
// ---------------------------------------------------------------------------

void Engine::dense_init() {
    dense = new DensePlan();
    DenseSpec sp{n, L, h, d_params, d_energy, d_grad, nullptr};
    dense->build({sp}, 1);
}

void Engine::dense_free() {
    delete dense;
    dense = nullptr;
}

void Engine::dense_run(hipStream_t s, bool want_grad, const double *params, const double *scale,
                       double *energy_out, double *grad_out) {
    dense->run(s, want_grad, params, energy_out, want_grad ? grad_out : nullptr, scale);
}

}  // namespace rie
