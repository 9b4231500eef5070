// FP32 multilayer perceptron kernels for the learned warm start: training
// (forward, backward, Adam) and inference of x -> GELU(x W1 + b1) ->
// GELU(. W2 + b2) -> . W3 + b3, all row-major with one sample per row.
//
// No counterpart in the reference.  One GEMM on the FP32 matrix cores with
// fused epilogues serves every product of the forward and backward pass:
//   forward  Z = X W + b, A = GELU(Z)           (epilogue kBiasGelu / kBias)
//   loss     dY = 2 / count (X W + b - T) and its squares (epilogue kMse)
//   backward dA = dZn W^T, dZ = dA * GELU'(Z)     (transposed B, epilogue kDGelu)
//            [dW; db] = [A 1]^T dZ                (transposed A with a row of ones)
// GELU is the exact form 0.5 x (1 + erf(x / sqrt 2)) (torch.nn.GELU's
// default), evaluated with the device library's erff / expf.
//
// The products are small (a few hundred to a few thousand rows by 256), so what
// bounds them is the number of workgroups and the chain over k: a workgroup
// forms a 16 x 16 (or, from 512 such blocks of 32 x 32 on, 32 x 32) tile, its four
// waves split k, and operands come straight from L2.  512 rows, 3-256-256-80: 842
// us a loss and gradient through the host-array call with 64 x 64 LDS tiles (8 to
// 32 workgroups), a column sum per bias in one thread per column (3 x 95 us) and
// a serial loss sum; 135 us now.
#include <hip/hip_runtime.h>

#include "rie_kernels.hpp"
#include "rie_mlp_shape.hpp"

namespace rie {

namespace {

typedef float float4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float gelu(float x) {
    return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f));
}

__device__ __forceinline__ float gelu_grad(float x) {
    const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
    const float pdf = expf(-0.5f * x * x) * 0.39894228040143268f;
    return cdf + x * pdf;
}

}  // namespace

// C[M x N] = op(A)[M x K] * op(B)[K x N]; op(A) = A (M x K) or A^T (A is K x
// Ma; row Ma of A^T, if M > Ma, is ones); op(B) = B (K x N) or B^T (B is N x K).
// v_mfma_f32_16x16x4f32 lane layout: A[i][k] in lane i + 16k, B[k][j] in lane
// j + 16k, D[4(lane / 16) + e][lane % 16] in element e.  A lane (i, g) holds k =
// 4g .. 4g + 3 of a block of 16, one k per MFMA step, so an operand stored along
// k is one 16-byte load (where its rows are 16-byte aligned: wide_a, wide_b).
struct MlpGemm {
    const float *A;
    const float *B;
    float *C;
    int M;
    int N;
    int K;
    int Ma;             // rows of A^T that A holds
    int wide_a;
    int wide_b;
    const float *bias;
    float *act;         // kBiasGelu: GELU(C)
    const float *zin;   // kDGelu: Z; kMse: the targets
    float *partials;    // kMse: a sum of squares per workgroup
    float scale;        // kMse: 2 / count
};

template <bool kTA, bool kTB, int kEpi, int kSub>
__global__ __launch_bounds__(256) void mlp_gemm_kernel(MlpGemm g) {
    __shared__ float part[4][kSub * kSub][4][64];
    __shared__ float red[4];
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = t >> 6;
    const int i = lane & 15;
    const int q = lane >> 4;
    const unsigned row_tile = blockIdx.z * gridDim.y + blockIdx.y;
    const int m0 = (int)row_tile * 16 * kSub;
    const int n0 = blockIdx.x * 16 * kSub;
    if (m0 >= g.M) {
        return;
    }
    float4_t acc[kSub][kSub];
#pragma unroll
    for (int a = 0; a < kSub; ++a) {
#pragma unroll
        for (int b = 0; b < kSub; ++b) {
            acc[a][b] = (float4_t){0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    // four consecutive k of row (of the stored operand) r
    auto along_k = [](const float *p, int r, int rows, int K, int k, bool wide, float (&v)[4]) {
        if (r >= rows) {
            v[0] = v[1] = v[2] = v[3] = 0.0f;
        } else if (wide && k + 3 < K) {
            const float4 x = *reinterpret_cast<const float4 *>(p + (size_t)r * K + k);
            v[0] = x.x;
            v[1] = x.y;
            v[2] = x.z;
            v[3] = x.w;
        } else {
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                v[m] = k + m < K ? p[(size_t)r * K + k + m] : 0.0f;
            }
        }
    };
    // column c of four consecutive rows k
    auto down_k = [](const float *p, int c, int cols, int K, int k, float (&v)[4]) {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            v[m] = (c < cols && k + m < K) ? p[(size_t)(k + m) * cols + c] : 0.0f;
        }
    };
#pragma unroll 2
    for (int k0 = 16 * wave; k0 < g.K; k0 += 64) {
        const int k = k0 + 4 * q;
        float fa[kSub][4];
        float fb[kSub][4];
#pragma unroll
        for (int s = 0; s < kSub; ++s) {
            const int row = m0 + 16 * s + i;
            const int col = n0 + 16 * s + i;
            if constexpr (kTA) {
                down_k(g.A, row, g.Ma, g.K, k, fa[s]);
                if (row == g.Ma) {
#pragma unroll
                    for (int m = 0; m < 4; ++m) {
                        fa[s][m] = k + m < g.K ? 1.0f : 0.0f;
                    }
                }
            } else {
                along_k(g.A, row, g.M, g.K, k, g.wide_a != 0, fa[s]);
            }
            if constexpr (kTB) {
                along_k(g.B, col, g.N, g.K, k, g.wide_b != 0, fb[s]);
            } else {
                down_k(g.B, col, g.N, g.K, k, fb[s]);
            }
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) {
#pragma unroll
            for (int a = 0; a < kSub; ++a) {
#pragma unroll
                for (int b = 0; b < kSub; ++b) {
                    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[a][m], fb[b][m],
                                                                     acc[a][b], 0, 0, 0);
                }
            }
        }
    }
#pragma unroll
    for (int s = 0; s < kSub * kSub; ++s) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            part[wave][s][e][lane] = acc[s / kSub][s % kSub][e];
        }
    }
    __syncthreads();
    float squares = 0.0f;
#pragma unroll
    for (int s = 0; s < kSub * kSub; ++s) {
        // wave w finishes element w of every lane
        const int e = wave;
        float v = (part[0][s][e][lane] + part[1][s][e][lane]) +
                  (part[2][s][e][lane] + part[3][s][e][lane]);
        const int gm = m0 + 16 * (s / kSub) + 4 * q + e;
        const int gn = n0 + 16 * (s % kSub) + i;
        if (gm >= g.M || gn >= g.N) {
            continue;
        }
        const size_t o = (size_t)gm * g.N + gn;
        if (kEpi == kMlpEpiBias || kEpi == kMlpEpiBiasGelu || kEpi == kMlpEpiMse) {
            v += g.bias[gn];
        }
        if (kEpi == kMlpEpiDGelu) {
            v *= gelu_grad(g.zin[o]);
        }
        if (kEpi == kMlpEpiMse) {
            const float d = v - g.zin[o];
            squares += d * d;
            v = g.scale * d;
        }
        g.C[o] = v;
        if (kEpi == kMlpEpiBiasGelu) {
            g.act[o] = gelu(v);
        }
    }
    if constexpr (kEpi == kMlpEpiMse) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            squares += __shfl_xor(squares, off, 64);
        }
        if (lane == 0) {
            red[wave] = squares;
        }
        __syncthreads();
        if (t == 0) {
            g.partials[row_tile * gridDim.x + blockIdx.x] =
                (red[0] + red[1]) + (red[2] + red[3]);
        }
    }
}

// loss = sum of the workgroups' squares / count, in a fixed order.
__global__ __launch_bounds__(256) void mlp_loss_kernel(const float *__restrict__ partials, int n,
                                                       long long count,
                                                       float *__restrict__ loss_out) {
    __shared__ float red[4];
    float acc = 0.0f;
    for (int i = threadIdx.x; i < n; i += 256) {
        acc += partials[i];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        acc += __shfl_xor(acc, off, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        red[threadIdx.x >> 6] = acc;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        loss_out[0] = ((red[0] + red[1]) + (red[2] + red[3])) / (float)count;
    }
}

namespace {

template <bool kTA, bool kTB, int kEpi>
void gemm(const MlpGemm &g, hipStream_t s) {
    const MlpGrid shape = mlp_grid(g.M, g.N);
    const dim3 grid(shape.x, shape.y, shape.z);
    if (shape.sub == 2) {
        mlp_gemm_kernel<kTA, kTB, kEpi, 2><<<grid, 256, 0, s>>>(g);
    } else {
        mlp_gemm_kernel<kTA, kTB, kEpi, 1><<<grid, 256, 0, s>>>(g);
    }
}

bool wide_rows(const float *p, int ld) {
    return ld % 4 == 0 && reinterpret_cast<uintptr_t>(p) % 16 == 0;
}

}  // namespace

void launch_mlp_forward(const float *X, const float *W, const float *bias, float *Z, float *act,
                        int rows, int cols, int K, hipStream_t s) {
    MlpGemm g{X, W, Z, rows, cols, K, 0, wide_rows(X, K), 0, bias, act, nullptr, nullptr, 0.0f};
    if (act != nullptr) {
        gemm<false, false, kMlpEpiBiasGelu>(g, s);
    } else {
        gemm<false, false, kMlpEpiBias>(g, s);
    }
}

void launch_mlp_output_loss(const float *X, const float *W, const float *bias, const float *T,
                            float *dY, int rows, int cols, int K, float *partials,
                            float *loss_out, hipStream_t s) {
    const long long count = mlp_elements(rows, cols);
    MlpGemm g{X, W, dY, rows, cols, K, 0, wide_rows(X, K), 0, bias, nullptr, T, partials,
              2.0f / (float)count};
    gemm<false, false, kMlpEpiMse>(g, s);
    const MlpGrid grid = mlp_grid(rows, cols);
    mlp_loss_kernel<<<1, 256, 0, s>>>(partials, (int)(grid.rows * grid.x), count, loss_out);
}

void launch_mlp_backward_data(const float *dY, const float *W, const float *Z, float *dZ, int rows,
                              int cols, int K, hipStream_t s) {
    MlpGemm g{dY, W, dZ, rows, cols, K, 0, wide_rows(dY, K), wide_rows(W, K), nullptr, nullptr, Z,
              nullptr, 0.0f};
    gemm<false, true, kMlpEpiDGelu>(g, s);
}

void launch_mlp_backward_weights(const float *X, const float *dY, float *dWb, int in, int cols,
                                 int rows, hipStream_t s) {
    MlpGemm g{X, dY, dWb, in + 1, cols, rows, in, 0, 0, nullptr, nullptr, nullptr, nullptr, 0.0f};
    gemm<true, false, kMlpEpiNone>(g, s);
}

// Adam on the packed FP32 parameters (torch.optim.Adam arithmetic), step t.
__global__ void mlp_adam_kernel(float *__restrict__ p, const float *__restrict__ g,
                                float *__restrict__ m, float *__restrict__ v, int count, float lr,
                                float b1, float b2, float eps, int t) {
    const float bc1 = 1.0f - powf(b1, (float)t);
    const float bc2 = 1.0f - powf(b2, (float)t);
    const float step_size = lr / bc1;
    const float bc2_sqrt = sqrtf(bc2);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.0f - b1) * gi;
        const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        p[i] = p[i] - step_size * (mi / (sqrtf(vi) / bc2_sqrt + eps));
    }
}

void launch_mlp_adam(float *p, const float *g, float *m, float *v, int count, float lr, float b1,
                     float b2, float eps, int t, hipStream_t s) {
    const int blocks = (count + 255) / 256;
    mlp_adam_kernel<<<blocks < 1024 ? blocks : 1024, 256, 0, s>>>(p, g, m, v, count, lr, b1, b2,
                                                                  eps, t);
}

}  // namespace rie
