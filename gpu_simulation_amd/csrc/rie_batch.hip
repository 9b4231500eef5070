// Optimizer-step kernels of a batch (the circuits themselves: rie_regcircuit.hip,
// rie_dense.hip).
#include <hip/hip_runtime.h>

#include "rie_kernels.hpp"

namespace rie {

// ---------------------------------------------------------------------------
// Optimizer steps over a packed parameter array.
// ---------------------------------------------------------------------------

__global__ void gd_update_kernel(double *__restrict__ p, const double *__restrict__ g,
                                 uint64_t count, double lr) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) {
        p[i] = p[i] - lr * g[i];
    }
}

// Adam as torch.optim.Adam computes it (no weight decay, no amsgrad):
// m = b1 m + (1 - b1) g; v = b2 v + (1 - b2) g^2;
// p -= (lr / (1 - b1^t)) * m / (sqrt(v) / sqrt(1 - b2^t) + eps), t = step + 1.
__global__ void adam_update_kernel(double *__restrict__ p, const double *__restrict__ g,
                                   double *__restrict__ m, double *__restrict__ v, uint64_t count,
                                   double lr, double b1, double b2, double eps,
                                   const int *__restrict__ step) {
    const double tt = (double)(*step + 1);
    const double bc1 = 1.0 - pow(b1, tt);
    const double bc2 = 1.0 - pow(b2, tt);
    const double step_size = lr / bc1;
    const double bc2_sqrt = sqrt(bc2);
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) {
        const double gi = g[i];
        const double mi = b1 * m[i] + (1.0 - b1) * gi;
        const double vi = b2 * v[i] + (1.0 - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        const double denom = sqrt(vi) / bc2_sqrt + eps;
        p[i] = p[i] - step_size * (mi / denom);
    }
}

// history[step][j] = energies[j] while step < capacity.
__global__ void record_energies_kernel(const double *__restrict__ energies, int count,
                                       double *__restrict__ history, const int *__restrict__ step,
                                       int capacity) {
    const int s = *step;
    if (s >= capacity) {
        return;
    }
    for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < count; j += gridDim.x * blockDim.x) {
        history[(size_t)s * count + j] = energies[j];
    }
}

__global__ void step_advance_kernel(int *__restrict__ step) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        step[0] = step[0] + 1;
    }
}

__global__ void fill_kernel(double *__restrict__ p, uint64_t count, double value) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) {
        p[i] = value;
    }
}

__global__ void set_int_kernel(int *__restrict__ p, int value) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        p[0] = value;
    }
}

void launch_gd_update(double *p, const double *g, uint64_t count, double lr, hipStream_t s) {
    gd_update_kernel<<<elementwise_grid(count), 256, 0, s>>>(p, g, count, lr);
}

void launch_adam_update(double *p, const double *g, double *m, double *v, uint64_t count,
                        double lr, double b1, double b2, double eps, const int *step,
                        hipStream_t s) {
    adam_update_kernel<<<elementwise_grid(count), 256, 0, s>>>(p, g, m, v, count, lr, b1, b2, eps,
                                                               step);
}

void launch_record_energies(const double *energies, int count, double *history, const int *step,
                            int capacity, hipStream_t s) {
    const int grid = (count + 255) / 256;
    record_energies_kernel<<<grid > 0 ? grid : 1, 256, 0, s>>>(energies, count, history, step,
                                                               capacity);
}

void launch_step_advance(int *step, hipStream_t s) { step_advance_kernel<<<1, 64, 0, s>>>(step); }

void launch_fill(double *p, uint64_t count, double value, hipStream_t s) {
    fill_kernel<<<elementwise_grid(count), 256, 0, s>>>(p, count, value);
}

void launch_set_int(int *p, int value, hipStream_t s) { set_int_kernel<<<1, 64, 0, s>>>(p, value); }

}  // namespace rie
