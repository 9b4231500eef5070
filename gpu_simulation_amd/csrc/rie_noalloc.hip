// Allocation-free energy_and_grad for small circuits (structured_adjoint,
// 2 <= n <= 14), for callers that cannot allocate device memory: code under
// HIP graph capture, tight serving loops, harnesses that forbid hipMalloc.
//
// The whole circuit runs in one workgroup: psi and lambda in registers for
// n <= 13, for n = 14 the adjoint sweep in two halves through a global scratch
// (rie_regcircuit.hip).  Everything beyond the caller's inputs and outputs -- the
// layers' records, and at n = 14 the state and that scratch -- lives in the
// file-scope array `scratch` below, one copy per device, held until the process
// ends.  Its address on each device comes from hipGetSymbolAddress once per
// device (with that device current) and is the only form in which host code
// hands it to kernels.
//
// Every call on a device shares that device's array: calls that overlap on
// one device (different streams, or different host threads) race.  Nothing
// in it needs to start at zero: the records kernel writes every entry the
// circuit reads, and the circuit kernels write the states they read.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>

#include "rie.h"
#include "rie_engine_internal.hpp"
#include "rie_kernels.hpp"

namespace rie {
namespace {

constexpr size_t kNoAllocMaxQubits = RIE_NOALLOC_MAX_QUBITS;
constexpr size_t kNoAllocMaxLayers = RIE_NOALLOC_MAX_LAYERS;
static_assert(kNoAllocMaxQubits <= (size_t)kBatchMaxQubits, "the whole-circuit kernel's limit");
constexpr size_t kRecordBytes = 1024 * kNoAllocMaxLayers;  // at most 1 KB a layer
constexpr size_t kStateBytes = sizeof(double2) * (size_t{1} << kNoAllocMaxQubits);
constexpr size_t kScratchBytes = kRecordBytes + kStateBytes + sizeof(double2) * kReg14Scratch;
static_assert(kScratchBytes == RIE_NOALLOC_SCRATCH_BYTES, "the size the header states");

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
unsigned char *g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device, looked up on the
// device's first call.
unsigned char *device_scratch() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        fail(RIE_DEVICE_ERROR, "no current HIP device");
    }
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void *ptr = nullptr;
        const hipError_t err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (err != hipSuccess || ptr == nullptr) {
            fail(RIE_DEVICE_ERROR, std::string("hipGetSymbolAddress(scratch): ") +
                                       hipGetErrorString(err));
        }
        g_scratch_ptr[dev] = static_cast<unsigned char *>(ptr);
    }
    return g_scratch_ptr[dev];
}

}  // namespace
}  // namespace rie

rie_status rie_energy_and_grad_noalloc(size_t num_qubits, size_t num_layers, double field,
                                       const double *params_device, size_t num_params,
                                       size_t structured_rotation_chunk_width,
                                       double *energy_device, double *gradient_device,
                                       void *stream_handle) {
    using namespace rie;
    return guard([&]() {
        if (num_qubits < 2 || num_qubits > kNoAllocMaxQubits) {
            fail(RIE_INVALID_ARGUMENT, "the allocation-free entry point takes 2 <= num_qubits <= " +
                                           std::to_string(kNoAllocMaxQubits) + ".");
        }
        if (num_layers < 1 || num_layers > kNoAllocMaxLayers) {
            fail(RIE_INVALID_ARGUMENT, "the allocation-free entry point takes 1 <= num_layers <= " +
                                           std::to_string(kNoAllocMaxLayers) + ".");
        }
        if (num_params != 2 * num_qubits * num_layers) {
            fail(RIE_INVALID_ARGUMENT, "num_params does not match the circuit.");
        }
        if (structured_rotation_chunk_width < 1 || structured_rotation_chunk_width > 8) {
            fail(RIE_INVALID_ARGUMENT, "structured_rotation_chunk_width must be in [1, 8].");
        }
        if (!std::isfinite(field)) {
            fail(RIE_INVALID_ARGUMENT, "field must be finite.");
        }
        if (params_device == nullptr || energy_device == nullptr) {
            fail(RIE_INVALID_ARGUMENT, "params and energy must be device pointers.");
        }
        const hipStream_t stream = static_cast<hipStream_t>(stream_handle);
        unsigned char *base = device_scratch();
        const int n = (int)num_qubits;
        const int layers = (int)num_layers;
        if (circuit_record_bytes(n, layers) > kRecordBytes) {
            fail(RIE_DEVICE_ERROR, "internal: records exceed the scratch");
        }
        double *rec = reinterpret_cast<double *>(base);
        launch_circuit_records(nullptr, RecordJob{params_device, rec, n, 0}, nullptr, layers,
                               stream);
        RegJob job{};
        job.rec = rec;
        job.energy = energy_device;
        job.grad = gradient_device;  // nullptr: energy only
        job.field = field;
        job.layers = layers;
        if (n <= kRegMaxQubits) {
            launch_regcircuit(n, nullptr, job, 1, stream);
        } else {
            double2 *psi = reinterpret_cast<double2 *>(base + kRecordBytes);
            launch_reg14(nullptr, Reg14Job{job, psi}, nullptr, nullptr, 1, 1,
                         psi + (size_t{1} << kNoAllocMaxQubits), stream);
        }
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) {
            fail(RIE_DEVICE_ERROR, std::string("allocation-free launch: ") + hipGetErrorString(err));
        }
    });
}
