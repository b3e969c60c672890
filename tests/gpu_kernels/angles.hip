// Test-only kernels: atan2f_rn and acosf_rn of hvx_device.h against atan2f_ and
// acosf_ of hvx_math.h. Built into tests/_build/libhvx_testkernels.so.
#include <hip/hip_runtime.h>

#include "../../hellovulkan_amd/csrc/hvx_device.h"

namespace {
__global__ void angles_kernel(const float* y, const float* x, uint32_t n, unsigned long long* mismatches) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    auto differ = [](float a, float b) { return hvx::f2u(a) != hvx::f2u(b) && !(a != a && b != b); };
    if (differ(hvx::atan2f_rn(y[i], x[i]), hvx::atan2f_(y[i], x[i]))) atomicAdd(mismatches, 1ull);
    if (differ(hvx::acosf_rn(x[i]), hvx::acosf_(x[i]))) atomicAdd(mismatches + 1, 1ull);
}
}  // namespace

extern "C" int hvxt_angles_check(const float* d_y, const float* d_x, uint32_t n, unsigned long long* d_mismatches) {
    hipLaunchKernelGGL(angles_kernel, dim3((n + 255) / 256), dim3(256), 0, 0, d_y, d_x, n, d_mismatches);
    return (int)hipGetLastError();
}
