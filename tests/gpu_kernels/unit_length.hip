// Test-only kernels: inv_unit_length and div_rn_normal of hvx_device.h against
// the compiler's IEEE square root and divisions. Built into
// tests/_build/libhvx_testkernels.so.
#include <hip/hip_runtime.h>

#include "../../hellovulkan_amd/csrc/hvx_device.h"

namespace {
__global__ void unit_kernel(uint32_t first_bits, uint32_t n, unsigned long long* mismatches) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float x = hvx::u2f(first_bits + i);
    if (hvx::f2u(hvx::inv_unit_length(x)) != hvx::f2u(1.0f / hvx::sqrtf_(x))) atomicAdd(mismatches, 1ull);
}
__global__ void div_kernel(const float* a, const float* b, uint32_t n, unsigned long long* mismatches) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (hvx::f2u(hvx::div_rn_normal(a[i], b[i])) != hvx::f2u(a[i] / b[i])) atomicAdd(mismatches, 1ull);
}
}  // namespace

extern "C" int hvxt_unit_length_check(uint32_t first_bits, uint32_t n, unsigned long long* d_mismatches) {
    hipLaunchKernelGGL(unit_kernel, dim3((n + 255) / 256), dim3(256), 0, 0, first_bits, n, d_mismatches);
    return (int)hipGetLastError();
}
extern "C" int hvxt_div_check(const float* d_a, const float* d_b, uint32_t n, unsigned long long* d_mismatches) {
    hipLaunchKernelGGL(div_kernel, dim3((n + 255) / 256), dim3(256), 0, 0, d_a, d_b, n, d_mismatches);
    return (int)hipGetLastError();
}
