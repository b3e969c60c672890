// Test-only kernel: repeat_sum of hvx_math.h against the additions one by one.
// Built into tests/_build/libhvx_testkernels.so.
#include <hip/hip_runtime.h>

#include "../../hellovulkan_amd/csrc/hvx_math.h"

namespace {
__global__ void repeat_kernel(const uint32_t* terms, const uint32_t* counts, uint32_t n, unsigned long long* mismatches) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float t = hvx::u2f(terms[i]);
    float a = 0.0f;
    for (uint32_t k = 0; k < counts[i]; ++k) a = a + t;
    const float r = hvx::repeat_sum(t, counts[i]);
    if (hvx::f2u(r) != hvx::f2u(a) && !(r != r && a != a)) atomicAdd(mismatches, 1ull);
}
}  // namespace

extern "C" int hvxt_repeat_sum_check(const uint32_t* d_terms, const uint32_t* d_counts, uint32_t n,
                                     unsigned long long* d_mismatches) {
    hipLaunchKernelGGL(repeat_kernel, dim3((n + 255) / 256), dim3(256), 0, 0, d_terms, d_counts, n, d_mismatches);
    return (int)hipGetLastError();
}
