// Every float of [2^-96, 2^60): the short square root and reciprocal of the tile passes against sqrtf and 1 / x (correctly
// rounded with the flags that the library is built with).  Built as tests/libarith_check.so for the test beside it.
#include "wc_arith.hpp"

namespace {

constexpr uint32_t kFirst = (127u - 96u) << 23, kLast = (127u + 60u) << 23;  // bits of 2^-96 and 2^60

__global__ __launch_bounds__(256) void k_compare(unsigned long long* bad) {
    const uint32_t stride = gridDim.x * 256u;
    uint32_t roots = 0, reciprocals = 0;
    for (uint32_t u = kFirst + blockIdx.x * 256u + threadIdx.x; u < kLast; u += stride) {
        const float x = __uint_as_float(u);
        roots += __float_as_uint(wc::sqrt_in_range(x)) != __float_as_uint(sqrtf(x)) ? 1u : 0u;
        reciprocals += __float_as_uint(wc::rcp_in_range(x)) != __float_as_uint(1.0f / x) ? 1u : 0u;
        reciprocals += __float_as_uint(wc::rcp_in_range(-x)) != __float_as_uint(1.0f / -x) ? 1u : 0u;
    }
    if (roots) atomicAdd(&bad[0], (unsigned long long)roots);
    if (reciprocals) atomicAdd(&bad[1], (unsigned long long)reciprocals);
}

// the given values' square roots and reciprocals
__global__ __launch_bounds__(256) void k_values(const float* x, float* root, float* reciprocal, uint32_t n) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    root[i] = wc::sqrt_in_range(x[i]);
    reciprocal[i] = wc::rcp_in_range(x[i]);
}

}  // namespace

// Values compared, and the numbers of square roots and of reciprocals (of both signs) that differ.
extern "C" int arith_compare(unsigned long long* values, unsigned long long* roots, unsigned long long* reciprocals) {
    unsigned long long *bad = nullptr, host[2] = {0, 0};
    if (hipMalloc(&bad, sizeof(host)) != hipSuccess) return 1;
    bool ok = hipMemcpy(bad, host, sizeof(host), hipMemcpyHostToDevice) == hipSuccess;
    if (ok) hipLaunchKernelGGL(k_compare, dim3(8192), dim3(256), 0, 0, bad);
    ok = ok && hipGetLastError() == hipSuccess && hipMemcpy(host, bad, sizeof(host), hipMemcpyDeviceToHost) == hipSuccess;
    (void)hipFree(bad);
    *values = kLast - kFirst;
    *roots = host[0];
    *reciprocals = host[1];
    return ok ? 0 : 1;
}

extern "C" int arith_values(const float* x, float* root, float* reciprocal, uint32_t n) {
    float* d = nullptr;
    if (n == 0 || hipMalloc(&d, (size_t)n * 12) != hipSuccess) return 1;
    bool ok = hipMemcpy(d, x, (size_t)n * 4, hipMemcpyHostToDevice) == hipSuccess;
    if (ok) hipLaunchKernelGGL(k_values, dim3((n + 255) / 256), dim3(256), 0, 0, d, d + n, d + 2 * (size_t)n, n);
    ok = ok && hipGetLastError() == hipSuccess &&
         hipMemcpy(root, d + n, (size_t)n * 4, hipMemcpyDeviceToHost) == hipSuccess &&
         hipMemcpy(reciprocal, d + 2 * (size_t)n, (size_t)n * 4, hipMemcpyDeviceToHost) == hipSuccess;
    (void)hipFree(d);
    return ok ? 0 : 1;
}
