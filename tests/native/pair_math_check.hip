// Checks of the pair kernels' arithmetic (device_math.hpp) against the same
// expressions with the compiler's square root and division, for every float
// squared distance of a range. Built by physica_amd.build into
// tests/native/libphx_pair_math_check.so and driven from
// tests/test_pair_math.py.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "device_math.hpp"

namespace phx {
PbfKernel pbf_kernel(float h);
KernelConstants kernel_constants(float h);
}  // namespace phx

namespace {

using namespace phx;

__device__ bool same(float a, float b) {
    return __float_as_uint(a) == __float_as_uint(b) || (a == 0.0F && b == 0.0F);
}

// [0] poly6_value, [1] spiky_factor, [2] cubic_gradient_factor<true>, [3] cubic_value
__global__ void __launch_bounds__(256)
    pair_check_kernel(uint32_t first, uint32_t count, PbfKernel k, KernelConstants c, unsigned long long* wrong) {
    const uint32_t stride = gridDim.x * blockDim.x;
    unsigned long long bad[4] = {0, 0, 0, 0};
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < count; t += stride) {
        const float d2 = __uint_as_float(first + t);
        const float h = k.h;
        const float diff = h * h - d2;
        const float w = d2 >= h * h ? 0.0F : 315.0F * diff * diff * diff / k.poly6;
        bad[0] += same(poly6_value(d2, k), w) && poly6_vanishes(d2, k) == (w == 0.0F) ? 0u : 1u;
        const float dist = sqrtf(d2);
        const float gap = h - dist;
        const float s = dist == 0.0F || dist >= h ? 0.0F : k.spiky * gap * gap / dist;
        bad[1] += same(spiky_factor(d2, k), s) ? 0u : 1u;
        const float q = dist / h;
        const float deriv = q <= 0.5F ? 18.0F * q * q - 12.0F * q : -6.0F * (1.0F - q) * (1.0F - q);
        const float f = dist == 0.0F || dist >= h ? 0.0F : c.cubic * deriv / (h * dist);
        bad[2] += same(cubic_gradient_factor<true>(sqrt_rn(d2), c), f) ? 0u : 1u;
        const float v = dist >= h ? 0.0F
                        : q <= 0.5F ? c.cubic * (6.0F * q * q * q - 6.0F * q * q + 1.0F)
                                    : c.cubic * 2.0F * (1.0F - q) * (1.0F - q) * (1.0F - q);
        bad[3] += same(cubic_value(sqrt_rn(d2), c), v) ? 0u : 1u;
    }
    for (int i = 0; i < 4; ++i)
        if (bad[i] != 0u) atomicAdd(wrong + i, bad[i]);
}

// over_rest(x, rest) against x / rest, x the only mass of the step
__global__ void __launch_bounds__(256)
    rest_check_kernel(uint32_t first, uint32_t count, float rest, unsigned long long* wrong) {
    const uint32_t stride = gridDim.x * blockDim.x;
    unsigned long long bad = 0;
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < count; t += stride) {
        const float x = __uint_as_float(first + t);
        const RestDensity density = rest_density_of(rest, outside_quick_range(x));
        bad += same(over_rest(x, density), x / rest) ? 0u : 1u;
    }
    if (bad != 0u) atomicAdd(wrong, bad);
}

// Counts mismatches on the device: launch(counter) starts the check.
template <class Launch>
int count_mismatches(uint32_t first, uint32_t count, unsigned long long* mismatches, int counters, Launch&& launch) {
    if (mismatches == nullptr || count == 0u || first + (count - 1u) < first) return static_cast<int>(hipErrorInvalidValue);
    unsigned long long* device = nullptr;
    const size_t bytes = static_cast<size_t>(counters) * sizeof(unsigned long long);
    hipError_t e = hipMalloc(&device, bytes);
    if (e != hipSuccess) return static_cast<int>(e);
    e = hipMemset(device, 0, bytes);
    if (e == hipSuccess) {
        launch(device);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(mismatches, device, bytes, hipMemcpyDeviceToHost);
    const hipError_t f = hipFree(device);
    return static_cast<int>(e != hipSuccess ? e : f);
}

}  // namespace

// Mismatches of the four functions over the floats with bit patterns
// [first, first + count); returns a hipError_t.
extern "C" int phx_test_pair_math(float h, uint32_t first, uint32_t count, unsigned long long* mismatches) {
    return count_mismatches(first, count, mismatches, 4, [&](unsigned long long* wrong) {
        pair_check_kernel<<<4096, 256>>>(first, count, phx::pbf_kernel(h), phx::kernel_constants(h), wrong);
    });
}

// Mismatches of over_rest for the masses with bit patterns
// [first, first + count) over the rest density `rest`; returns a hipError_t.
extern "C" int phx_test_over_rest(float rest, uint32_t first, uint32_t count, unsigned long long* mismatches) {
    return count_mismatches(first, count, mismatches, 1, [&](unsigned long long* wrong) {
        rest_check_kernel<<<4096, 256>>>(first, count, rest, wrong);
    });
}
