// short_div.hip -- sr_check_short_forms: the short divisions and roots of
// short_div.h against the compiler's IEEE ones, on the device.

#include <hip/hip_runtime.h>

#include <cstring>

#include "common.h"
#include "runtime.h"
#include "short_div.h"
#include "swraster.h"

namespace sr {
namespace {

constexpr uint32_t LOW = (127u - 96u) << 23, FLOATS = (192u << 23) + 1u;      // the floats in [2^-96, 2^96]

__device__ __forceinline__ uint64_t mix(uint64_t x) {         // splitmix64
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

__device__ __forceinline__ bool differ(float a, float b) { return __float_as_uint(a) != __float_as_uint(b); }

// bad: mismatches of the reciprocal, of 1 / sqrt and of the quotient.
__global__ void __launch_bounds__(256) k_check_short(uint64_t seed, uint64_t pairs, unsigned long long *bad) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x, i0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t n[3] = {0u, 0u, 0u};
    for (uint64_t i = i0; i < FLOATS; i += stride) {
        const float x = __uint_as_float(LOW + (uint32_t)i);
        n[0] += differ(rcp_ieee(x), 1.0f / x);
        n[1] += differ(rsqrt_ieee<true>(x), rsqrt_ieee<false>(x));
    }
    for (uint64_t i = i0; i < pairs; i += stride) {
        const uint64_t r = mix(seed + i), q = mix(r);
        auto operand = [](uint64_t bits) {         // any sign and mantissa, exponent within +-40
            const uint32_t e = 87u + (uint32_t)((bits >> 32) % 81u);
            return __uint_as_float(((uint32_t)bits & 0x807FFFFFu) | (e << 23));
        };
        const float a = operand(r), b = fabsf(operand(q));
        n[2] += differ(div_in_range(a, b), a / b);
    }
    for (int k = 0; k < 3; k++)
        if (n[k]) atomicAdd(&bad[k], (unsigned long long)n[k]);
}

}  // namespace
}  // namespace sr

using namespace sr;

extern "C" SR_API int sr_check_short_forms(int32_t device, uint64_t seed, uint64_t pairs, uint64_t mismatches[3]) {
    if (!mismatches) return fail(SR_ERR_INVALID_ARGUMENT, "null argument");
    if (hipSetDevice(device) != hipSuccess) return fail(SR_ERR_HIP, "device %d", device);
    unsigned long long *bad = nullptr, out[3] = {0, 0, 0};
    hipError_t e = hipMalloc((void **)&bad, sizeof(out));
    if (e == hipSuccess) e = hipMemcpy(bad, out, sizeof(out), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_check_short, dim3(4096), dim3(256), 0, nullptr, seed, pairs, bad);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(out, bad, sizeof(out), hipMemcpyDeviceToHost);
    if (bad) (void)hipFree(bad);
    if (e != hipSuccess) return fail(SR_ERR_HIP, "short forms: %s", hipGetErrorString(e));
    for (int k = 0; k < 3; k++) mismatches[k] = out[k];
    return SR_OK;
}
