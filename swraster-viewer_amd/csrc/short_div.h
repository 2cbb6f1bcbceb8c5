// short_div.h -- divisions and square roots with fewer instructions than the
// compiler's (which scale their operands and fix up every special case), for
// operands known to be in range: each gives the IEEE result.  The corrections
// are Markstein's: a fused residual of the hardware's approximation, then a
// fused step that rounds once.
//
// sr_check_short_forms (short_div.hip) compares them on the device with IEEE
// division and square root: the reciprocal, the root, and both in turn for
// every float in [2^-96, 2^96], the quotient for seeded random pairs (1.7e10
// of them in the widest run).
#pragma once

#include <hip/hip_runtime.h>

namespace sr {

// 1 / b for b in [2^-96, 2^96].
__device__ __forceinline__ float rcp_in_range(float b) {
    float y = __builtin_amdgcn_rcpf(b);
    return fmaf(fmaf(-b, y, 1.0f), y, y);
}
// 1 / b for any b.  (The 1/w that a sample interpolates is between its
// vertices' only inside the triangle; covered samples of a triangle whose
// integer edge constants wrap lie anywhere, and it can be zero there.)
__device__ __forceinline__ float rcp_ieee(float b) {
    if (b >= 0x1p-96f && b <= 0x1p96f) return rcp_in_range(b);
    return 1.0f / b;
}
// a / b from y = rcp(b), correctly rounded: with the correctly rounded
// reciprocal of b, one fused correction of a y by its exact residual.  That
// holds while neither the quotient nor the residual leaves the floats' range:
// for b within 2^+-40, while a is a zero or within 2^+-80.
__device__ __forceinline__ float div_by_rcp(float a, float b, float y) {
    float q = a * y;
    return fmaf(fmaf(-b, q, a), y, q);
}
__device__ __forceinline__ float div_in_range(float a, float b) { return div_by_rcp(a, b, rcp_in_range(b)); }
// 1 / sqrt(x), each rounded.  SHORT: with the short forms where x is in range.
template <bool SHORT = true> __device__ __forceinline__ float rsqrt_ieee(float x) {
    if (SHORT && x >= 0x1p-96f && x <= 0x1p96f) {
        float y = __builtin_amdgcn_rsqf(x), g = x * y;
        return rcp_in_range(fmaf(fmaf(-g, g, x), 0.5f * y, g));
    }
    return 1.0f / sqrtf(x);
}

}  // namespace sr
