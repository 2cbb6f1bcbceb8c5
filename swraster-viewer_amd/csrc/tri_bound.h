// tri_bound.h -- a depth that no covered sample of a snapped triangle goes
// below, from the triangle's vertices (setup, kernels.hip).  Plain C++ for the
// host compiler too, which the CPU tests use.
#pragma once

#include <math.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define SR_BOUND_FN __host__ __device__ __forceinline__
#else
#define SR_BOUND_FN inline
#endif

namespace sr {

// How far b1 + b2 of a covered sample can go above 1 (the triangle's own
// points have b1, b2 >= 0 and b1 + b2 <= 1, and coverage keeps the first two),
// or infinity where the integer edge constants can wrap.
//
// An edge value is (A X + B Y) + C in f32 at the walk's origin, with the i32
// edge constants converted, and up to 14 steps added to it: each rounding is
// off by u = 2^-24 of the rounded magnitude at most.  With w and h the extents
// of the triangle and X, Y the largest coordinates of its vertices and samples
// (samples reach 24 sub-pixels beyond the box), |A| <= h and |B| <= w, the
// terms and C are at most P = h X + w Y, and the edge function itself is at
// most Q = h (w + 32) + w (h + 32) over the walked samples; so a value is off
// by M = u (4 P + 16 Q) at most.  The three edge functions add up to the area,
// less the fill-rule biases, and a covered sample has the first at -M or more,
// so the other two add up to the area + 3 M at most; the reciprocal of the
// area, the products and their sum add less than 4e-7.  P also bounds the
// unwrapped constants and the area (P >= w h), so nothing wraps below 2^31.
// A compact 70-px triangle in the far corner of a 4K frame has 1e-4, a
// pixel-thin one across it 0.1 and more.
SR_BOUND_FN float bary_excess(const int32_t px[3], const int32_t py[3], float ooa) {
    const float x0 = (float)px[0], x1 = (float)px[1], x2 = (float)px[2];
    const float y0 = (float)py[0], y1 = (float)py[1], y2 = (float)py[2];
    const float xl = fminf(x0, fminf(x1, x2)), xh = fmaxf(x0, fmaxf(x1, x2));
    const float yl = fminf(y0, fminf(y1, y2)), yh = fmaxf(y0, fmaxf(y1, y2));
    const float w = xh - xl, h = yh - yl;
    const float X = fmaxf(fabsf(xl), fabsf(xh)) + 32.0f, Y = fmaxf(fabsf(yl), fabsf(yh)) + 32.0f;
    const float P = h * X + w * Y, Q = h * (w + 32.0f) + w * (h + 32.0f);
    if (!(P < 2.14e9f) || !(fmaxf(w, h) < 0x1p24f)) return INFINITY;
    return 4e-7f + (3.0f * 0x1p-24f) * ((4.0f * P + 16.0f * Q) * ooa);
}

// A depth that no covered sample's goes below, from the vertices' z/w (1/w)
// and 1/w; false if there is none to give.
//
// The depth is ((za + b1 zda) + b2 zdb) / ((oa + b1 oda) + b2 odb), a ratio of
// affine functions of the barycentrics.  Inside the triangle it lies between
// its values z0, z1, z2 at the vertices (the denominator keeps its sign).  A
// sample beyond the edge opposite vertex 0 is (1 + t) p for a point p of that
// edge and t <= e, the excess above; its depth differs from p's by
// t D0 (z(p) - z0) / D, D0 and D the denominators there, and D is at least
// (1 - (r - 1) t) times the vertices' smallest, r the ratio of their largest
// and smallest.  With r e <= 1/4 that is below 2 r e (zmax - zmin).  The
// operations round: with r <= 16 numerator, denominator and quotient are
// together off by less than 8e-5 of the largest vertex depth, and the vertex
// depths here (hardware reciprocal) by an ulp, within 1e-4 of it.
SR_BOUND_FN bool tri_zmin(const int32_t px[3], const int32_t py[3], float ooa, const float zow[3], const float oow[3],
                          float &lo) {
    const float dmin = fminf(oow[0], fminf(oow[1], oow[2])), dmax = fmaxf(oow[0], fmaxf(oow[1], oow[2]));
    if (!(dmin > 1e-30f) || !(dmax < 1e30f) || !(dmax <= 16.0f * dmin)) return false;
#if defined(__HIP_DEVICE_COMPILE__)
    const float z0 = zow[0] * __builtin_amdgcn_rcpf(oow[0]), z1 = zow[1] * __builtin_amdgcn_rcpf(oow[1]);
    const float z2 = zow[2] * __builtin_amdgcn_rcpf(oow[2]), r = dmax * __builtin_amdgcn_rcpf(dmin);
#else
    const float z0 = zow[0] * (1.0f / oow[0]), z1 = zow[1] * (1.0f / oow[1]);
    const float z2 = zow[2] * (1.0f / oow[2]), r = dmax * (1.0f / dmin);
#endif
    const float re = r * bary_excess(px, py, ooa);
    const float zabs = fmaxf(fabsf(z0), fmaxf(fabsf(z1), fabsf(z2)));
    if (!(z0 == z0 && z1 == z1 && z2 == z2) || !(zabs < 1e30f) || !(re <= 0.25f)) return false;
    const float zmin = fminf(z0, fminf(z1, z2)), zmax = fmaxf(z0, fmaxf(z1, z2));
    lo = zmin - (2.0f * re * (zmax - zmin) + zabs * 1e-4f + 1e-30f);
    return true;
}

}  // namespace sr
