// Walks random triangles as the reference's raster does (64-px tiles, 16-px
// blocks with their corner test, 2x2 quads, f32 edge values from the walk's
// origin by serial steps: src/tilerasterizer.rs:114-381) and compares every
// covered sample's depth with the triangle's bound (tri_bound.h).  This walk
// is written apart from the kernels'.
#include <stdlib.h>

#include <algorithm>
#include <cmath>
#include <random>

#include "tri_bound.h"

namespace {

int32_t wrap(int64_t v) { return (int32_t)(uint32_t)(uint64_t)v; }
int64_t prod(int32_t a, int32_t b) { return wrap((int64_t)a * b); }

struct Tri {
    int32_t x[3], y[3];
    float zow[3], oow[3];
};

struct Count {
    long tris, bounded, samples, below;
    double worst;                 // largest distance below the bound, relative to the depth
};

void walk(const Tri &t, int W, int H, Count &n) {
    const int32_t *x = t.x, *y = t.y;
    const int32_t area = wrap(prod(wrap((int64_t)x[1] - x[0]), wrap((int64_t)y[2] - y[0])) -
                              prod(wrap((int64_t)x[2] - x[0]), wrap((int64_t)y[1] - y[0])));
    if (area > 0) return;
    const float ooa = 1.0f / (float)(area < 0 ? wrap(-(int64_t)area) : area);
    n.tris++;
    float lo;
    if (!sr::tri_zmin(x, y, ooa, t.zow, t.oow, lo)) return;
    n.bounded++;
    float A[3], B[3], C[3], SX[3], SY[3];
    for (int e = 0; e < 3; e++) {         // edge e: from vertex e + 1 to e + 2
        const int p = (e + 1) % 3, q = (e + 2) % 3;
        const int32_t a = wrap((int64_t)y[q] - y[p]), b = wrap((int64_t)x[p] - x[q]);
        const int32_t bias = (a < 0 || (a == 0 && b > 0)) ? 0 : -1;
        const int32_t c = wrap((int64_t)wrap(prod(x[q], y[p]) - prod(x[p], y[q])) + bias);
        A[e] = (float)a;
        B[e] = (float)b;
        C[e] = (float)c;
        SX[e] = (float)wrap((int64_t)a * 32);
        SY[e] = (float)wrap((int64_t)b * 32);
    }
    const float oda = t.oow[1] - t.oow[0], odb = t.oow[2] - t.oow[0];
    const float zda = t.zow[1] - t.zow[0], zdb = t.zow[2] - t.zow[0];
    const int mnx = std::max(std::min({x[0], x[1], x[2]}), 0) >> 4, mny = std::max(std::min({y[0], y[1], y[2]}), 0) >> 4;
    const int mxx = (std::min(std::max({x[0], x[1], x[2]}), W * 16) + 16) >> 4;
    const int mxy = (std::min(std::max({y[0], y[1], y[2]}), H * 16) + 16) >> 4;
    for (int ry = mny / 64 * 64; ry < mxy; ry += 64)
        for (int rx = mnx / 64 * 64; rx < mxx; rx += 64) {
            const int x0 = std::max(mnx, rx), y0 = std::max(mny, ry), x1 = std::min(mxx, rx + 64), y1 = std::min(mxy, ry + 64);
            if (x0 >= x1 || y0 >= y1) continue;
            const bool coarse = x1 - x0 > 16 || y1 - y0 > 16;
            for (int by = y0 & ~1; by < y1; by += 16)
                for (int bx = x0 & ~1; bx < x1; bx += 16) {
                    bool out = false;
                    for (int e = 0; e < 3 && coarse; e++) {
                        float m = -INFINITY;
                        for (int k = 0; k < 4; k++) {
                            const float X = (float)(bx * 16 + (k & 1 ? 248 : 8)), Y = (float)(by * 16 + (k & 2 ? 248 : 8));
                            m = std::max(m, (A[e] * X + B[e] * Y) + C[e]);
                        }
                        out = out || m < 0.0f;
                    }
                    if (out) continue;
                    for (int s = 0; s < 4; s++) {
                        const float X = (float)(bx * 16 + 8 + 16 * (s & 1)), Y = (float)(by * 16 + 8 + 16 * (s >> 1));
                        float row[3];
                        for (int e = 0; e < 3; e++) row[e] = (A[e] * X + B[e] * Y) + C[e];
                        for (int j = 0; j < 8 && by + 2 * j < y1; j++) {
                            float v[3] = {row[0], row[1], row[2]};
                            for (int i = 0; i < 8 && bx + 2 * i < x1; i++) {
                                if (v[0] >= 0.0f && v[1] >= 0.0f && v[2] >= 0.0f) {
                                    const float b1 = v[1] * ooa, b2 = v[2] * ooa;
                                    const float w = 1.0f / ((t.oow[0] + b1 * oda) + b2 * odb);
                                    const float z = ((t.zow[0] + b1 * zda) + b2 * zdb) * w;
                                    n.samples++;
                                    if (z < lo) {
                                        n.below++;
                                        n.worst = std::max(n.worst, std::fabs((double)lo - z) / std::fabs((double)z));
                                    }
                                }
                                for (int e = 0; e < 3; e++) v[e] += SX[e];
                            }
                            for (int e = 0; e < 3; e++) row[e] += SY[e];
                        }
                    }
                }
        }
}

}  // namespace

// kind 0: slivers of up to `size` px, 0.1 to 1 px thin, every other one seen
// along its length (its short edge at one depth); 1: triangles of up to that
// radius anywhere; 2: compact ones of about that radius.  Depths differ by a
// factor of up to `ratio` over a triangle.
extern "C" void tri_bound_sweep(uint64_t seed, int count, int W, int H, int kind, double size, double ratio, Count *out) {
    std::mt19937_64 rng(seed);
    auto uni = [&](double a, double b) { return a + (b - a) * (double)(rng() >> 11) * 0x1p-53; };
    for (int k = 0; k < count; k++) {
        Tri t;
        double cx = uni(0, W), cy = uni(0, H), an = uni(0, 2 * M_PI);
        for (int v = 0; v < 3; v++) {
            double px, py;
            if (kind == 0) {
                const double along = v == 0 ? -0.5 : 0.5, len = size * (v < 2 ? 1.0 : uni(0.98, 1.0));
                px = cx + along * len * cos(an) - (v == 2 ? uni(0.1, 1.0) : 0.0) * sin(an);
                py = cy + along * len * sin(an) + (v == 2 ? uni(0.1, 1.0) : 0.0) * cos(an);
            } else {
                const double a = kind == 1 ? uni(0, 2 * M_PI) : an + v * 2.1 + uni(-0.4, 0.4);
                const double r = size * uni(kind == 1 ? 0.1 : 0.7, 1.0);
                px = cx + r * cos(a);
                py = cy + r * sin(a);
            }
            t.x[v] = (int32_t)lround(std::min(std::max(px, 0.0), (double)W) * 16.0);
            t.y[v] = (int32_t)lround(std::min(std::max(py, 0.0), (double)H) * 16.0);
        }
        const double area = (double)(t.x[1] - t.x[0]) * (t.y[2] - t.y[0]) - (double)(t.x[2] - t.x[0]) * (t.y[1] - t.y[0]);
        if (area > 0) {
            std::swap(t.x[1], t.x[2]);
            std::swap(t.y[1], t.y[2]);
        }
        const double near = uni(1.0, 20.0);
        const double far = near * exp(uni(0.0, log(ratio)));
        const bool along = kind == 0 && k % 2 == 0;
        for (int v = 0; v < 3; v++) {
            const float w = (float)(along ? (v == 0 ? far : near) : near * exp(uni(0.0, log(ratio))));
            const float z = (w - 0.1f) * (150.0f / 149.9f);
            t.oow[v] = 1.0f / w;
            t.zow[v] = z * t.oow[v];
        }
        if (area != 0) walk(t, W, H, *out);
    }
}
