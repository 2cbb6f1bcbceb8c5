// gi.hip -- the voxel GI bake on the GPU (bake_voxel_gi, src/gi.rs:316-412;
// blur_gi_sh4, src/voxelgrid.rs:422-472).
//
// One wavefront per active voxel, four per workgroup: lane s traces primary
// direction s of the voxel's direction set (GI_SAMPLES == 64 == the wave
// width).  The workgroup's rays that hit a surface are numbered densely, and
// their transmittance rays (one to the sun and four to the sky each) are
// shared out over all its lanes; each hit's lane then finishes its bounce.
// The 64 radiances of a voxel meet in LDS and lane 0 reduces them in sample
// order (gi_finish_voxel).  Arithmetic and visiting order are gi_core.h's, so
// every voxel's coefficients are the host bake's.  A 3x3x3 blur kernel over
// the whole grid follows.
//
// Bound by the latency of the traversals' dependent loads (nodes and
// triangles come from the L2), so what counts is loads per step, steps per
// ray, idle lanes and waves in flight.  A node holds both children's boxes
// (64 B, tested before anything is pushed, so a ray visits a child's node
// only if its box is hit), a leaf's triangles are copied in leaf order with
// their edges (48 B each), and the stacks hold the tree's own depth.  Boxes
// tested after their pop, triangles behind an index, lanes without a hit idle
// during the others' five rays and stacks of 48 entries (three waves per
// SIMD) took 12.7 ms on 16 icospheres (20,480 triangles) at 64^3; this 3.6.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "gi_host.h"
#include "runtime.h"

namespace sr {
namespace {

static_assert(GI_SAMPLES == 64, "one lane per primary direction");

// An inner node: its children's boxes and references.  A reference is the
// index of an inner node, or GI_LEAF | first triangle << 2 | count - 1 (the
// median split leaves one to four triangles in a leaf).
struct alignas(16) GiPair {
    float l_lo[3], l_hi[3], r_lo[3], r_hi[3];
    uint32_t left, right, pad[2];
};
#define GI_LEAF 0x80000000u

// A triangle in leaf order: vertex 0, the edges to vertices 1 and 2, its
// index among the scene's triangles and its (checked) material.
struct alignas(16) GiLeafTri {
    float p0[3];
    int32_t index;
    float e1[3];
    int32_t material;
    float e2[3];
    uint32_t pad;
};

struct GiDev {
    GiScene S;                    // (its nodes and order stay on the host)
    const GiPair *pairs;
    const GiLeafTri *leaf_tris;
    GiNode root_box;
    uint32_t root;                // reference; the scene has triangles
    int depth;                    // most entries a stack holds
    const float *dirs;            // GI_SETS * GI_SAMPLES * 3
    const uint32_t *voxels;       // active voxel indices
    uint32_t nactive;
    int grid;
    float cmin[3], vs[3];
    float primary_bias;
    GiRayParams P;
    const float *light;           // per voxel sun visibility
    float *coeffs;                // per voxel 16 floats
    uint32_t *over;               // set if a transmittance ray met more than GI_HIT_CAP surfaces
};

// initialize_voxel_gi_from_scene with scale 1 (src/gi.rs:123-149).
__global__ void k_gi_init(GiDev G, size_t nvox) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < nvox; i += (size_t)gridDim.x * blockDim.x) {
        float o[16];
        for (int c = 0; c < 4; c++) {
            for (int k = 0; k < 3; k++) o[4 * c + k] = G.S.sh[c][k] * 1.0f;
            o[4 * c + 3] = 0.0f;
        }
        o[3] = G.light[i];
        o[7] = 1.0f;
        float4 *dst = reinterpret_cast<float4 *>(G.coeffs + 16 * i);
        for (int c = 0; c < 4; c++) dst[c] = make_float4(o[4 * c], o[4 * c + 1], o[4 * c + 2], o[4 * c + 3]);
    }
}

// gi_hit_box in two steps: the ray's entry t0 and exit t1 of a box, then the
// test against the exit or a nearer limit (which is the same: the bound grows
// with its argument, so testing the smaller of two limits is testing both).
__device__ __forceinline__ void gi_slab(const float lo[3], const float hi[3], G3 o, G3 inv, float &t0, float &t1) {
    const float op[3] = {o.x, o.y, o.z}, ip[3] = {inv.x, inv.y, inv.z};
    t0 = 0.0f;
    t1 = INFINITY;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        float ta = (lo[a] - op[a]) * ip[a], tb = (hi[a] - op[a]) * ip[a];
        const bool swap = ta > tb;
        const float n = swap ? tb : ta, f = swap ? ta : tb;
        ta = n != n ? -INFINITY : n;   // 0 * inf
        tb = f != f ? INFINITY : f;
        t0 = t0 < ta ? ta : t0;
        t1 = tb < t1 ? tb : t1;
    }
}
__device__ __forceinline__ bool gi_beyond(float t0, float limit) { return t0 > limit * 1.0000001f + 1e-7f; }

// gi_ray_tri on a leaf triangle.
__device__ __forceinline__ bool gi_ray_leaf_tri(G3 o, G3 d, const GiLeafTri &t, float tmin, float tmax, float &tt,
                                                float &u, float &v) {
    G3 p0 = g3(t.p0[0], t.p0[1], t.p0[2]), e1 = g3(t.e1[0], t.e1[1], t.e1[2]), e2 = g3(t.e2[0], t.e2[1], t.e2[2]);
    G3 pv = gcross(d, e2);
    float det = gdot(e1, pv);
    if (fabsf(det) <= 1.0e-8f) return false;
    float inv = 1.0f / det;
    G3 tv = gsub(o, p0);
    u = gdot(tv, pv) * inv;
    if (!(u >= 0.0f && u <= 1.0f)) return false;
    G3 qv = gcross(tv, e1);
    v = gdot(d, qv) * inv;
    if (v < 0.0f || (u + v) > 1.0f) return false;
    tt = gdot(e2, qv) * inv;
    if (tt < tmin || tt > tmax) return false;
    return true;
}

// Depth-first walk of gi_trace_nearest and gi_trace_transmittance: right
// child first; leaf(first, count) returns true to end the walk; limit()
// bounds the boxes' entries, when they are met and, for NEAREST, again when
// they are popped.  The stack is this lane's column in LDS (entries 256 words
// apart; NEAREST keeps each entry's box entry in a second column behind).
template <bool NEAREST, class Limit, class Leaf>
__device__ __forceinline__ void gi_walk(const GiDev &G, G3 o, G3 d, uint32_t *stack, Limit limit, Leaf leaf) {
    const G3 inv = g3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
    float t0, t1;
    gi_slab(G.root_box.lo, G.root_box.hi, o, inv, t0, t1);
    if (gi_beyond(t0, t1) || gi_beyond(t0, limit())) return;
    uint32_t ref = G.root;
    int n = 0;
    float *entry = reinterpret_cast<float *>(stack + 256 * G.depth);
    for (;;) {
        if (!(ref & GI_LEAF)) {
            const GiPair p = G.pairs[ref];
            float l0, l1, r0, r1;
            gi_slab(p.l_lo, p.l_hi, o, inv, l0, l1);
            gi_slab(p.r_lo, p.r_hi, o, inv, r0, r1);
            const float far = limit();
            const bool left = !(gi_beyond(l0, l1) || gi_beyond(l0, far));
            const bool right = !(gi_beyond(r0, r1) || gi_beyond(r0, far));
            if (left && right) {
                stack[256 * n] = p.left;
                if (NEAREST) entry[256 * n] = l0;
                n++;
            }
            if (left || right) {
                ref = right ? p.right : p.left;
                continue;
            }
        } else if (leaf((ref & ~GI_LEAF) >> 2, (ref & 3u) + 1u)) {
            return;
        }
        for (;;) {
            if (n == 0) return;
            n--;
            ref = stack[256 * n];
            if (!NEAREST || !gi_beyond(entry[256 * n], limit())) break;
        }
    }
}

// gi_trace_nearest.
__device__ __forceinline__ bool gi_nearest(const GiDev &G, G3 o, G3 d, GiHit &hit, uint32_t *stack) {
    float best = INFINITY, bu = 0.0f, bv = 0.0f;
    int32_t best_tri = -1;
    gi_walk<true>(
        G, o, d, stack, [&] { return best; },
        [&](uint32_t first, uint32_t count) {
            for (uint32_t k = first; k < first + count; k++) {
                const GiLeafTri tri = G.leaf_tris[k];
                float t, u, v;
                if (!gi_ray_leaf_tri(o, d, tri, G.P.tmin, best, t, u, v)) continue;
                if (t < best || (t == best && tri.index < best_tri)) {
                    best = t;
                    best_tri = tri.index;
                    bu = u;
                    bv = v;
                }
            }
            return false;
        });
    hit.tri = best_tri;
    hit.t = best;
    hit.u = bu;
    hit.v = bv;
    return best_tri >= 0;
}

// gi_trace_transmittance; without TR (no material is translucent) every hit
// is opaque.
template <bool TR>
__device__ __forceinline__ float gi_transmittance(const GiDev &G, G3 o, G3 d, bool &over, uint32_t *stack) {
    if constexpr (!TR) {
        bool clear = true;
        gi_walk<false>(
            G, o, d, stack, [&] { return INFINITY; },
            [&](uint32_t first, uint32_t count) {
                for (uint32_t k = first; k < first + count && clear; k++) {
                    float t, u, v;
                    clear = !gi_ray_leaf_tri(o, d, G.leaf_tris[k], G.P.tmin, INFINITY, t, u, v);
                }
                return !clear;
            });
        return clear ? 1.0f : 0.0f;
    }
    float ht[GI_HIT_CAP];
    int32_t hi[GI_HIT_CAP], hm[GI_HIT_CAP];
    int nh = 0;
    bool opaque = false;
    gi_walk<false>(
        G, o, d, stack, [&] { return INFINITY; },
        [&](uint32_t first, uint32_t count) {
            for (uint32_t k = first; k < first + count; k++) {
                const GiLeafTri tri = G.leaf_tris[k];
                float t, u, v;
                if (!gi_ray_leaf_tri(o, d, tri, G.P.tmin, INFINITY, t, u, v)) continue;
                if (!G.S.mats[tri.material].translucent) {       // any opaque hit
                    opaque = true;
                    return true;
                }
                if (nh == GI_HIT_CAP) {
                    over = true;
                    continue;
                }
                int j = nh++;
                while (j > 0 && (ht[j - 1] > t || (ht[j - 1] == t && hi[j - 1] > tri.index))) {
                    ht[j] = ht[j - 1];
                    hi[j] = hi[j - 1];
                    hm[j] = hm[j - 1];
                    j--;
                }
                ht[j] = t;
                hi[j] = tri.index;
                hm[j] = tri.material;
            }
            return false;
        });
    if (opaque) return 0.0f;
    float tr = 1.0f;
    for (int j = 0; j < nh; j++) {
        tr *= G.S.mats[hm[j]].transmission;
        if (tr <= 0.0001f) return 0.0f;
    }
    return tr;
}

// Words of LDS behind the workgroup's 256 lanes: the stacks (the primary
// rays' with box entries; the transmittance rays' with what they share), and
// the radiances.
#define GI_SHARED_ROWS 11         // shading origin and normal of each hit, five visibilities
__host__ __device__ static inline uint32_t gi_stack_rows(int depth) {
    return (uint32_t)(2 * depth > depth + GI_SHARED_ROWS ? 2 * depth : depth + GI_SHARED_ROWS);
}

// Four waves, one active voxel each.
template <bool TR>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) void k_gi_voxels(GiDev G, uint32_t first) {
    extern __shared__ uint32_t lds[];
    __shared__ float rad[4][GI_SAMPLES * 3];
    __shared__ uint32_t wave_hits[4];
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const uint32_t a = first + blockIdx.x * 4 + w;
    const bool live = a < G.nactive;
    uint32_t *stack = lds + tid;
    float *shared = reinterpret_cast<float *>(lds + 256 * max(G.depth, 0));      // rows of 256 (after the primary rays)
    uint32_t vi = 0;
    int set = 0;
    bool sky = false, over = false, shade = false;
    G3 r = g3(0.0f, 0.0f, 0.0f), albedo = r, emissive = r, normal = r, origin = r;
    float ndl = 0.0f;
    const G3 L = g3(G.S.light_dir[0], G.S.light_dir[1], G.S.light_dir[2]);
    // ---- primary rays (gi_primary_ray, and gi_bounce up to its rays) ----
    if (live) {
        vi = G.voxels[a];
        const int x = (int)(vi % (uint32_t)G.grid), y = (int)((vi / (uint32_t)G.grid) % (uint32_t)G.grid);
        const int z = (int)(vi / ((uint32_t)G.grid * (uint32_t)G.grid));
        set = ((x % 3) + 3 * (y % 3) + (z % 3)) % GI_SETS;
        G3 c = g3(G.cmin[0] + (float)x * G.vs[0], G.cmin[1] + (float)y * G.vs[1], G.cmin[2] + (float)z * G.vs[2]);
        const float *dp = G.dirs + ((size_t)set * GI_SAMPLES + lane) * 3;
        const G3 dir = g3(dp[0], dp[1], dp[2]);
        const G3 o = gadd(c, gscale(dir, G.primary_bias));
        GiHit hit;
        if (G.depth >= 0 && gi_nearest(G, o, dir, hit, stack)) {
            shade = gi_bounce_surface(G.S, hit, o, dir, G.P, normal, albedo, emissive, origin);
        } else {
            sky = true;
            r = gi_sky_radiance(G.S, dir);
        }
        ndl = gmaxf(gdot(normal, L), 0.0f);
    }
    const uint64_t hm = __ballot(shade);
    if (lane == 0) wave_hits[w] = (uint32_t)__popcll(hm);
    __syncthreads();                              // (also: the primary stacks are done with)
    uint32_t h = (uint32_t)__popcll(hm & ((1ull << lane) - 1ull)), hits = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        if (k < w) h += wave_hits[k];
        hits += wave_hits[k];
    }
    if (shade) {
        const float v[6] = {origin.x, origin.y, origin.z, normal.x, normal.y, normal.z};
#pragma unroll
        for (int k = 0; k < 6; k++) shared[256 * k + (int)h] = v[k];
    }
    __syncthreads();
    // ---- transmittance rays: ray k of hit i is job k * hits + i ----
    const float dir_bias = G.P.hit_bias * 0.5f;
    for (uint32_t job = tid; job < 5u * hits; job += 256u) {
        const uint32_t k = job / hits, i = job - k * hits;
        const G3 so = g3(shared[i], shared[256 + i], shared[512 + i]);
        const G3 sn = g3(shared[768 + i], shared[1024 + i], shared[1280 + i]);
        float vis = 0.0f;
        if (k == 0u) {
            if (gmaxf(gdot(sn, L), 0.0f) > 0.0f)
                vis = gi_transmittance<TR>(G, gadd(so, gscale(L, dir_bias)), L, over, stack);
        } else {
            const G3 dir = gi_sky_dir(sn, (int)k - 1);
            vis = gi_transmittance<TR>(G, gadd(so, gscale(dir, dir_bias)), dir, over, stack);
        }
        shared[256 * (6 + (int)k) + (int)i] = vis;
    }
    if (over) *G.over = 1u;
    __syncthreads();
    if (shade) {
        float vis[5];
#pragma unroll
        for (int k = 0; k < 5; k++) vis[k] = shared[256 * (6 + k) + (int)h];
        const float skyv = ((((0.0f + vis[1]) + vis[2]) + vis[3]) + vis[4]) * 0.25f;
        r = gi_bounce_finish(G.S, normal, albedo, emissive, ndl, vis[0], skyv);
    }
    rad[w][3 * lane] = r.x;
    rad[w][3 * lane + 1] = r.y;
    rad[w][3 * lane + 2] = r.z;
    const uint32_t sky_hits = (uint32_t)__popcll(__ballot(sky));
    __syncthreads();
    if (live && lane == 0) {
        float o[16];
        gi_finish_voxel(G.S, G.dirs + (size_t)set * GI_SAMPLES * 3, rad[w], sky_hits, G.light[vi], o);
        float4 *dst = reinterpret_cast<float4 *>(G.coeffs + 16 * (size_t)vi);
        for (int c = 0; c < 4; c++) dst[c] = make_float4(o[4 * c], o[4 * c + 1], o[4 * c + 2], o[4 * c + 3]);
    }
}

// blur_gi_sh4 (src/voxelgrid.rs:422-472)
__global__ void k_gi_blur(const float *src, float *dst, int grid) {
    size_t n = (size_t)grid * grid * grid;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        int x = (int)(i % grid), y = (int)((i / grid) % grid), z = (int)(i / ((size_t)grid * grid));
        float o[16];
        gi_blur_voxel(src, grid, grid, grid, x, y, z, o);
        float4 *d = reinterpret_cast<float4 *>(dst + 16 * i);
        for (int c = 0; c < 4; c++) d[c] = make_float4(o[4 * c], o[4 * c + 1], o[4 * c + 2], o[4 * c + 3]);
    }
}

struct DevMem {
    std::vector<void *> ptrs;
    ~DevMem() {
        for (void *p : ptrs) hipFree(p);
    }
    template <class T> hipError_t get(T *&p, size_t count) {
        void *q = nullptr;
        hipError_t e = hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(T));
        if (e == hipSuccess) ptrs.push_back(q);
        p = (T *)q;
        return e;
    }
    template <class T> hipError_t put(const T *&p, const T *host, size_t count) {
        T *q;
        hipError_t e = get(q, count);
        if (e == hipSuccess && count) e = hipMemcpy(q, host, count * sizeof(T), hipMemcpyHostToDevice);
        p = q;
        return e;
    }
};

inline uint32_t blocks(size_t n) { return (uint32_t)std::min<size_t>(std::max<size_t>((n + 255) / 256, 1), 65536); }

}  // namespace

#define GI_TRY(expr)                                                                           \
    do {                                                                                       \
        hipError_t _e = (expr);                                                                \
        if (_e != hipSuccess) return fail(SR_ERR_HIP, "%s: %s", #expr, hipGetErrorString(_e)); \
    } while (0)

int gi_bake_device(const GiHost &h, const std::vector<uint8_t> &active, const std::vector<float> &light, int device,
                   float *out) {
    const int grid = h.frame.grid;
    const size_t nvox = (size_t)grid * grid * grid;
    if (active.size() != nvox || light.size() != nvox) return fail(SR_ERR_INVALID_ARGUMENT, "GI grid size mismatch");
    std::vector<uint32_t> list;
    for (size_t i = 0; i < nvox; i++)
        if (active[i]) list.push_back((uint32_t)i);
    GI_TRY(hipSetDevice(device));
    DevMem mem;
    GiDev G;
    memset(&G, 0, sizeof(G));
    G.S = gi_scene_view(h);
    GI_TRY(mem.put(G.S.tris, h.tris.data(), h.tris.size()));
    // the tree as the device walks it: inner nodes with both children's boxes,
    // triangles in leaf order; the deepest inner node bounds the stacks
    std::vector<GiPair> pairs;
    std::vector<GiLeafTri> leaf_tris(h.order.size());
    G.depth = -1;
    if (!h.nodes.empty()) {
        std::vector<int32_t> pair_of(h.nodes.size(), -1), level(h.nodes.size(), 0);
        for (size_t i = 0; i < h.nodes.size(); i++)
            if (h.nodes[i].left >= 0) {
                pair_of[i] = (int32_t)pairs.size();
                pairs.push_back(GiPair());
            }
        auto ref = [&](int32_t i) {
            const GiNode &n = h.nodes[i];
            return n.left >= 0 ? (uint32_t)pair_of[i] : GI_LEAF | (uint32_t)n.first << 2 | (uint32_t)(n.count - 1);
        };
        G.depth = 0;
        for (size_t i = 0; i < h.nodes.size(); i++) {       // (parents come before their children)
            const GiNode &n = h.nodes[i];
            if (n.left < 0) {
                if (n.count < 1 || n.count > 4 || n.first >= (1 << 29))
                    return fail(SR_ERR_UNSUPPORTED, "a GI tree leaf of %d triangles", n.count);
                continue;
            }
            level[n.left] = level[n.right] = level[i] + 1;
            G.depth = std::max(G.depth, level[i] + 1);
            GiPair &p = pairs[pair_of[i]];
            memset(&p, 0, sizeof(p));
            memcpy(p.l_lo, h.nodes[n.left].lo, 12);
            memcpy(p.l_hi, h.nodes[n.left].hi, 12);
            memcpy(p.r_lo, h.nodes[n.right].lo, 12);
            memcpy(p.r_hi, h.nodes[n.right].hi, 12);
            p.left = ref(n.left);
            p.right = ref(n.right);
        }
        G.root = ref(0);
        G.root_box = h.nodes[0];
        for (size_t k = 0; k < h.order.size(); k++) {
            const GiTri &t = h.tris[h.order[k]];
            GiLeafTri &q = leaf_tris[k];
            memset(&q, 0, sizeof(q));
            for (int c = 0; c < 3; c++) {
                q.p0[c] = t.p[c];
                q.e1[c] = t.p[3 + c] - t.p[c];
                q.e2[c] = t.p[6 + c] - t.p[c];
            }
            q.index = h.order[k];
            q.material = t.material >= 0 && t.material < G.S.nmat ? t.material : 0;
        }
    }
    G.S.nodes = nullptr;
    G.S.order = nullptr;
    GI_TRY(mem.put(G.pairs, pairs.data(), pairs.size()));
    GI_TRY(mem.put(G.leaf_tris, leaf_tris.data(), leaf_tris.size()));
    GI_TRY(mem.put(G.S.mats, h.mats.data(), h.mats.size()));
    GI_TRY(mem.put(G.S.texs, h.texs.data(), h.texs.size()));
    GI_TRY(mem.put(G.S.texels, h.texels.data(), h.texels.size()));
    GI_TRY(mem.put(G.S.cubemap, h.cubemap, (size_t)6 * h.cube_size * h.cube_size));
    GI_TRY(mem.put(G.dirs, h.dirs.data(), h.dirs.size()));
    GI_TRY(mem.put(G.voxels, list.data(), list.size()));
    GI_TRY(mem.put(G.light, light.data(), nvox));
    float *blurred;
    GI_TRY(mem.get(G.coeffs, nvox * 16));
    GI_TRY(mem.get(blurred, nvox * 16));
    GI_TRY(mem.get(G.over, 1));
    GI_TRY(hipMemset(G.over, 0, 4));
    G.nactive = (uint32_t)list.size();
    G.grid = grid;
    memcpy(G.cmin, h.frame.cmin, 12);
    memcpy(G.vs, h.frame.vs, 12);
    G.primary_bias = h.primary_bias;
    G.P = h.params;
    hipLaunchKernelGGL(k_gi_init, dim3(blocks(nvox)), dim3(256), 0, nullptr, G, nvox);
    GI_TRY(hipGetLastError());
    if (list.empty()) {     // nothing active: the scene SH, not blurred (src/gi.rs:338-341)
        GI_TRY(hipMemcpy(out, G.coeffs, nvox * 64, hipMemcpyDeviceToHost));
        return SR_OK;
    }
    bool translucent = false;
    for (const GiMat &m : h.mats) translucent = translucent || m.translucent != 0;
    // launches of at most 65536 voxels each
    for (uint32_t first = 0; first < G.nactive; first += 65536) {
        uint32_t n = std::min<uint32_t>(65536, G.nactive - first);
        const uint32_t lds = gi_stack_rows(std::max(G.depth, 0)) * 1024u;
        if (translucent) hipLaunchKernelGGL(k_gi_voxels<true>, dim3((n + 3) / 4), dim3(256), lds, nullptr, G, first);
        else hipLaunchKernelGGL(k_gi_voxels<false>, dim3((n + 3) / 4), dim3(256), lds, nullptr, G, first);
        GI_TRY(hipGetLastError());
    }
    hipLaunchKernelGGL(k_gi_blur, dim3(blocks(nvox)), dim3(256), 0, nullptr, (const float *)G.coeffs, blurred, grid);
    GI_TRY(hipGetLastError());
    uint32_t over = 0;
    GI_TRY(hipMemcpy(&over, G.over, 4, hipMemcpyDeviceToHost));
    if (over) return fail(SR_ERR_CAPACITY, "a GI ray met more than %d translucent surfaces", GI_HIT_CAP);
    GI_TRY(hipMemcpy(out, blurred, nvox * 64, hipMemcpyDeviceToHost));
    return SR_OK;
}

}  // namespace sr
