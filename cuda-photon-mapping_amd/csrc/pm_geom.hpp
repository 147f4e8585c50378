// Device geometry shared by photon tracing and the eye-ray renderer: FP32
// vector helpers in the reference's host evaluation order (the library is
// built with -ffp-contract=off, and division / sqrtf are IEEE correctly
// rounded), ray-triangle and ray-box tests, the scene hit, and the per-path
// Philox4x32-10 stream.
#pragma once
#include <cfloat>
#include <cstring>
#include <vector>

#include "pm_internal.hpp"

namespace pmg {

struct V3 {
    float x, y, z;
};
__device__ __forceinline__ V3 v3(float x, float y, float z) { return V3{x, y, z}; }
__device__ __forceinline__ V3 add(V3 a, V3 b) { return V3{a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ V3 sub(V3 a, V3 b) { return V3{a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ V3 mul(V3 a, float f) { return V3{a.x * f, a.y * f, a.z * f}; }
__device__ __forceinline__ V3 mulv(V3 a, V3 b) { return V3{a.x * b.x, a.y * b.y, a.z * b.z}; }
__device__ __forceinline__ V3 neg(V3 a) { return V3{-a.x, -a.y, -a.z}; }
// vec3::dot host branch (vec3.cuh:258-274)
__device__ __forceinline__ float dot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
// vec3::cross host branch (vec3.cuh:276-300)
__device__ __forceinline__ V3 cross(V3 a, V3 b) {
    return V3{a.y * b.z - a.z * b.y, -(a.x * b.z - a.z * b.x), a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ float length(V3 a) { return sqrtf(a.x * a.x + a.y * a.y + a.z * a.z); }
__device__ __forceinline__ bool is_null(V3 a) { return a.x == 0.f && a.y == 0.f && a.z == 0.f; }
// static vec3::normalize: division by the length (vec3.cuh:226-240)
__device__ __forceinline__ V3 normalize_div(V3 a) {
    if (is_null(a)) return a;
    float l = length(a);
    return V3{a.x / l, a.y / l, a.z / l};
}
// member vec3::normalize: multiply by 1/length (vec3.cuh:211-224, :156-169)
__device__ __forceinline__ V3 normalize_rcp(V3 a) {
    if (is_null(a)) return a;
    float u = 1.0f / length(a);
    return V3{a.x * u, a.y * u, a.z * u};
}
__device__ __forceinline__ float maxc(V3 a) { return fmaxf(fmaxf(a.x, a.y), a.z); }

struct Ray {
    V3 o, d;
};

// Per-model record on the device (material of Material.cuh:4-31, the
// triangle range of the model, its AABB and id). bvh is the model's root
// node in the scene's BVH node array, or -1 to test every triangle; rec is its
// first slot in the scene's triangle records (where there are any).
struct DevModel {
    uint32_t t0, t1, rec;
    float kd[3], ks[3], ke[3];
    float ior, opaque, shininess;
    int32_t id, bvh;
    float box[6];
};

}  // namespace pmg

// The most models of a scene whose rays take the records (a bit each in a mask).
constexpr int kRecModels = 32;

// Scene acceleration structure: per-model AABBs and triangle BVHs, built once
// per geometry and shared by photon tracing and eye-ray rendering.
struct pm_accel {
    uint32_t n_tris = 0;
    int32_t n_models = 0;
    std::vector<uint32_t> ranges;  // [n_models][2] triangle range the BVH was built for
    std::vector<float> boxes;      // [n_models][6] exact model AABB
    std::vector<int32_t> roots;    // [n_models] root node, -1 = no BVH (every triangle tested)
    uint32_t n_nodes = 0;
    float4* nodes = nullptr;  // [n_nodes][4]
    // Triangle records (pmg::TriRec, 5 float4 each), for scenes of at most
    // kRecModels models: every model's own, from slot slots[model] on (ranges may
    // overlap, and a BVH's are in its leaf order), else in index order.
    float4* recs = nullptr;
    std::vector<uint32_t> slots;  // [n_models]
    float4* wide = nullptr;   // [n_nodes][8]: the four-wide trees, by binary node (with recs)
};

namespace pmg {

__device__ __forceinline__ V3 load_v(const float* __restrict__ t9, uint32_t t, int k) {
    const float* p = t9 + 9 * (size_t)t + 3 * k;
    return v3(p[0], p[1], p[2]);
}

// AABB::intersects_with_ray (AABB.cuh:103-111, update_tmin_tmax :115-127)
__device__ __forceinline__ bool box_hit(const float* c, const Ray& r) {
    float tmin = 0.0f, tmax = __builtin_inff();
    const float o[3] = {r.o.x, r.o.y, r.o.z}, d[3] = {r.d.x, r.d.y, r.d.z};
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        bool sign = __builtin_signbit(d[i]);
        float bmin = sign ? c[3 + i] : c[i];
        float bmax = sign ? c[i] : c[3 + i];
        float dmin = (bmin - o[i]) / d[i];
        float dmax = (bmax - o[i]) / d[i];
        tmin = fmaxf(dmin, tmin);
        tmax = fminf(dmax, tmax);
    }
    return tmin <= tmax;
}

// traingle_intersection (Model.cuh:69-120)
__device__ __forceinline__ bool tri_hit(const Ray& r, V3 v0, V3 v1, V3 v2, float& t, V3& uvw) {
    V3 N = cross(sub(v1, v0), sub(v2, v0));
    float denom = 1.0f / dot(N, N);
    float nd = dot(N, r.d);
    if (fabsf(nd) < 1e-6f) return false;
    t = (dot(N, v0) - dot(N, r.o)) / nd;
    if (t < 0) return false;
    V3 P = add(r.o, mul(r.d, t));
    float w = dot(N, cross(sub(v1, v0), sub(P, v0)));
    if (w < 0) return false;
    float v = dot(N, cross(sub(v0, v2), sub(P, v2)));
    if (v < 0) return false;
    w *= denom;
    v *= denom;
    float u = 1.f - v - w;
    if (u < 0) return false;
    uvw = v3(u, v, w);
    return true;
}

// A triangle with the ray-independent parts of tri_hit worked out once, by
// tri_hit's own expressions (so its values are the same to the bit): the
// unnormalised normal N, 1 / N.N, N.v0, and the edges v1 - v0 and v0 - v2.
// Five float4 a triangle, one cache line and a quarter.
struct TriRec {
    V3 N, v0, e10, e02, v2;
    float denom, nv0;
};
__device__ __forceinline__ TriRec make_rec(V3 v0, V3 v1, V3 v2) {
    TriRec T;
    T.N = cross(sub(v1, v0), sub(v2, v0));
    T.denom = 1.0f / dot(T.N, T.N);
    T.nv0 = dot(T.N, v0);
    T.v0 = v0;
    T.e10 = sub(v1, v0);
    T.e02 = sub(v0, v2);
    T.v2 = v2;
    return T;
}
__device__ __forceinline__ void store_rec(float4* __restrict__ recs, uint32_t slot, uint32_t t, const TriRec& T) {
    float4* r = recs + 5 * (size_t)slot;
    r[0] = make_float4(T.N.x, T.N.y, T.N.z, T.denom);
    r[1] = make_float4(T.v0.x, T.v0.y, T.v0.z, T.nv0);
    r[2] = make_float4(T.e10.x, T.e10.y, T.e10.z, T.v2.x);
    r[3] = make_float4(T.e02.x, T.e02.y, T.e02.z, T.v2.y);
    r[4] = make_float4(T.v2.z, __uint_as_float(t), 0.f, 0.f);
}
// tri_hit on the record in a slot; tri = its triangle.
__device__ __forceinline__ bool rec_hit(const float4* __restrict__ recs, uint32_t slot, const Ray& r, float& t,
                                        V3& uvw, uint32_t& tri) {
    const float4* q = recs + 5 * (size_t)slot;
    const float4 a = q[0], b = q[1], c = q[2], e = q[3];
    const float2 f = *reinterpret_cast<const float2*>(q + 4);
    const float v2z = f.x;
    tri = __float_as_uint(f.y);
    const V3 N = v3(a.x, a.y, a.z), v0 = v3(b.x, b.y, b.z);
    const float nd = dot(N, r.d);
    if (fabsf(nd) < 1e-6f) return false;
    t = (b.w - dot(N, r.o)) / nd;
    if (t < 0) return false;
    const V3 P = add(r.o, mul(r.d, t));
    float w = dot(N, cross(v3(c.x, c.y, c.z), sub(P, v0)));
    if (w < 0) return false;
    float v = dot(N, cross(v3(e.x, e.y, e.z), sub(P, v3(c.w, e.w, v2z))));
    if (v < 0) return false;
    w *= a.w;
    v *= a.w;
    const float u = 1.f - v - w;
    if (u < 0) return false;
    uvw = v3(u, v, w);
    return true;
}

// box_hit decided from hardware reciprocals of the direction, where that is
// certain: each slab distance (b - o) * inv is within 2^-22 of the divided
// one, relative, and box_hit is "no entry distance above another axis's exit
// distance, and none above an exit below 0" (an axis's own entry never
// exceeds its own exit). hit: every such exit clearly exceeds the largest
// entry; miss: one clearly lies below. Neither is left to box_hit (rays
// through an edge, or with a component below 1e-30: `safe` is false).
struct RayInv {
    V3 inv;
    bool safe;
};
__device__ __forceinline__ RayInv ray_inv(const Ray& r) {
    RayInv R;
    // a zero component becomes a tiny one of the same sign: its slab is then
    // all of t when the origin lies inside it and empty otherwise
    auto one = [](float d) {
        return __builtin_amdgcn_rcpf(fabsf(d) >= 1e-30f ? d : copysignf(1e-30f, d));
    };
    R.inv = v3(one(r.d.x), one(r.d.y), one(r.d.z));
    R.safe = fabsf(r.d.x) >= 1e-30f && fabsf(r.d.y) >= 1e-30f && fabsf(r.d.z) >= 1e-30f &&
             fabsf(r.o.x) + fabsf(r.o.y) + fabsf(r.o.z) < 1e30f;
    return R;
}
__device__ __forceinline__ void box_quick(const float* __restrict__ c, const Ray& r, V3 inv, bool& hit, bool& miss) {
    const float ax = (c[0] - r.o.x) * inv.x, bx = (c[3] - r.o.x) * inv.x;
    const float ay = (c[1] - r.o.y) * inv.y, by = (c[4] - r.o.y) * inv.y;
    const float az = (c[2] - r.o.z) * inv.z, bz = (c[5] - r.o.z) * inv.z;
    const float lx = fminf(ax, bx), ux = fmaxf(ax, bx);
    const float ly = fminf(ay, by), uy = fmaxf(ay, by);
    const float lz = fminf(az, bz), uz = fmaxf(az, bz);
    const float mx = fmaxf(fmaxf(ly, lz), 0.f), my = fmaxf(fmaxf(lx, lz), 0.f), mz = fmaxf(fmaxf(lx, ly), 0.f);
    const float dx = ux - mx, dy = uy - my, dz = uz - mz;
    const float tx = (fabsf(ux) + mx) * 0x1p-20f, ty = (fabsf(uy) + my) * 0x1p-20f, tz = (fabsf(uz) + mz) * 0x1p-20f;
    // (the constant stands above what underflow can hide)
    hit = dx > tx + 1e-35f && dy > ty + 1e-35f && dz > tz + 1e-35f;
    miss = dx < -tx - 1e-35f || dy < -ty - 1e-35f || dz < -tz - 1e-35f;
}

// ---- per-model triangle BVH ------------------------------------------------
// A node is 4 float4: child 0 box (lo.xyz, hi.xyz), child 1 box, then the two
// child codes as int bits (>= 0: node index; < 0: ~triangle index). Boxes
// are inflated by a margin far above the rounding error of tri_hit, so a
// triangle that tri_hit accepts always lies inside every box on its path.
constexpr int kBvhStack = 64;  // a node's key prefix grows down the tree: depth <= 64
// The top kLdsStack entries of each lane's traversal stack live in LDS
// (lane-interleaved, one 8-byte entry per lane per level, so a wave's
// accesses are conflict-free whatever its lanes' depths); deeper entries,
// rare in practice, fall back to a per-lane array.
constexpr int kLdsStack = 12;
constexpr int kRayWaves = 4;  // waves of a block of every kernel that traces rays
// One wave's LDS: the traversal stacks (a column of [kLdsStack][64] per lane,
// or of [kWideStack][16] per group of four lanes), and with records what the
// groups of tree_nearest pass to and from the rays' own lanes.
constexpr int kWideStack = kLdsStack * 4;
template <bool kRecs>
struct RayLds {
    uint2 stack[kLdsStack * 64];
};
template <>
struct RayLds<true> : RayLds<false> {
    float4 hit[64];    // t, u, v, w
    uint2 who[64];     // model, triangle
    uint32_t list[64];
};
struct BvhStack {
    uint2* lds;  // this lane's column
};

// The four-wide trees (made from the binary ones): a node is four children of
// two float4, one 128-byte line: lo.xyz, hi.x | hi.yz, code, unused. Codes:
// >= 0 the node index, < 0 a leaf of 1..4 consecutive record slots,
// kWideNone an unused child.
constexpr int kWideNone = 0x7FFFFFFF;
__host__ __device__ __forceinline__ int wide_leaf(int slot, int count) { return ~((slot << 2) | (count - 1)); }

__device__ __forceinline__ bool slab(float lx, float ly, float lz, float hx, float hy, float hz, V3 o, V3 inv,
                                     float tb, float& tn) {
    const float ax = (lx - o.x) * inv.x, bx = (hx - o.x) * inv.x;
    const float ay = (ly - o.y) * inv.y, by = (hy - o.y) * inv.y;
    const float az = (lz - o.z) * inv.z, bz = (hz - o.z) * inv.z;
    const float tmin = fmaxf(fmaxf(fminf(ax, bx), fminf(ay, by)), fmaxf(fminf(az, bz), 0.f));
    const float tmax = fminf(fminf(fmaxf(ax, bx), fmaxf(ay, by)), fminf(fmaxf(az, bz), tb));
    tn = tmin;
    return tmin <= tmax;
}

__device__ __forceinline__ V3 inv_dir(V3 d) {
    // a zero component becomes a tiny one of the same sign: its slab is then
    // all of t when the origin lies inside it and empty otherwise
    return v3(1.0f / (d.x != 0.f ? d.x : copysignf(1e-30f, d.x)), 1.0f / (d.y != 0.f ? d.y : copysignf(1e-30f, d.y)),
              1.0f / (d.z != 0.f ? d.z : copysignf(1e-30f, d.z)));
}

// Nearest triangle of one model through its BVH: the smallest t among the
// triangles tri_hit accepts, the lowest index on ties -- exactly what testing
// every triangle in index order returns. Triangles with t >= limit may be
// skipped (the caller discards them). A box is pruned only when its entry t
// exceeds the bound by a relative 2^-16, far above the slab test's rounding.
__device__ __forceinline__ bool bvh_hit(const float4* __restrict__ nodes, int root, const float* __restrict__ t9,
                                        const Ray& r, V3 inv, float limit, float& mt, uint32_t& ti, V3& uvw,
                                        BvhStack S) {
    int stack[kBvhStack - kLdsStack];
    float stn[kBvhStack - kLdsStack];
    int sp = 0;
    int node = root;
    bool found = false;
    mt = FLT_MAX;
    for (;;) {
        const float bound = fminf(limit, mt);
        const float tb = bound + bound * 0x1p-16f;
        if (node >= 0) {
            const float4* nd = nodes + 4 * (size_t)node;
            const float4 a = nd[0], b = nd[1], c = nd[2], e = nd[3];
            float t0, t1;
            const bool h0 = slab(a.x, a.y, a.z, a.w, b.x, b.y, r.o, inv, tb, t0);
            const bool h1 = slab(b.z, b.w, c.x, c.y, c.z, c.w, r.o, inv, tb, t1);
            const int c0 = __float_as_int(e.x), c1 = __float_as_int(e.y);
            if (h0 && h1) {
                const bool first0 = t0 <= t1;
                const int cn = first0 ? c1 : c0;
                const float ct = first0 ? t1 : t0;
                if (sp < kLdsStack)
                    S.lds[sp * 64] = make_uint2((uint32_t)cn, __float_as_uint(ct));
                else
                    stack[sp - kLdsStack] = cn, stn[sp - kLdsStack] = ct;
                ++sp;
                node = first0 ? c0 : c1;
                continue;
            }
            if (h0 || h1) {
                node = h0 ? c0 : c1;
                continue;
            }
        } else {
            const uint32_t t = ~(uint32_t)node;
            float pt;
            V3 pu;
            if (tri_hit(r, load_v(t9, t, 0), load_v(t9, t, 1), load_v(t9, t, 2), pt, pu) &&
                (pt < mt || (found && pt == mt && t < ti))) {
                mt = pt;
                ti = t;
                uvw = pu;
                found = true;
            }
        }
        // next deferred subtree that can still hold a closer hit
        const float bnd = fminf(limit, mt);
        const float tcut = bnd + bnd * 0x1p-16f;
        node = 0x7FFFFFFF;
        while (sp > 0) {
            --sp;
            int cn;
            float ct;
            if (sp < kLdsStack) {
                const uint2 e = S.lds[sp * 64];
                cn = (int)e.x;
                ct = __uint_as_float(e.y);
            } else {
                cn = stack[sp - kLdsStack];
                ct = stn[sp - kLdsStack];
            }
            if (ct <= tcut) {
                node = cn;
                break;
            }
        }
        if (node == 0x7FFFFFFF) break;
    }
    return found;
}

// Nearest hit over all models (find_intersection, PhotonTracing.cu:178-213 /
// Raytracer.cuh:66-93) with Model::intersection (Model.cuh:366-446): per
// model an AABB test, then the model's nearest triangle (the first of equal
// t in index order), normal = normalised barycentric blend of the vertex
// normals; a model's hit replaces the current one if the current t is 0 or
// the new t is smaller. A model with a BVH finds its nearest triangle by
// traversal (same result); the others test every triangle, with triangle
// data read at wave-uniform indices (scalar loads). A lane that is not alive joins the
// (wave-uniform) triangle loops and hits nothing: it opens no model's box (a
// null ray in its place opened all boxes behind or above it, and walked their
// trees: traces of 1000 photons in 45 models took 1958 us instead of 762).
__device__ __forceinline__ bool scene_hit(const DevModel* __restrict__ M, int n_models,
                                          const float* __restrict__ t9, const float* __restrict__ n9,
                                          const float4* __restrict__ bvh, bool alive, const Ray& r, float& t_out,
                                          V3& n_out, int& m_out, BvhStack S) {
    float best = 0.f;
    int bm = -1;
    V3 bn = v3(0, 0, 0);
    V3 inv = v3(0, 0, 0);
    bool have_inv = false;
    for (int m = 0; m < n_models; ++m) {
        const bool in_box = alive && box_hit(M[m].box, r);
        if (!__builtin_amdgcn_ballot_w64(in_box)) continue;
        float mt = FLT_MAX;
        bool found = false;
        V3 uvw = v3(0, 0, 0);
        uint32_t ti = 0;
        const int root = M[m].bvh;
        if (root >= 0) {
            if (!have_inv) {
                inv = inv_dir(r.d);
                have_inv = true;
            }
            // a later model matters only below the current best (unless best is 0)
            const float limit = (bm >= 0 && best != 0.f) ? best : FLT_MAX;
            if (in_box) found = bvh_hit(bvh, root, t9, r, inv, limit, mt, ti, uvw, S);
        } else {
            const uint32_t t0 = M[m].t0, t1 = M[m].t1;
            for (uint32_t t = t0; t < t1; ++t) {
                float pt;
                V3 pu;
                if (in_box && tri_hit(r, load_v(t9, t, 0), load_v(t9, t, 1), load_v(t9, t, 2), pt, pu) && pt < mt) {
                    mt = pt;
                    uvw = pu;
                    ti = t;
                    found = true;
                }
            }
        }
        if (!found) continue;
        V3 n = add(add(mul(load_v(n9, ti, 0), uvw.x), mul(load_v(n9, ti, 1), uvw.y)), mul(load_v(n9, ti, 2), uvw.z));
        n = normalize_rcp(n);
        if (bm < 0 || best == 0.f || mt < best) {
            best = mt;
            bm = m;
            bn = n;
        }
    }
    if (bm < 0) return false;
    t_out = best;
    n_out = bn;
    m_out = bm;
    return true;
}

// The scene as the ray kernels see it. recs (with an acceleration structure,
// at most kRecModels models): scene_nearest; brute / tree are the model masks without
// and with a BVH (models of no triangles in neither).
struct SceneGeo {
    const DevModel* models;
    int n_models;
    const float* tris;
    const float* nrms;
    const float4* bvh;
    const float4* wide;
    const float4* recs;
    uint32_t brute, tree;
};

template <int kCtrl>
__device__ __forceinline__ uint32_t quad(uint32_t v) {  // quad_perm: a lane of the same four
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, kCtrl, 0xf, 0xf, true);
}
constexpr int kQuadX1 = 0xB1, kQuadX2 = 0x4E, kQuadX3 = 0x1B;  // lane ^ 1, ^ 2, ^ 3
template <int kCtrl>
__device__ __forceinline__ float quadf(float v) {
    return __uint_as_float(quad<kCtrl>(__float_as_uint(v)));
}

// The nearest hit of every ray with `pend` models (their BVHs) left, four
// lanes to a ray: the lanes of a group test a node's four children, or a
// leaf's up to four triangles, side by side. Of a wave's rays only some reach
// a BVH's box (10 of 64 on a Cornell box's diffuse bounces), and they need
// very different numbers of nodes (16 on average, 47 the most of a wave's):
// one ray a lane ran the walk at 5% of the lanes. Groups take the next
// waiting ray when theirs is done. On entry best / bm / bt hold the ray's
// nearest hit so far; on return the overall one (smallest t, lowest model,
// lowest triangle). lost: the ray's stack was too small; its result is not to
// be used. All 64 lanes take part.
__device__ __forceinline__ void tree_nearest(const SceneGeo& G, uint32_t pend, const Ray& r, float& best, int& bm,
                                             uint32_t& bt, V3& uvw, bool& lost, RayLds<true>& L) {
    const uint32_t lane = __lane_id(), j = lane & 3u, g = lane >> 2;
    const uint64_t wait = __builtin_amdgcn_ballot_w64(pend != 0);
    const uint32_t n_wait = (uint32_t)__builtin_popcountll(wait);
    if (pend) L.list[__builtin_amdgcn_mbcnt_hi((uint32_t)(wait >> 32),
                                               __builtin_amdgcn_mbcnt_lo((uint32_t)wait, 0u))] = lane;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    uint32_t next = 0;        // (wave-uniform) first waiting ray not taken
    int own = -1;             // the lane whose ray the group works on
    uint32_t models = 0, gt = 0;
    int node = kWideNone, sp = 0, cm = 0, gm = -1;
    Ray q{v3(0, 0, 0), v3(0, 0, 0)};
    V3 inv = v3(0, 0, 0), gu = v3(0, 0, 0);
    float gb = FLT_MAX, T = FLT_MAX;  // this lane's nearest hit, the group's bound
    bool over = false;
    for (;;) {
        const uint64_t idle = __builtin_amdgcn_ballot_w64(own < 0 && j == 0);
        if (idle && next < n_wait) {
            const uint32_t rank = (uint32_t)__builtin_popcountll(idle & ((1ull << (lane & ~3u)) - 1ull));
            bool take = false;
            if (own < 0 && next + rank < n_wait) {
                own = (int)L.list[next + rank];
                take = true;
            }
            next += (uint32_t)__builtin_popcountll(idle);
            const int src = own < 0 ? 0 : own;
            const float ox = __shfl(r.o.x, src, 64), oy = __shfl(r.o.y, src, 64), oz = __shfl(r.o.z, src, 64);
            const float dx = __shfl(r.d.x, src, 64), dy = __shfl(r.d.y, src, 64), dz = __shfl(r.d.z, src, 64);
            const float b0 = __shfl(best, src, 64);
            const int m0 = __shfl(bm, src, 64);
            const uint32_t t0 = (uint32_t)__shfl((int)bt, src, 64), p0 = (uint32_t)__shfl((int)pend, src, 64);
            if (take) {
                q.o = v3(ox, oy, oz);
                q.d = v3(dx, dy, dz);
                inv = ray_inv(q).inv;
                gb = T = b0;
                gm = m0;
                gt = t0;
                models = p0;
                node = kWideNone;
                sp = 0;
                over = false;
            }
        }
        if (!__builtin_amdgcn_ballot_w64(own >= 0)) break;
        // internal nodes, until no group holds one
        for (;;) {
            const float tb = T + T * 0x1p-16f;
            if (own >= 0 && node == kWideNone) {
                while (sp > 0) {
                    --sp;
                    const uint2 e = L.stack[sp * 16 + (int)g];
                    if (__uint_as_float(e.y) <= tb) {
                        node = (int)e.x;
                        break;
                    }
                }
                if (node == kWideNone && models) {
                    cm = __builtin_ctz(models);
                    models &= models - 1;
                    node = G.models[cm].bvh;
                }
            }
            const bool in = node >= 0 && node != kWideNone;
            if (!__builtin_amdgcn_ballot_w64(in)) break;
            if (in) {
                const float4* nd = G.wide + 8 * (size_t)node + 2 * j;
                const float4 a = nd[0], b = nd[1];
                float tn;
                const int code = __float_as_int(b.z);
                const bool h = slab(a.x, a.y, a.z, a.w, b.x, b.y, q.o, inv, tb, tn) && code != kWideNone;
                // keys in entry order, distinct (the entry's low bits give
                // way to the lane: a lower bound still)
                const uint32_t key = h ? ((__float_as_uint(tn) & ~3u) | j) : 0xFFFFFFFFu;
                const uint32_t k1 = quad<kQuadX1>(key), k2 = quad<kQuadX2>(key), k3 = quad<kQuadX3>(key);
                const uint32_t rank = (k1 < key) + (k2 < key) + (k3 < key);
                const int nh = (int)h + (k1 != 0xFFFFFFFFu) + (k2 != 0xFFFFFFFFu) + (k3 != 0xFFFFFFFFu);
                // the nearest child next, the others onto the stack, the
                // farthest first
                uint32_t first = h && rank == 0 ? (uint32_t)code : 0u;
                first |= quad<kQuadX1>(first);
                first |= quad<kQuadX2>(first);
                node = nh > 0 ? (int)first : kWideNone;
                if (nh > 1) {
                    if (sp + nh - 1 > kWideStack) {
                        over = true;
                        node = kWideNone;
                        sp = 0;
                        models = 0;
                    } else {
                        if (h && rank > 0) L.stack[(sp + nh - 1 - (int)rank) * 16 + (int)g] = make_uint2((uint32_t)code, key);
                        sp += nh - 1;
                    }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        // rays with nothing left: the lanes' nearest, to the ray's own lane
        const bool done = own >= 0 && node == kWideNone;
        if (__builtin_amdgcn_ballot_w64(done)) {
            if (done) {
                auto merge = [&](float ob, uint32_t om, uint32_t ot, V3 ou) {
                    const bool less = ob < gb || (ob == gb && (om < (uint32_t)gm || (om == (uint32_t)gm && ot < gt)));
                    gb = less ? ob : gb;
                    gm = less ? (int)om : gm;
                    gt = less ? ot : gt;
                    gu.x = less ? ou.x : gu.x;
                    gu.y = less ? ou.y : gu.y;
                    gu.z = less ? ou.z : gu.z;
                };
                merge(quadf<kQuadX1>(gb), quad<kQuadX1>((uint32_t)gm), quad<kQuadX1>(gt),
                      v3(quadf<kQuadX1>(gu.x), quadf<kQuadX1>(gu.y), quadf<kQuadX1>(gu.z)));
                merge(quadf<kQuadX2>(gb), quad<kQuadX2>((uint32_t)gm), quad<kQuadX2>(gt),
                      v3(quadf<kQuadX2>(gu.x), quadf<kQuadX2>(gu.y), quadf<kQuadX2>(gu.z)));
                if (j == 0) {
                    L.hit[own] = make_float4(gb, gu.x, gu.y, gu.z);
                    L.who[own] = make_uint2(over ? 0xFFFFFFFEu : (uint32_t)gm, gt);
                }
                own = -1;
            }
        }
        // leaves: a triangle a lane
        if (node < 0) {
            const uint32_t leaf = ~(uint32_t)node;
            const uint32_t cnt = (leaf & 3u) + 1u;
            if (j < cnt) {
                float pt;
                V3 pu;
                uint32_t tri;
                if (rec_hit(G.recs, (leaf >> 2) + j, q, pt, pu, tri) &&
                    (pt < gb || (pt == gb && gm >= 0 && (cm < gm || (cm == gm && tri < gt))))) {
                    gb = pt;
                    gm = cm;
                    gt = tri;
                    gu = pu;
                }
            }
            T = fminf(gb, quadf<kQuadX1>(gb));
            T = fminf(T, quadf<kQuadX2>(T));
            node = kWideNone;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    lost = false;
    if (pend) {
        const uint2 w = L.who[lane];
        lost = w.x == 0xFFFFFFFEu;
        if (!lost && (w.x != (uint32_t)bm || w.y != bt)) {
            const float4 h = L.hit[lane];
            best = h.x;
            uvw = v3(h.y, h.z, h.w);
            bm = (int)w.x;
            bt = w.y;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// scene_hit, lane by lane. scene_hit goes through the models with the whole
// wave, so each of its loops costs the wave the most that any lane needs, and
// it works out a normal for every model that any lane hits. Here
//   * the model boxes are tested by reciprocals (box_quick, box_hit where
//     that leaves a doubt);
//   * each lane then goes through the triangles of its own models without a
//     BVH, one a step, so a step holds different models in different lanes;
//     triangles come from records;
//   * the rays that reach a BVH's box are walked four lanes to a ray
//     (tree_nearest);
//   * one nearest hit (smallest t; on ties the lowest model, then the lowest
//     triangle) is kept over all models, and the normal is worked out for it
//     alone.
// That is scene_hit's result unless a hit has t == 0 exactly (its fold lets
// any later model replace such a hit): those rays, and any whose stack was
// too small, take scene_hit itself, by the models' trees (a single ray of
// 65536 paths past every triangle of a scene of 44k cost 3.4 ms). `alive`: lanes without a ray take part in
// nothing; all 64 lanes call.
__device__ __forceinline__ bool scene_nearest(const SceneGeo& G, bool alive, const Ray& r, float& t_out, V3& n_out,
                                              int& m_out, RayLds<true>& L) {
    const RayInv R = ray_inv(r);
    uint32_t mask = 0, doubt = 0;
    for (int m = 0; m < G.n_models; ++m) {
        bool hit, miss;
        box_quick(G.models[m].box, r, R.inv, hit, miss);
        mask |= hit ? 1u << m : 0u;
        doubt |= !hit && !miss ? 1u << m : 0u;
    }
    if (!R.safe) {
        mask = 0;
        doubt = G.brute | G.tree;
    }
    if (!alive) mask = doubt = 0;
    doubt &= G.brute | G.tree;
    if (__builtin_amdgcn_ballot_w64(doubt != 0)) {
        for (int m = 0; m < G.n_models; ++m) {
            if ((doubt >> m & 1u) && box_hit(G.models[m].box, r)) mask |= 1u << m;
        }
    }
    float best = FLT_MAX;
    int bm = -1;
    uint32_t bt = 0;
    V3 uvw = v3(0, 0, 0);
    {
        uint32_t pend = mask & G.brute, t = 0, te = 0;
        int cm = 0;
        for (;;) {
            if (t == te && pend) {
                cm = __builtin_ctz(pend);
                pend &= pend - 1;
                t = G.models[cm].rec;
                te = t + (G.models[cm].t1 - G.models[cm].t0);
            }
            if (!__builtin_amdgcn_ballot_w64(t < te)) break;
            if (t < te) {
                float pt;
                V3 pu;
                uint32_t tri;
                // (models and triangles ascend: a tie keeps the first)
                if (rec_hit(G.recs, t, r, pt, pu, tri) && pt < best) {
                    best = pt;
                    bm = cm;
                    bt = tri;
                    uvw = pu;
                }
                ++t;
            }
        }
    }
    const uint32_t pend = mask & G.tree;
    bool lost = false;
    if (__builtin_amdgcn_ballot_w64(pend != 0)) tree_nearest(G, pend, r, best, bm, bt, uvw, lost, L);
    bool found = bm >= 0;
    if (found) {
        t_out = best;
        m_out = bm;
        const V3 n = add(add(mul(load_v(G.nrms, bt, 0), uvw.x), mul(load_v(G.nrms, bt, 1), uvw.y)),
                         mul(load_v(G.nrms, bt, 2), uvw.z));
        n_out = normalize_rcp(n);
    }
    const bool again = lost || (found && best == 0.f);
    if (__builtin_amdgcn_ballot_w64(again)) {
        if (again)
            found = scene_hit(G.models, G.n_models, G.tris, G.nrms, G.bvh, true, r, t_out, n_out, m_out,
                              BvhStack{L.stack + __lane_id()});
    }
    return found;
}

// The nearest hit of each lane's ray; all 64 lanes call. kRecs: the scene has
// records (G.recs).
template <bool kRecs>
__device__ __forceinline__ bool find_hit(const SceneGeo& G, bool alive, const Ray& r, float& t_out, V3& n_out,
                                         int& m_out, RayLds<kRecs>& L) {
    if constexpr (kRecs)
        return scene_nearest(G, alive, r, t_out, n_out, m_out, L);
    else
        return scene_hit(G.models, G.n_models, G.tris, G.nrms, G.bvh, alive, r, t_out, n_out, m_out,
                         BvhStack{L.stack + __lane_id()});
}

inline SceneGeo scene_geo(const pm_scene* scene, const DevModel* d_models) {
    SceneGeo G{};
    G.models = d_models;
    G.n_models = scene->n_models;
    G.tris = scene->d_tris9;
    G.nrms = scene->d_normals9;
    const pm_accel* acc = scene->accel;
    if (!acc || acc->n_models != scene->n_models) return G;  // (upload_models refuses another scene's)
    G.bvh = acc->nodes;
    if (scene->n_models > kRecModels) return G;
    G.recs = acc->recs;
    G.wide = acc->wide;
    for (int i = 0; i < scene->n_models; ++i) {
        if (acc->ranges[2 * i] == acc->ranges[2 * i + 1]) continue;
        (acc->roots[i] >= 0 ? G.tree : G.brute) |= 1u << i;
    }
    return G;
}

// Host side: copy the scene's model table to the device as DevModel records
// with their AABBs -- from the scene's acceleration structure when it has
// one, else computed on the device over each model's triangles (the live
// effect of create_kd_tree, KdTree.cu:395-464). d_tmp needs 32 * n_models
// bytes. On return host_out holds the same records.
// `tail` (nullable): a further table, at d_tail behind d_models in the same block.
inline pm_status upload_models(pm_ctx* ctx, const pm_scene* scene, DevModel* d_models, void* d_tmp,
                               std::vector<DevModel>& host_out, void* d_tail = nullptr, const void* tail = nullptr,
                               size_t tail_bytes = 0) {
    const int nm = scene->n_models;
    const pm_accel* acc = scene->accel;
    std::vector<DevModel>& hm = host_out;
    hm.assign(nm, DevModel{});
    if (acc && (acc->n_models != nm || acc->n_tris != scene->n_tris))
        return pm::fail(ctx, PM_ERR_INVALID, "scene: acceleration structure built for another scene");
    for (int i = 0; i < nm; ++i) {
        const pm_model& s = scene->h_models[i];
        if (s.tri_end > scene->n_tris || s.tri_begin > s.tri_end)
            return pm::fail(ctx, PM_ERR_INVALID, "scene: model %d triangle range", i);
        if (acc && (acc->ranges[2 * i] != s.tri_begin || acc->ranges[2 * i + 1] != s.tri_end))
            return pm::fail(ctx, PM_ERR_INVALID, "scene: model %d differs from its acceleration structure", i);
        DevModel& d = hm[i];
        d.t0 = s.tri_begin;
        d.t1 = s.tri_end;
        for (int c = 0; c < 3; ++c) {
            d.kd[c] = s.kd[c];
            d.ks[c] = s.ks[c];
            d.ke[c] = s.ke[c];
        }
        d.ior = s.refr_index;
        d.opaque = s.opaque;
        d.shininess = s.shininess;
        d.id = s.id;
        d.bvh = acc ? acc->roots[i] : -1;
        d.rec = acc && acc->recs ? acc->slots[i] : 0u;
        if (acc)
            for (int c = 0; c < 6; ++c) d.box[c] = acc->boxes[6 * (size_t)i + c];
    }
    if (!acc) {
        uint32_t* d_tb = static_cast<uint32_t*>(d_tmp);
        float* d_box = reinterpret_cast<float*>(static_cast<char*>(d_tmp) + 8 * (size_t)nm);
        std::vector<uint32_t> tb(2 * (size_t)nm);
        for (int i = 0; i < nm; ++i) {
            tb[2 * i] = hm[i].t0;
            tb[2 * i + 1] = hm[i].t1;
        }
        PM_HIP(ctx, hipMemcpyAsync(d_tb, tb.data(), tb.size() * 4, hipMemcpyHostToDevice, ctx->stream));
        pm_status st;
        for (int i = 0; i < nm; ++i)
            if ((st = pm::model_aabb_launch(ctx, scene->d_tris9, d_tb + 2 * i, 1, d_box + 6 * i)) != PM_OK) return st;
        std::vector<float> boxes((size_t)nm * 6);
        PM_HIP(ctx, hipMemcpyAsync(boxes.data(), d_box, boxes.size() * 4, hipMemcpyDeviceToHost, ctx->stream));
        PM_HIP(ctx, hipStreamSynchronize(ctx->stream));
        for (int i = 0; i < nm; ++i)
            for (int c = 0; c < 6; ++c) hm[i].box[c] = boxes[(size_t)i * 6 + c];
    }
    if (tail_bytes == 0) return pm::put(ctx, d_models, hm.data(), nm * sizeof(DevModel));
    const size_t at = (size_t)(static_cast<char*>(d_tail) - reinterpret_cast<char*>(d_models));
    std::vector<char> both(at + tail_bytes);
    std::memcpy(both.data(), hm.data(), nm * sizeof(DevModel));
    std::memcpy(both.data() + at, tail, tail_bytes);
    return pm::put(ctx, d_models, both.data(), both.size());
}

// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11); one stream per
// (seed, stream id, path id), four uniforms per block, u in (0, 1].
//
// A block costs twenty 32 x 32 -> 64 products (quarter rate) whatever the
// lanes that need one, and lanes run out of words at different draws; so a
// lane holds a second block ahead, and `ensure` makes one for every lane that
// has none as soon as any lane would run short. In a rejection loop the wave
// then pays one block per two trials instead of one per draw.
__device__ __forceinline__ void philox4x32_10(uint32_t k0, uint32_t k1, uint32_t path, uint32_t blk, uint32_t sid,
                                              uint32_t (&w)[4]) {
    uint32_t c0 = path, c1 = blk, c2 = sid, c3 = 0x7068u;
    uint32_t a = k0, b = k1;
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
        const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ a, n2 = (uint32_t)(p0 >> 32) ^ c3 ^ b;
        c0 = n0;
        c1 = (uint32_t)p1;
        c2 = n2;
        c3 = (uint32_t)p0;
        a += 0x9E3779B9u;
        b += 0xBB67AE85u;
    }
    w[0] = c0;
    w[1] = c1;
    w[2] = c2;
    w[3] = c3;
}
__device__ __forceinline__ float uniform01(uint32_t x) { return (float)((x >> 8) + 1u) * (1.0f / 16777216.0f); }

struct Stream {
    uint32_t k0, k1, path, sid, blk;
    uint32_t left, more;  // words left in buf, 1 when nxt holds block blk - 1
    uint32_t buf[4], nxt[4];
    __device__ __forceinline__ void init(uint64_t seed, uint32_t stream_id, uint32_t path_id) {
        k0 = (uint32_t)seed;
        k1 = (uint32_t)(seed >> 32);
        path = path_id;
        sid = stream_id;
        blk = 0;
        left = 0;
        more = 0;
    }
    // Resume with one word left of the block before `block`.
    __device__ __forceinline__ void resume(uint32_t block, uint32_t word) {
        blk = block;
        left = 1;
        more = 0;
        buf[0] = word;
        for (int c = 1; c < 4; ++c) buf[c] = 0;
        for (int c = 0; c < 4; ++c) nxt[c] = 0;
    }
    // At least n (1..4) words for every calling lane.
    __device__ __forceinline__ void ensure(uint32_t n) {
        if (!__builtin_amdgcn_ballot_w64(left + 4u * more < n)) return;
        if (more) return;
        philox4x32_10(k0, k1, path, blk, sid, nxt);
        ++blk;
        more = 1;
    }
    // The next uniform; an `ensure` before it covers the draw. buf is a shift
    // register: the next word is always buf[0], so no lane state is ever
    // indexed dynamically.
    __device__ __forceinline__ float next() {
        if (left == 0) {
            for (int c = 0; c < 4; ++c) buf[c] = nxt[c];
            left = 4;
            more = 0;
        }
        const uint32_t x = buf[0];
        buf[0] = buf[1];
        buf[1] = buf[2];
        buf[2] = buf[3];
        --left;
        return uniform01(x);
    }
};

}  // namespace pmg
