// k-nearest-photon gather and radiance estimate on the hash grid.
//
// Replaces PhotonGrid::find_nearests + PhotonMaxHeap (PhotonGrid.cu:222-284,
// PhotonMaxHeap.cuh:90-107) and Raytracer::get_color_from_photon_grid
// (Raytracer.cuh:110-138). A wave64 walks one query at a time, and a small
// number of queries one after the other (stream_wave):
//   1. the candidate box (query cell +- ceil(r/cell), clamped) is split into
//      contiguous photon runs (one per (y,z) row of cells in the linear
//      layout, one per cell in the Morton layout), one run per lane;
//   2. the candidates stream 64 at a time (coalesced SoA loads, next step
//      prefetched); d2 = (dx*dx + dy*dy) + dz*dz exactly as the reference
//      host computes it, radius test d2 <= T with T the largest float whose
//      sqrtf is <= r (identical to the reference's sqrtf(d2) <= r);
//   3. in-radius keys (d2 bits << 32 | grid slot) are appended to an LDS
//      buffer with ballot + mbcnt; when it fills, a histogram over the top
//      float bits of d2 (two bins per octave) finds the smallest bin edge
//      keeping >= k keys, the buffer is compacted to it and the acceptance
//      bound tightens (a refinement splits a crowded bin 64 ways);
//   4. lists: a counting sort over bins linear in d2 orders the survivors (at
//      most 512 keys; k_knn_large's bitonic network sorts longer ones); the
//      first k are the answer, the exact k smallest by (d2, slot);
//   5. estimates: the buffer is narrowed to exactly those k, which the same
//      wave sums unsorted (k_gather_wide, from k = 513 on, keeps no keys).
// A two-pass variant (histogram pass, then collect pass) is kept selectable
// for tuning.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "pm_select.hpp"

namespace {

using pmd::GridGeom;
using namespace pms;

constexpr int kWaves = 4;  // queries per 256-thread workgroup
constexpr int kMaxK = 2048;

struct KnnParams {
    GridGeom G;
    const uint32_t* starts;
    const uint32_t* sizes;
    const float* px;
    const float* py;
    const float* pz;
    const float* power;  // 3 planes of n
    const float* dir;    // 3 planes of n
    uint32_t n;
    const float* qx;
    const float* qy;
    const float* qz;
    const float* nrm;  // 3 planes of nq (radiance only)
    uint32_t nq;
    const uint32_t* order;  // optional processing order
    float r;
    float T;      // largest d2 with sqrtf(d2) <= r
    uint32_t bT;  // bits(T) >> 22
    int rc;
    int k;
    uint32_t* out_idx;
    float* out_dist;
    uint32_t* out_count;
    float* rgb;  // 3 planes of nq (radiance only)
    int remap;
    int h;  // inner box half-width in cells (0: walk the whole box at once)
    // Streaming gathers: wave u of n_waves takes the queries at u,
    // u + n_waves, ... (at most gq) of the processing order. nr > 0: the first walked box (the inner one, or the
    // whole) has at most nr = (2 w + 1)^2 rows, gq nr <= 64, and one lane
    // works out each row of all the wave's queries; nr = 0 (Morton, or more
    // than 64 rows): gq = 1 and the rows are taken 64 at a time.
    int nr, w, gq;
    uint32_t n_waves;
    float guess;         // candidates that the guessed bound aims at (stream_wave)
    float within;        // share of a box's candidates expected within the radius
    uint32_t xcd_shift;  // log2 of the workgroups in an XCD's chunk (remap 2)
    // (nullable) the query count on the device, at most nq: positions past
    // it are skipped; nq stays the planes' stride
    const uint32_t* nq_dev;
};

struct Box {
    int lo[3], hi[3];
};

// One FP32 plane as a raw buffer: loads take a 32-bit byte offset (one VALU
// address for the three position planes) and return 0 past the plane's end.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t plane_rsrc(const float* p, uint32_t n) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), (short)0, (int)(n * 4u), 0x00020000);
}
__device__ __forceinline__ float bload(__amdgpu_buffer_rsrc_t r, uint32_t byte_off) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, (int)byte_off, 0, 0));
}

// Lower bound of |v - p| along one axis over the photons hashed into cell c
// (cells 0 and g-1 also hold every photon clamped into them). The cell's
// bounds are widened by a relative 1e-6, far above the rounding of the hash
// (p - mn) / cell and of the bounds themselves.
__device__ __forceinline__ float axis_gap(float v, int c, int g, float mn, float cell) {
    const float lo = mn + (float)c * cell, hi = mn + (float)(c + 1) * cell;
    const float e = (fabsf(lo) + fabsf(hi) + fabsf(mn)) * 1e-6f;
    if (c > 0 && v < lo - e) return (lo - e) - v;
    if (c < g - 1 && v > hi + e) return v - (hi + e);
    return 0.f;
}

// Lower bound of |v - p| along one axis over the photons hashed outside the
// cells [lo, hi] (cells 0 and g-1 are unbounded outward, so a side at the
// grid's edge has no photons beyond it). The cell edges are widened by a
// relative 1e-6, far above the rounding of the hash and of the edges.
__device__ __forceinline__ float inner_gap(float v, int lo, int hi, int g, float mn, float cell) {
    float gap = __builtin_inff();
    if (lo > 0) {
        const float b = mn + (float)lo * cell;
        gap = fminf(gap, v - (b + (fabsf(b) + fabsf(mn)) * 1e-6f));
    }
    if (hi < g - 1) {
        const float b = mn + (float)(hi + 1) * cell;
        gap = fminf(gap, (b - (fabsf(b) + fabsf(mn)) * 1e-6f) - v);
    }
    return fmaxf(gap, 0.f);
}

// Photon run s of the box (linear layout: the cells of one (y, z) row;
// Morton: one cell) as [b, b + len) in grid-slot order, pruned to the cells
// that can hold a photon within the radius: a row whose (y, z) gap alone
// exceeds it is skipped, and the x extent is cut to the cells meeting the
// slab |x - qx| <= sqrt(T - gap_yz^2). Every bound is widened so that a
// photon passing the FP32 test d2 <= T is never cut: the squared gaps are
// compared with T (1 + 1e-3) (rounding of d2 and of the gaps is a few ulps),
// and the slab half-width is sqrt(T (1 + 1e-3) - gap_yz^2 + 1e-3 T) plus a
// relative 1e-6 before its cells are bounded (cell_bounds, conservative
// against the grid's own monotone cell_coord).
// The kept candidates are a subset of the reference's box holding all of
// its candidates within r, so results are unchanged.
// The cells [xl, xh] that the grid's hash (cell_coord: the correctly
// rounded quotient (p - mn) / cell, truncated and clamped to [0, g - 1];
// monotone in p) gives the positions in [lo, hi]: the quotients are taken
// with the hardware reciprocal, within 2^-21 relative of the divided ones,
// moved out by a relative and an absolute 2^-20, floored and clamped like
// the hash, so every such position's cell is inside (a bound can only come
// out one cell wider).
__device__ __forceinline__ void cell_bounds(float lo, float hi, float mn, float rcell, int g, int& xl, int& xh) {
    float tl = (lo - mn) * rcell, th = (hi - mn) * rcell;
    tl = tl - (fabsf(tl) * 0x1p-20f + 0x1p-20f);
    th = th + (fabsf(th) * 0x1p-20f + 0x1p-20f);
    const float top = (float)(g - 1);
    xl = (int)floorf(fminf(fmaxf(tl, 0.f), top));  // (NaN gives 0 and g - 1)
    xh = (int)floorf(fmaxf(fminf(th, top), 0.f));
}

// q = s / d and r = s % d for s < 2^20 (and d >= 1): (s + 0.5) / d is at
// least 0.5 / d from the integers around it, and the product with the
// hardware reciprocal is within (s + 0.5) 2^-22 / d of it.
__device__ __forceinline__ void small_divmod(int s, int d, float rd, int& q, int& r) {
    q = (int)(((float)s + 0.5f) * rd);
    r = s - q * d;
}

// The run of one (y, z) row (linear layout) over the cells [xlo, xhi] that
// can hold a photon within the bound T.
__device__ __forceinline__ bool row_cells(const GridGeom& G, const uint32_t* __restrict__ starts,
                                          const uint32_t* __restrict__ sizes, int y, int z, int xlo, int xhi, float qx,
                                          float qy, float qz, float T, uint32_t& b, uint32_t& len) {
    const float thr = T * 1.001f;
    const float gy = axis_gap(qy, y, G.g[1], G.mn[1], G.cell), gz = axis_gap(qz, z, G.g[2], G.mn[2], G.cell);
    const float dyz2 = gy * gy + gz * gz;
    if (!(dyz2 <= thr)) return false;
    // (the hardware square root: its ulp is far inside the margins)
    const float dx = __builtin_amdgcn_sqrtf(thr - dyz2 + 1e-3f * T);
    const float e = (fabsf(qx) + dx) * 1e-6f;
    int xl, xh;
    cell_bounds(qx - dx - e, qx + dx + e, G.mn[0], __builtin_amdgcn_rcpf(G.cell), G.g[0], xl, xh);
    xl = max(xlo, xl);
    xh = min(xhi, xh);
    if (xl > xh) return false;
    const uint32_t c0 = pmd::cell_index(G, xl, y, z);
    const uint32_t c1 = c0 + (uint32_t)(xh - xl);
    b = starts[c0];
    len = starts[c1] + sizes[c1] - b;
    return true;
}

__device__ __forceinline__ bool row_span(const GridGeom& G, const uint32_t* __restrict__ starts,
                                         const uint32_t* __restrict__ sizes, const Box& B, int s, float qx, float qy,
                                         float qz, float T, uint32_t& b, uint32_t& len) {
    const int nx = B.hi[0] - B.lo[0] + 1, ny = B.hi[1] - B.lo[1] + 1;
    b = 0;
    len = 0;
    if (G.layout == PM_LAYOUT_LINEAR) {
        const int nz = B.hi[2] - B.lo[2] + 1;
        int zi, yi;
        if (ny * nz < (1 << 20))
            small_divmod(s, ny, __builtin_amdgcn_rcpf((float)ny), zi, yi);
        else
            zi = s / ny, yi = s % ny;
        return row_cells(G, starts, sizes, B.lo[1] + yi, B.lo[2] + zi, B.lo[0], B.hi[0], qx, qy, qz, T, b, len);
    }
    const int x = B.lo[0] + s % nx, t = s / nx;
    const int y = B.lo[1] + t % ny, z = B.lo[2] + t / ny;
    const float gx = axis_gap(qx, x, G.g[0], G.mn[0], G.cell), gy = axis_gap(qy, y, G.g[1], G.mn[1], G.cell),
                gz = axis_gap(qz, z, G.g[2], G.mn[2], G.cell);
    if (!(gx * gx + gy * gy + gz * gz <= T * 1.001f)) return false;
    const uint32_t c = pmd::cell_index(G, x, y, z);
    b = starts[c];
    len = sizes[c];
    return true;
}

// Visit every candidate of the box, 64 per step, calling
// f(valid, slot, d2) on all lanes (valid = lane holds a candidate; d2 is
// computed on every lane). Runs of photons (rows) are held one per lane; a
// scalar cursor walks them (all control is wave-uniform, in SGPRs), and the
// next step's positions are loaded, unconditionally, before the current step
// is processed: a lane past its run reads a neighbouring photon, or 0 past
// the end of the block, and is masked by `valid`.
template <class F>
__device__ __forceinline__ void walk(const KnnParams& P, uint32_t lane, const Box& B, float qx, float qy, float qz,
                                     F&& f) {
    const int nx = B.hi[0] - B.lo[0] + 1, ny = B.hi[1] - B.lo[1] + 1, nz = B.hi[2] - B.lo[2] + 1;
    const bool linear = P.G.layout == PM_LAYOUT_LINEAR;
    const int nseg = linear ? ny * nz : nx * ny * nz;
    const __amdgpu_buffer_rsrc_t rx = plane_rsrc(P.px, P.n), ry = plane_rsrc(P.py, P.n), rz = plane_rsrc(P.pz, P.n);
    for (int sbase = 0; sbase < nseg; sbase += 64) {
        const int s = sbase + (int)lane;
        uint32_t b = 0, len = 0;
        if (s < nseg) row_span(P.G, P.starts, P.sizes, B, s, qx, qy, qz, P.T, b, len);
        const int ns = min(64, nseg - sbase);
        // Non-empty rows as a lane mask; the cursor visits them in order.
        uint64_t rows = wballot(len > 0) & (ns == 64 ? ~0ull : ((1ull << ns) - 1));
        if (!rows) continue;
        int cs = __builtin_ctzll(rows);
        rows &= rows - 1;
        uint32_t rb = __builtin_amdgcn_readlane(b, cs), rl = __builtin_amdgcn_readlane(len, cs), cc = 0;
        bool v0 = lane < rl;
        uint32_t o0 = (rb + lane) * 4u;
        float x0 = bload(rx, o0), y0 = bload(ry, o0), z0 = bload(rz, o0);
        for (;;) {
            // next step: same row if it has more, else the next non-empty row
            bool has_next = true;
            uint32_t ncc = cc + 64, nrb = rb, nrl = rl;
            if (ncc >= rl) {
                if (!rows) {
                    has_next = false;
                } else {
                    int ncs = __builtin_ctzll(rows);
                    rows &= rows - 1;
                    nrb = __builtin_amdgcn_readlane(b, ncs);
                    nrl = __builtin_amdgcn_readlane(len, ncs);
                    ncc = 0;
                }
            }
            // (after the last step this reads past the row once, harmlessly)
            const bool v1 = ncc + lane < nrl;
            const uint32_t o1 = (nrb + ncc + lane) * 4u;
            const float x1 = bload(rx, o1), y1 = bload(ry, o1), z1 = bload(rz, o1);
            f(v0, o0 >> 2, dist2(x0, y0, z0, qx, qy, qz));
            if (!has_next) break;
            cc = __builtin_amdgcn_readfirstlane(ncc);
            rb = __builtin_amdgcn_readfirstlane(nrb);
            rl = __builtin_amdgcn_readfirstlane(nrl);
            v0 = v1;
            o0 = o1;
            x0 = x1;
            y0 = y1;
            z0 = z1;
        }
    }
}

// walk with 128-candidate steps over the runs laid end to end: a step is
// the next 128 positions of the concatenated runs (lane l holds positions
// p + l and p + 64 + l), so runs shorter than a step share one instead of
// leaving lanes idle, and the candidates arrive in the same order as run by
// run. Position t of run j (its stream start pre_j, first slot b_j) is slot
// b_j + t - pre_j: each lane carries the byte offset 4 (b_j - pre_j) of the
// run holding its position, updated only for the runs that start inside the
// step. The cursor (step start, next run, its start) is wave-uniform, in
// SGPRs. f(am, sa, d2a, bm, sb, d2b): am / bm are the lane masks of the
// lanes that hold a candidate (wave-uniform, SGPRs); d2 is computed on every
// lane.
//
// walk_runs: the runs held by the lanes in the mask `rows`, end = the run's
// end in the stream (the next run's start) and d4 = 4 (b - its start)
// (mod 2^32); total = the stream's length (> 0: at least one run).
template <class F>
__device__ __forceinline__ void walk_runs(__amdgpu_buffer_rsrc_t rx, __amdgpu_buffer_rsrc_t ry,
                                          __amdgpu_buffer_rsrc_t rz, uint32_t lane, uint64_t rows, uint32_t d4,
                                          uint32_t end, uint32_t total, float qx, float qy, float qz, F&& f) {
    const int ilane = (int)lane;
    const uint32_t lane4 = lane * 4u;
    // the first non-empty run starts the stream at 0
    uint32_t nstart = 0, cur = 0;
    struct Step {
        int left;  // stream positions left from the step's first
        uint32_t oa, ob;
        float xa, ya, za, xb, yb, zb;
    };
    // offsets and positions of the step at p; the runs starting before
    // p + 128 are entered (lanes at or past a run's start take its offset)
    auto load = [&](Step& w, uint32_t p) {
        uint32_t da = cur, db = cur;
        while (rows && nstart < p + 128u) {
            const int j = __builtin_ctzll(rows);
            rows &= rows - 1;
            const uint32_t dj = __builtin_amdgcn_readlane(d4, j);
            const int t0 = (int)(nstart - p);
            da = ilane >= t0 ? dj : da;
            db = ilane >= t0 - 64 ? dj : db;
            cur = dj;
            nstart = __builtin_amdgcn_readlane(end, j);
        }
        w.left = (int)(total - p);
        w.oa = da + lane4 + p * 4u;
        w.ob = db + lane4 + p * 4u + 256u;
        w.xa = bload(rx, w.oa), w.ya = bload(ry, w.oa), w.za = bload(rz, w.oa);
        w.xb = bload(rx, w.ob), w.yb = bload(ry, w.ob), w.zb = bload(rz, w.ob);
    };
    // Two register sets: each half of the loop body loads the next step
    // into one set while the other is processed, so nothing is copied.
    Step s0, s1;
    uint32_t p = 0;
    load(s0, 0);
    auto half = [&](const Step& c, Step& nxt) -> bool {
        const uint32_t pn = p + 128u;
        const bool more = pn < total;
        if (more) load(nxt, pn);
        // (each mask is one lane compare's ballot)
        f(wballot(ilane < c.left), c.oa >> 2, dist2(c.xa, c.ya, c.za, qx, qy, qz), wballot(ilane + 64 < c.left),
          c.ob >> 2, dist2(c.xb, c.yb, c.zb, qx, qy, qz));
        p = pn;
        return more;
    };
    while (half(s0, s1) && half(s1, s0)) {
    }
}

// Radiance estimate of Raytracer.cuh:110-138 over the m kept photons held in
// v (sorted); lanes own elements j*64 + lane.
template <int R>
__device__ __forceinline__ void radiance_epilogue(const KnnParams& P, const uint64_t (&v)[R], uint32_t m,
                                                  uint32_t lane, uint32_t q) {
    const float alpha = 1.818f, beta = 1.953f;
    const float pi_f = 3.141592654f;
    float res0 = 0.f, res1 = 0.f, res2 = 0.f;
    float rmax = 0.f;
    if (m > 0) {
        const int jm = (int)((m - 1) / 64);
        float dm = 0.f;
#pragma unroll
        for (int j = 0; j < R; ++j)
            if (j == jm) dm = sqrtf(__uint_as_float((uint32_t)(v[j] >> 32)));
        rmax = __shfl(dm, (int)((m - 1) & 63), 64);
        const float filter_r = __fmul_rn(rmax, rmax);
        const float denom = 1.f - expf(-beta);
        const float nx = P.nrm[q], ny = P.nrm[P.nq + q], nz = P.nrm[2 * (size_t)P.nq + q];
#pragma unroll
        for (int j = 0; j < R; ++j) {
            uint32_t e = (uint32_t)j * 64 + lane;
            if (e < m) {
                uint32_t idx = (uint32_t)v[j];
                float dx = P.dir[idx], dy = P.dir[P.n + idx], dz = P.dir[2 * (size_t)P.n + idx];
                float cosNL = __fadd_rn(__fadd_rn(__fmul_rn(nx, -dx), __fmul_rn(ny, -dy)), __fmul_rn(nz, -dz));
                if (cosNL > 0.f) {
                    float d = sqrtf(__uint_as_float((uint32_t)(v[j] >> 32)));
                    float x = __fdiv_rn(__fmul_rn(__fmul_rn(-beta, d), d), __fmul_rn(2.f, filter_r));
                    float w = __fmul_rn(alpha, 1.f - __fdiv_rn(1.f - expf(x), denom));
                    res0 += P.power[idx] * w;
                    res1 += P.power[P.n + idx] * w;
                    res2 += P.power[2 * (size_t)P.n + idx] * w;
                }
            }
        }
    }
    res0 = wave_sum_f32(res0);
    res1 = wave_sum_f32(res1);
    res2 = wave_sum_f32(res2);
    if (lane == 0) {
        float coef = 1.f;
        if (m > 0) coef = __fdiv_rn(1.f, __fmul_rn(__fmul_rn(pi_f, __fmul_rn(rmax, rmax)), 1.f));
        P.rgb[q] = m > 0 ? res0 * coef : 0.f;
        P.rgb[P.nq + q] = m > 0 ? res1 * coef : 0.f;
        P.rgb[2 * (size_t)P.nq + q] = m > 0 ? res2 * coef : 0.f;
    }
}

template <int R, int CAP>
__device__ __forceinline__ void sort_and_emit(const KnnParams& P, WaveLds<CAP>& L, uint32_t lane, uint32_t q,
                                              uint32_t cnt, uint32_t m, uint32_t hi) {
    uint64_t v[R];
    sort_keys<R, CAP>(L, lane, cnt, hi, v);
    if (P.out_idx) {
#pragma unroll
        for (int j = 0; j < R; ++j) {
            uint32_t e = (uint32_t)j * 64 + lane;
            if (e < (uint32_t)P.k) {
                bool keep = e < m;
                P.out_idx[(size_t)q * P.k + e] = keep ? (uint32_t)v[j] : 0xFFFFFFFFu;
                P.out_dist[(size_t)q * P.k + e] =
                    keep ? sqrtf(__uint_as_float((uint32_t)(v[j] >> 32))) : __builtin_inff();
            }
        }
        // slots beyond the sorted registers (k > 64*R >= cnt >= m) are empty
        for (uint32_t e = 64u * R + lane; e < (uint32_t)P.k; e += 64) {
            P.out_idx[(size_t)q * P.k + e] = 0xFFFFFFFFu;
            P.out_dist[(size_t)q * P.k + e] = __builtin_inff();
        }
    }
    if (P.out_count && lane == 0) P.out_count[q] = m;
    if (P.rgb) radiance_epilogue<R>(P, v, m, lane, q);
}

// Largest d2 of the m keys in the LDS buffer.
template <int CAP>
__device__ __forceinline__ float buffer_dmax(const WaveLds<CAP>& L, uint32_t lane, uint32_t m) {
    float d = 0.f;
    for (uint32_t e = lane; e < m; e += 64) d = fmaxf(d, __uint_as_float((uint32_t)(L.buf[e] >> 32)));
    return wave_max_nonneg_f32(d);
}

// Radiance estimate (Raytracer.cuh:110-138) over the m kept keys left in
// the LDS buffer, unsorted: the filter radius is their largest distance
// (dmax = its square) and the sum runs in buffer order (lane-strided, then a
// wave reduction of the three channels together).
//
// The filter weight w = alpha (1 - (1 - e^{-beta d^2 / (2 r^2)}) / (1 - e^{-beta}))
// is evaluated as A + B e^{x} with x = d^2 (-beta / (2 r^2)) from the squared
// distance itself (no square root), the hardware exponential, and the
// filter radius and the per-query factors (-beta / (2 r^2), 1 / (pi r^2))
// from the hardware square root and reciprocal; against the reference's FP32
// sequence of square roots, divisions and expf this moves the estimate by a
// few 1e-7 relative, inside its 1e-5 bound. The cos > 0 test keeps the
// reference's rounding. The six power and direction planes are read as raw
// buffers with one 32-bit offset per lane.
template <int CAP>
__device__ __forceinline__ void radiance_buffer(const KnnParams& P, const WaveLds<CAP>& L, uint32_t lane, uint32_t q,
                                                uint32_t m, float dmax) {
    const float alpha = 1.818f, beta = 1.953f;
    const float pi_f = 3.141592654f;
    // 1 / (1 - e^{-beta}) and log2(e), rounded to FP32
    const float inv_denom = 1.16529458f, log2e = 1.44269504f;
    // hardware square root and reciprocals (a few 1e-7 relative on the
    // estimate, inside its 1e-5 bound)
    const float rmax = __builtin_amdgcn_sqrtf(dmax);
    const float filter_r = __fmul_rn(rmax, rmax);
    float res0 = 0.f, res1 = 0.f, res2 = 0.f;
    if (m > 0) {
        // x log2(e) = d^2 * s
        const float s = -beta * __builtin_amdgcn_rcpf(2.f * filter_r) * log2e;
        const float wa = alpha * (1.f - inv_denom), wb = alpha * inv_denom;
        const float nx = P.nrm[q], ny = P.nrm[P.nq + q], nz = P.nrm[2 * (size_t)P.nq + q];
        const __amdgpu_buffer_rsrc_t rd0 = plane_rsrc(P.dir, P.n), rd1 = plane_rsrc(P.dir + P.n, P.n),
                                     rd2 = plane_rsrc(P.dir + 2 * (size_t)P.n, P.n);
        const __amdgpu_buffer_rsrc_t rp0 = plane_rsrc(P.power, P.n), rp1 = plane_rsrc(P.power + P.n, P.n),
                                     rp2 = plane_rsrc(P.power + 2 * (size_t)P.n, P.n);
        for (uint32_t base = 0; base < m; base += 64) {
            const uint32_t e = base + lane;
            if (e < m) {
                const uint64_t v = L.buf[e];
                const uint32_t off = (uint32_t)v * 4u;
                // power is read with the direction (one memory round trip),
                // and used only where the photon faces the surface
                const float dx = bload(rd0, off), dy = bload(rd1, off), dz = bload(rd2, off);
                const float p0 = bload(rp0, off), p1 = bload(rp1, off), p2 = bload(rp2, off);
                const float cosNL = __fadd_rn(__fadd_rn(__fmul_rn(nx, -dx), __fmul_rn(ny, -dy)), __fmul_rn(nz, -dz));
                if (cosNL > 0.f) {
                    const float w = wa + wb * __builtin_amdgcn_exp2f(__uint_as_float((uint32_t)(v >> 32)) * s);
                    res0 += p0 * w;
                    res1 += p1 * w;
                    res2 += p2 * w;
                }
            }
        }
    }
    // channel 0 in lane 15, 2 in lane 31, 1 in lane 47
    const float tot = wave_sum3_f32(res0, res1, res2);
    if ((lane & 15) == 15 && lane < 63) {
        const float coef = __builtin_amdgcn_rcpf(__fmul_rn(pi_f, __fmul_rn(rmax, rmax)));
        const uint32_t plane = lane == 15 ? 0u : lane == 31 ? 2u : 1u;
        P.rgb[(size_t)plane * P.nq + q] = m > 0 ? tot * coef : 0.f;
    }
}

// The end of a query: cnt keys in the buffer, all of them with d2 bits below
// hi, hold the k nearest (or everything within the radius).
template <int CAP, bool kLists>
__device__ __forceinline__ void finish(const KnnParams& P, WaveLds<CAP>& L, uint32_t lane, uint32_t q, uint32_t cnt,
                                       uint32_t hi) {
    const uint32_t k = (uint32_t)P.k;
    const uint32_t m = cnt < k ? cnt : k;
    if (kLists && P.out_idx) {
        constexpr uint32_t kMost = CAP == 768 ? 512u : 256u;  // (the largest k of the buffer's lists)
        if (cnt > kMost) {
            uint64_t khi = (uint64_t)hi << 32;
            cnt = buf_select<CAP>(L, lane, cnt, k, kMost, P.bT, khi);
            hi = (uint32_t)((khi + 0xffffffffull) >> 32);
            wave_sync();
        }
        if (cnt <= 64)
            sort_and_emit<1, CAP>(P, L, lane, q, cnt, m, hi);
        else if (cnt <= 128)
            sort_and_emit<2, CAP>(P, L, lane, q, cnt, m, hi);
        else if (CAP != 768 || cnt <= 256)
            sort_and_emit<4, CAP>(P, L, lane, q, cnt, m, hi);
        else
            sort_and_emit<8, CAP>(P, L, lane, q, cnt, m, hi);
        return;
    }
    // no neighbour lists: narrow to exactly the k smallest and estimate
    // from the buffer without sorting
    if (P.out_count && lane == 0) P.out_count[q] = m;
    if (!P.rgb) return;
    float dmax;
    if (cnt > k)
        dmax = lin_select<CAP>(L, lane, cnt, k, hi, P.bT);
    else
        dmax = buffer_dmax<CAP>(L, lane, m);
    wave_sync();
    radiance_buffer<CAP>(P, L, lane, q, m, dmax);
}

// The candidate box of query q: its cell +- rc, clamped (PhotonGrid.cu:262-272).
__device__ __forceinline__ void box_of(const KnnParams& P, uint32_t q, Box& B, float& qx, float& qy, float& qz) {
    // the query is the wave's: its coordinates (and so the box, the row
    // count and the cursor of walk) are wave-uniform, held in SGPRs
    qx = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(P.qx[q])));
    qy = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(P.qy[q])));
    qz = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(P.qz[q])));
    const float qv[3] = {qx, qy, qz};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        int c = pmd::cell_coord(qv[a], P.G.mn[a], P.G.cell, P.G.g[a]);
        B.lo[a] = max(0, c - P.rc);
        B.hi[a] = min(P.G.g[a] - 1, c + P.rc);
    }
}

// XCD-chunked order: XCD x takes chunks x, x + 8, ... of 2^shift consecutive
// workgroups (the grid is rounded up to a multiple of 8 chunks).
constexpr uint32_t kXcdChunk = 256;  // queries / 4 in a chunk, at most
__device__ __forceinline__ uint32_t xcd_chunked(uint32_t b, uint32_t shift) {
    const uint32_t x = b % 8, i = b / 8;
    return ((((i >> shift) * 8 + x)) << shift) + (i & ((1u << shift) - 1u));
}
// The chunk of a launch of nblk workgroups of gq queries a wave: about
// kXcdChunk x 4 queries, and no more than leaves every XCD one (a small
// launch is not padded by more than 8 workgroups a chunk).
inline uint32_t xcd_shift_for(uint32_t nblk, uint32_t gq) {
    uint32_t s = 0;
    while ((2u << s) * gq <= kXcdChunk && (uint64_t)(16u << s) <= nblk) ++s;
    return s;
}
inline uint32_t xcd_round(uint32_t nblk, uint32_t shift) { return pm::div_up(nblk, 8u << shift) * (8u << shift); }

// Query of this wave in a one-wave-per-query launch (XCD-aware block order,
// optional processing order); false past the end (wave-uniform).
__device__ __forceinline__ bool query_of_wave(const KnnParams& P, uint32_t& q) {
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t blk = P.remap == 2 ? xcd_chunked(blockIdx.x, P.xcd_shift)
                         : P.remap   ? pmd::xcd_remap(blockIdx.x, gridDim.x)
                                     : blockIdx.x;
    const uint32_t ql = blk * kWaves + wave;
    if (ql >= P.nq || (P.nq_dev && ql >= *P.nq_dev)) return false;
    q = __builtin_amdgcn_readfirstlane(P.order ? P.order[ql] : ql);
    return true;
}

// A kernel parameter record read by scalar loads where it is used: from the
// launch's own argument segment, or a batch's job table. `opaque` keeps a
// use's loads from being hoisted (and held in SGPRs) across what is before
// it.
typedef const __attribute__((address_space(4))) KnnParams* ParamsPtr;
__device__ __forceinline__ ParamsPtr opaque(ParamsPtr p) {
    asm volatile("" : "+s"(p));
    return p;
}
__device__ __forceinline__ GridGeom geom_of(ParamsPtr kp) {
    GridGeom G;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        G.mn[a] = kp->G.mn[a];
        G.g[a] = kp->G.g[a];
    }
    G.cell = kp->G.cell;
    G.layout = kp->G.layout;
    return G;
}
// the finish's parameters (every field it reads)
__device__ __forceinline__ void finish_params(KnnParams& Pf, ParamsPtr kp) {
    Pf.k = kp->k;
    Pf.n = kp->n;
    Pf.nq = kp->nq;
    Pf.bT = kp->bT;
    Pf.power = kp->power;
    Pf.dir = kp->dir;
    Pf.nrm = kp->nrm;
    Pf.rgb = kp->rgb;
    Pf.out_idx = kp->out_idx;
    Pf.out_dist = kp->out_dist;
    Pf.out_count = kp->out_count;
}

// Keys that a narrowing of a buffer of CAP leaves at most: at least the
// largest k that the buffer serves (256, or 512), and room for a step.
template <int CAP>
constexpr uint32_t kNarrowTo = CAP == 512 ? 256 : 512;

// What a narrowing reads; kOne: held through the walk (two scalar reads at each
// narrowing, 1 us of 56 where a query's walk has dozens of them).
struct Narrow {
    uint32_t k, bT;
};

// One step of the streaming selection over two candidates per lane (index
// sa / sb, squared distance d2a / d2b, lanes holding one: masks am / bm):
// appends the keys whose d2 bits lie below the acceptance bound hi to the
// LDS buffer, and narrows the buffer first when the step would overflow it.
// hi never exceeds bits(T) + 1, so an accepted key is within the radius (d2
// >= 0: its bits order as its value; a NaN d2 is above every bound). A
// narrowing's bound on whole keys is rounded up to d2 bits: the keys this
// lets in besides lie above k kept ones, and are dropped by the finish.
// Every predicate is a ballot of a plain compare combined in SGPRs; the
// writing lanes come back from their mask.
template <int CAP, bool kOne>
__device__ __forceinline__ void push2(WaveLds<CAP>& L, uint32_t lane, ParamsPtr kp0, Narrow own, uint64_t am,
                                      uint32_t sa, float d2a, uint64_t bm, uint32_t sb, float d2b, uint32_t& cnt,
                                      uint32_t& hi) {
    uint64_t bala = am & wballot(__float_as_uint(d2a) < hi), balb = bm & wballot(__float_as_uint(d2b) < hi);
    uint32_t na = (uint32_t)__popcll(bala), nb = (uint32_t)__popcll(balb);
    if (cnt + na + nb > (uint32_t)CAP) {
        // leaves at most kNarrowTo keys, room for this step's 128
        wave_sync();
        if constexpr (!kOne) {
            ParamsPtr kp = opaque(kp0);
            own = Narrow{(uint32_t)kp->k, kp->bT};
        }
        uint64_t khi = (uint64_t)hi << 32;
        cnt = buf_select<CAP>(L, lane, cnt, own.k, kNarrowTo<CAP>, own.bT, khi);
        hi = (uint32_t)((khi + 0xffffffffull) >> 32);
        bala = am & wballot(__float_as_uint(d2a) < hi);
        balb = bm & wballot(__float_as_uint(d2b) < hi);
        na = (uint32_t)__popcll(bala);
        nb = (uint32_t)__popcll(balb);
    }
    // (the sum is pinned ahead of the lane branches: computed in both arms of
    // one it would come back as a per-lane value, and the count, the branch
    // above and the whole loop with it)
    const uint32_t cb = __builtin_amdgcn_readfirstlane(cnt + na);
    if (__builtin_amdgcn_inverse_ballot_w64(bala)) L.buf[cnt + mbcnt(bala)] = make_key(d2a, sa);
    if (__builtin_amdgcn_inverse_ballot_w64(balb)) L.buf[cb + mbcnt(balb)] = make_key(d2b, sb);
    cnt = cb + nb;
}

// Single pass: in-radius keys stream into an LDS buffer of CAP keys; when it
// would overflow, buf_select keeps only the smallest bin range holding >= k
// keys and tightens the acceptance bound. Exact: a dropped key has >= k kept
// keys below it.
//
// With h > 0 the walk first covers only the inner box (the query's cell
// +- h), and only keys closer than every photon outside it are kept (its
// squared face gap less a few ulps of rounding). Where the first walk's rows
// hold many more candidates N than k, its bound b is lowered to the squared
// radius expected to hold somewhat more than k of them, and the rows and
// cells are pruned to that: on surfaces the photons within b are about
// N / (1 + 0.6 cell / sqrt(b))^2 (the walked cells against the disc), evenly
// in d2; `guess` = 1.2 (k + 3 sqrt(k) + 2) (split_waves) leaves three standard deviations
// and a fifth for an uneven map (lists of k <= 128 do without the fifth). If the first walk finds at least k keys, the
// k smallest are the answer; otherwise the query walks the whole box again
// from an empty buffer, to the radius or, for lists, first to a bound sized
// from the count so far (next_bound). Every outcome is exact.
//
// One wave, the nqw <= gq queries at positions p0, p0 + stride, ... of
// `order` (entries less qb; null: the positions themselves). The set-up
// (cell, box, face gap, and the photon run of every row) is worked for all of
// them at once, lane i nr + s taking row s of query i: it is about 230 VALU
// instructions whatever the lanes in use, as many as one query's walk and
// finish on a dense map. Each query then walks its rows from those lanes.
// The stride is the launch's wave count: waves that run side by side are at
// neighbouring queries (their cells' lines are shared in L1 and L2), and a
// run of queries with crowded boxes (a caustic's focus) is spread over as
// many waves as one query a wave would give it. With consecutive queries per
// wave instead, L2 reads doubled and a frame's gathers took 2.9 ms, not 1.9.
// A wave's queries after their set-up: per lane, the query's index, position
// and first bound (d2 bits, exclusive), and the run of the lane's row (as
// walk_runs takes it); rows: the lanes whose run is not empty.
struct WaveQueries {
    uint32_t q, hib, d4, end;
    float x, y, z;
    uint64_t rows;
};
__device__ __forceinline__ void setup_queries(ParamsPtr kp0, uint32_t lane, const uint32_t* __restrict__ order,
                                              uint32_t p0, uint32_t stride, uint32_t qb, uint32_t nqw,
                                              WaveQueries& W) {
    ParamsPtr kp = opaque(kp0);
    const GridGeom G = geom_of(kp);
    const int nr = kp->nr;
    int i = 0, s = 0;
    if (nr > 0) small_divmod((int)lane, nr, __builtin_amdgcn_rcpf((float)nr), i, s);
    const bool mine = nr > 0 && (uint32_t)i < nqw;
    const uint32_t pos = p0 + min((uint32_t)i, nqw - 1u) * stride;
    const uint32_t q = (order ? order[pos] : pos) - qb;
    const float x = kp->qx[q], y = kp->qy[q], z = kp->qz[q];
    const int cx = pmd::cell_coord(x, G.mn[0], G.cell, G.g[0]), cy = pmd::cell_coord(y, G.mn[1], G.cell, G.g[1]),
              cz = pmd::cell_coord(z, G.mn[2], G.cell, G.g[2]);
    const float T = kp->T;
    uint32_t hib = __float_as_uint(T) + 1u, d4 = 0, end = 0;
    uint64_t rows_all = 0;
    float Trow = T;
    const int h = kp->h;
    if (h > 0) {
        const float gx = inner_gap(x, max(0, cx - h), min(G.g[0] - 1, cx + h), G.g[0], G.mn[0], G.cell),
                    gy = inner_gap(y, max(0, cy - h), min(G.g[1] - 1, cy + h), G.g[1], G.mn[1], G.cell),
                    gz = inner_gap(z, max(0, cz - h), min(G.g[2] - 1, cz + h), G.g[2], G.mn[2], G.cell);
        const float gap = fminf(fminf(gx, gy), gz);
        hib = min(__float_as_uint(gap * gap * 0.999f), hib);
        // (only keys below the bound are kept: the rows are pruned with it)
        Trow = fminf(T, __uint_as_float(hib));
    }
    if (nr > 0) {
        const int w = kp->w, side = 2 * w + 1;
        int zi, yi;
        small_divmod(s, side, __builtin_amdgcn_rcpf((float)side), zi, yi);
        const int yy = cy - w + yi, zz = cz - w + zi;
        const bool row = mine && yy >= 0 && yy < G.g[1] && zz >= 0 && zz < G.g[2];
        const int xlo = max(0, cx - w), xhi = min(G.g[0] - 1, cx + w);
        const float cr = 1.f + 0.6f * G.cell * __builtin_amdgcn_rsqf(Trow);
        const float aim = kp->guess * cr * cr;
        uint32_t len;
        for (bool first = true;; first = false) {
            uint32_t b = 0;
            len = 0;
            if (row) row_cells(G, kp->starts, kp->sizes, yy, zz, xlo, xhi, x, y, z, Trow, b, len);
            const uint32_t incl = wave_incl_scan(len, lane);
            // each query's stream starts at 0: less the lanes before its first
            const uint32_t before = __shfl(incl, i > 0 ? i * nr - 1 : 0, 64);
            end = incl - (i > 0 ? before : 0u);
            d4 = (b + len - end) * 4u;
            if (!first) break;
            // many more candidates than k: a smaller bound first, when
            // that is so for most of the wave's queries or far so for one
            const uint32_t all = __shfl(end, min(i * nr + nr - 1, 63), 64);
            const bool crowded = mine && aim < 0.7f * (float)all;
            const int nc = __builtin_popcountll(wballot(crowded));
            if (2 * nc < (int)nqw * nr && !wballot(mine && aim < 0.2f * (float)all)) break;
            if (crowded) {
                Trow = Trow * aim * __builtin_amdgcn_rcpf((float)all);
                hib = min(hib, __float_as_uint(Trow));
            }
        }
        rows_all = wballot(len > 0);
    }
    W.q = q;
    W.hib = hib;
    W.d4 = d4;
    W.end = end;
    W.x = x;
    W.y = y;
    W.z = z;
    W.rows = rows_all;
}

// setup_queries for the one query of a wave (at position p0), whose values are
// then wave-uniform: the three axes' cells and face gaps are worked side by side
// in lanes 0..2, and there is no guess. 83 VALU instructions fewer of a query's 455;
// 8000 to 14000 unsorted queries in 200k photons (k = 64 within r = 0.02, the mean
// of eight maps) 17.2 to 24.0 us with setup_queries, 16.2 to 22.0 so.
__device__ __forceinline__ void setup_query(ParamsPtr kp0, uint32_t lane, const uint32_t* __restrict__ order,
                                            uint32_t p0, uint32_t qb, WaveQueries& W) {
    ParamsPtr kp = opaque(kp0);
    const GridGeom G = geom_of(kp);
    const auto uni = [](float v) { return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v))); };
    const uint32_t q = __builtin_amdgcn_readfirstlane(order ? order[p0] : p0) - qb;
    const float x = uni(kp->qx[q]), y = uni(kp->qy[q]), z = uni(kp->qz[q]);
    const float v = lane == 1 ? y : lane == 2 ? z : x, mn = lane == 1 ? G.mn[1] : lane == 2 ? G.mn[2] : G.mn[0];
    const int g = lane == 1 ? G.g[1] : lane == 2 ? G.g[2] : G.g[0];
    const int c = pmd::cell_coord(v, mn, G.cell, g);
    const int cx = __builtin_amdgcn_readlane(c, 0), cy = __builtin_amdgcn_readlane(c, 1),
              cz = __builtin_amdgcn_readlane(c, 2);
    const float T = kp->T;
    uint32_t hib = __float_as_uint(T) + 1u, len = 0, b = 0;
    float Trow = T;
    const int h = kp->h, nr = kp->nr;
    if (h > 0) {
        const uint32_t gb = __float_as_uint(inner_gap(v, max(0, c - h), min(g - 1, c + h), g, mn, G.cell));
        const float gap = fminf(fminf(__uint_as_float(__builtin_amdgcn_readlane(gb, 0)),
                                      __uint_as_float(__builtin_amdgcn_readlane(gb, 1))),
                                __uint_as_float(__builtin_amdgcn_readlane(gb, 2)));
        hib = __builtin_amdgcn_readfirstlane(min(__float_as_uint(gap * gap * 0.999f), hib));
        Trow = fminf(T, __uint_as_float(hib));
    }
    W.end = W.d4 = 0;
    W.rows = 0;
    if (nr > 0) {
        const int w = kp->w, side = 2 * w + 1;
        int zi, yi;
        small_divmod((int)lane, side, __builtin_amdgcn_rcpf((float)side), zi, yi);
        const int yy = cy - w + yi, zz = cz - w + zi;
        if ((int)lane < nr && yy >= 0 && yy < G.g[1] && zz >= 0 && zz < G.g[2])
            row_cells(G, kp->starts, kp->sizes, yy, zz, max(0, cx - w), min(G.g[0] - 1, cx + w), x, y, z, Trow, b, len);
        W.end = wave_incl_scan(len, lane);
        W.d4 = (b + len - W.end) * 4u;
        W.rows = wballot(len > 0);
    }
    W.q = q;
    W.hib = hib;
    W.x = x;
    W.y = y;
    W.z = z;
}
// A value of the wave's queries for the one whose first lane is lb.
template <bool kOne>
__device__ __forceinline__ uint32_t of_query(uint32_t v, uint32_t lb) {
    return kOne ? __builtin_amdgcn_readfirstlane(v) : __builtin_amdgcn_readlane(v, lb);
}
template <bool kOne>
__device__ __forceinline__ float of_query(float v, uint32_t lb) {
    return __uint_as_float(of_query<kOne>(__float_as_uint(v), lb));
}

// f (as walk_runs calls it) over the candidates of the query whose first
// lane is lb: the rows set up for it (batch), or the whole box, or the inner
// one, looked up now, with rows and cells pruned to the d2 bits below hi.
template <bool kOne, class F>
__device__ __forceinline__ void walk_query(ParamsPtr kp0, uint32_t lane, const WaveQueries& W, uint32_t lb, bool batch,
                                           bool inner, uint32_t hi, F&& f) {
    ParamsPtr kp = opaque(kp0);
    const int nr = kp->nr;
    const float qx = of_query<kOne>(W.x, lb), qy = of_query<kOne>(W.y, lb), qz = of_query<kOne>(W.z, lb);
    const uint32_t n = kp->n;
    const __amdgpu_buffer_rsrc_t rx = plane_rsrc(kp->px, n), ry = plane_rsrc(kp->py, n), rz = plane_rsrc(kp->pz, n);
    for (int sbase = 0;; sbase += 64) {
        uint32_t cd4 = W.d4, cend = W.end, total;
        uint64_t rows;
        bool last = true;
        if (batch) {
            rows = kOne ? W.rows : W.rows & ((~0ull >> (64 - nr)) << lb);
            total = __builtin_amdgcn_readlane(W.end, lb + (uint32_t)nr - 1u);
        } else {
            // 64 rows (Morton: cells) of the box, one per lane
            ParamsPtr kc = opaque(kp0);
            const GridGeom G = geom_of(kc);
            const int w = inner ? kc->h : kc->rc;
            const float qv[3] = {qx, qy, qz};
            Box B;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const int c = __builtin_amdgcn_readfirstlane(pmd::cell_coord(qv[a], G.mn[a], G.cell, G.g[a]));
                B.lo[a] = max(0, c - w);
                B.hi[a] = min(G.g[a] - 1, c + w);
            }
            const int nx = B.hi[0] - B.lo[0] + 1, nyz = (B.hi[1] - B.lo[1] + 1) * (B.hi[2] - B.lo[2] + 1);
            const int nseg = G.layout == PM_LAYOUT_LINEAR ? nyz : nx * nyz;
            const int sr = sbase + (int)lane;
            const float Trow = fminf(kc->T, __uint_as_float(hi));
            uint32_t b = 0, len = 0;
            if (sr < nseg) row_span(G, kc->starts, kc->sizes, B, sr, qx, qy, qz, Trow, b, len);
            cend = wave_incl_scan(len, lane);
            cd4 = (b + len - cend) * 4u;
            rows = wballot(len > 0);
            total = __builtin_amdgcn_readlane(cend, 63);
            last = sbase + 64 >= nseg;
        }
        if (total > 0) walk_runs(rx, ry, rz, lane, rows, cd4, cend, total, qx, qy, qz, f);
        if (last) break;
    }
}

// The bound after a list query's first walk found too few keys (cnt < k below
// hi): a squared radius that should hold half as many again as needed, where
// that is well below the radius, else the radius. 3 % of the queries come
// here, but a whole box is several times a guessed walk and the longest of a
// wave's queries: 1M sorted queries in 4M photons, k = 50, cells of the radius:
// 1262 -> 1141 us. The estimates' kernels walk the whole box at once: there
// the loop's extra state costs the compiled walk 4 to 6 % (1480 -> 1537 us at a
// 1280x720 frame), as much as the shorter walks give.
__device__ __forceinline__ uint32_t next_bound(uint32_t hi, uint32_t cnt, bool first, ParamsPtr kp) {
    const float T = kp->T;
    if (first && cnt > 0) {
        const float est = __uint_as_float(hi) * 1.5f * (float)kp->k * __builtin_amdgcn_rcpf((float)cnt);
        if (est < 0.7f * T) return __builtin_amdgcn_readfirstlane(__float_as_uint(est));
    }
    return __float_as_uint(T) + 1u;
}

template <int CAP, bool kLists, bool kOne>
__device__ __forceinline__ void stream_wave(ParamsPtr kp0, WaveLds<CAP>& L, uint32_t lane,
                                            const uint32_t* __restrict__ order, uint32_t p0, uint32_t stride,
                                            uint32_t qb, uint32_t nqw) {
    WaveQueries W;
    if constexpr (kOne)
        setup_query(kp0, lane, order, p0, qb, W);
    else
        setup_queries(kp0, lane, order, p0, stride, qb, nqw, W);
    for (uint32_t i = 0; i < (kOne ? 1u : nqw); ++i) {
        uint32_t cnt, hi, lb;
        {
            ParamsPtr kp = opaque(kp0);
            lb = kOne ? 0u : i * (uint32_t)kp->nr;
            hi = of_query<kOne>(W.hib, lb);
            // (a first walk below the radius is of the inner box when there
            // is one)
            const uint32_t hit = __float_as_uint(kp->T) + 1u;
            bool batch = kp->nr > 0, inner = kp->h > 0 && kp->nr == 0, part = hi < hit;
            [[maybe_unused]] bool first = true;
            const Narrow own = kOne ? Narrow{(uint32_t)kp->k, kp->bT} : Narrow{};
            for (;;) {
                cnt = 0;
                walk_query<kOne>(kp0, lane, W, lb, batch, inner, hi,
                           [&](uint64_t am, uint32_t sa, float d2a, uint64_t bm, uint32_t sb, float d2b) {
                               push2<CAP, kOne>(L, lane, kp0, own, am, sa, d2a, bm, sb, d2b, cnt, hi);
                           });
                wave_sync();
                // with at least k such keys, the k smallest keys overall are
                // among them (the buffer holds every in-radius key below its
                // bound, or at least k of them once narrowed)
                if (!part) break;
                kp = opaque(kp0);
                if (cnt >= (uint32_t)kp->k) break;
                // otherwise the whole box from an empty buffer
                if constexpr (kLists) {
                    hi = next_bound(hi, cnt, first, kp);
                    part = hi <= __float_as_uint(kp->T);
                    inner = batch = first = false;
                } else {
                    inner = part = batch = false;
                    hi = __float_as_uint(kp->T) + 1u;
                }
                wave_sync();
            }
        }
        // The count within the radius that the finish needs is min(found, k),
        // and that is min(cnt, k): without a narrowing the buffer holds every
        // key within the radius (cnt = found), and a narrowing keeps at least
        // k (it starts above CAP - 128 >= k keys), so cnt >= k after one.
        KnnParams Pf;
        finish_params(Pf, opaque(kp0));
        finish<CAP, kLists>(Pf, L, lane, of_query<kOne>(W.q, lb), cnt, hi);
        if (!kOne) wave_sync();  // the buffer is read before the next query's keys
    }
}

// The queries of wave u among n_waves: u, u + n_waves, ...
__device__ __forceinline__ uint32_t wave_queries(uint32_t u, uint32_t n_waves, uint32_t gq, uint32_t nq) {
    return min(gq, (nq - u - 1u) / n_waves + 1u);  // u < nq
}

// The argument lines are read one after the other as their values are needed,
// each a first miss of the XCD's; here all at once (100 queries 9.6 -> 8.8 us).
__device__ __forceinline__ void touch_args() {
    typedef const __attribute__((address_space(4))) uint32_t* WordPtr;
    WordPtr w = (WordPtr)__builtin_amdgcn_kernarg_segment_ptr();
    static_assert(sizeof(KnnParams) > 3 * 64 && sizeof(KnnParams) <= 4 * 64, "four lines");
    asm volatile("" ::"s"(w[0]), "s"(w[16]), "s"(w[32]), "s"(w[48]));
}

// The single-map launch, waves in the XCD-aware order. CAP = 512: 17 KB of
// LDS per workgroup; CAP = 768 (256 < k <= 512): 25 KB, 6 waves
// per SIMD; CAP = 1024 (a tuning variant: fewer narrowings) is LDS-limited to
// 4.
template <int CAP, bool kLists, bool kOne = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(CAP == 512 ? 7 : CAP == 768 ? (kLists ? 5 : 6) : 4))) void k_knn_stream(
    KnnParams P) {
    __shared__ WaveLds<CAP> lds[kWaves];
    if (kOne) touch_args();
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t blk = P.remap == 2 ? xcd_chunked(blockIdx.x, P.xcd_shift)
                         : P.remap   ? pmd::xcd_remap(blockIdx.x, gridDim.x)
                                     : blockIdx.x;
    const uint32_t nq = P.nq_dev ? min(P.nq, *P.nq_dev) : P.nq;
    const uint32_t u = blk * kWaves + wave;
    if (u >= nq || u >= P.n_waves) return;  // wave-uniform; no workgroup barriers below
    stream_wave<CAP, kLists, kOne>((ParamsPtr)__builtin_amdgcn_kernarg_segment_ptr(), lds[wave], threadIdx.x & 63,
                                   P.order, u, P.n_waves, 0u, wave_queries(u, P.n_waves, (uint32_t)P.gq, nq));
}

// Neighbour lists of k = 513..2048 (and counts alone above k = 256): one wave
// per workgroup with a CAP-key LDS buffer (CAP >= 2k), 64 candidates a step;
// the final selection narrows the buffer to exactly the k smallest keys, which
// a bitonic network sorts in LDS. Up to k = 512 the stream with a 768-key buffer
// and a register sort took its place: 2482 lists of k = 400 532 -> 194 us, 100k of
// k = 300 2656 -> 650, of k = 512 4761 -> 1185.
template <int CAP>
__device__ __forceinline__ void large_one(const KnnParams& P, WaveLds<CAP>& L, uint32_t lane, uint32_t q) {
    Box B;
    float qx, qy, qz;
    box_of(P, q, B, qx, qy, qz);
    const float T = P.T;
    const uint32_t k = (uint32_t)P.k;
    uint32_t cnt = 0, found = 0;
    uint64_t khi = ~0ull;
    walk(P, lane, B, qx, qy, qz, [&](bool valid, uint32_t slot, float d2) {
        // each ballot is taken of a plain compare (no bool round trip): an
        // invalid lane gets a threshold no d2 >= 0 (or NaN) passes
        const bool in = d2 <= (valid ? T : -1.0f);
        const uint64_t bin = wballot(in);
        found += (uint32_t)__popcll(bin);
        uint64_t key = make_key(d2, slot);
        const bool below = key < khi;
        bool acc = in && below;
        uint64_t bal = bin & wballot(below);
        uint32_t na = (uint32_t)__popcll(bal);
        if (cnt + na > (uint32_t)CAP) {
            wave_sync();
            cnt = buf_select<CAP>(L, lane, cnt, k, CAP / 2, P.bT, khi);
            acc = acc && key < khi;
            bal = wballot(acc);
            na = (uint32_t)__popcll(bal);
        }
        if (acc) L.buf[cnt + mbcnt(bal)] = key;
        cnt += na;
    });
    wave_sync();
    const uint32_t m = found < k ? found : k;
    cnt = buf_select<CAP>(L, lane, cnt, k, k, P.bT, khi);  // exactly min(k, found) keys remain
    wave_sync();
    if (!P.out_idx) {  // radiance / counts only: no sort needed
        if (P.out_count && lane == 0) P.out_count[q] = m;
        if (P.rgb) radiance_buffer<CAP>(P, L, lane, q, m, buffer_dmax<CAP>(L, lane, m));
        return;
    }
    uint32_t n2 = 64;
    while (n2 < cnt) n2 <<= 1;
    for (uint32_t e = cnt + lane; e < n2; e += 64) L.buf[e] = ~0ull;
    wave_sync();
    lds_bitonic_sort(L.buf, n2, lane);
    if (P.out_idx) {
        for (uint32_t e = lane; e < k; e += 64) {
            const bool keep = e < m;
            const uint64_t v = keep ? L.buf[e] : 0ull;
            P.out_idx[(size_t)q * P.k + e] = keep ? (uint32_t)v : 0xFFFFFFFFu;
            P.out_dist[(size_t)q * P.k + e] = keep ? sqrtf(__uint_as_float((uint32_t)(v >> 32))) : __builtin_inff();
        }
    }
    if (P.out_count && lane == 0) P.out_count[q] = m;
    if (P.rgb) {
        // Raytracer.cuh:110-138 over the m kept photons
        const float alpha = 1.818f, beta = 1.953f;
        const float pi_f = 3.141592654f;
        float res0 = 0.f, res1 = 0.f, res2 = 0.f, rmax = 0.f;
        if (m > 0) {
            rmax = sqrtf(__uint_as_float((uint32_t)(L.buf[m - 1] >> 32)));
            const float filter_r = __fmul_rn(rmax, rmax);
            const float denom = 1.f - expf(-beta);
            const float nx = P.nrm[q], ny = P.nrm[P.nq + q], nz = P.nrm[2 * (size_t)P.nq + q];
            for (uint32_t e = lane; e < m; e += 64) {
                const uint64_t v = L.buf[e];
                const uint32_t idx = (uint32_t)v;
                float dx = P.dir[idx], dy = P.dir[P.n + idx], dz = P.dir[2 * (size_t)P.n + idx];
                float cosNL = __fadd_rn(__fadd_rn(__fmul_rn(nx, -dx), __fmul_rn(ny, -dy)), __fmul_rn(nz, -dz));
                if (cosNL > 0.f) {
                    float d = sqrtf(__uint_as_float((uint32_t)(v >> 32)));
                    float x = __fdiv_rn(__fmul_rn(__fmul_rn(-beta, d), d), __fmul_rn(2.f, filter_r));
                    float w = __fmul_rn(alpha, 1.f - __fdiv_rn(1.f - expf(x), denom));
                    res0 += P.power[idx] * w;
                    res1 += P.power[P.n + idx] * w;
                    res2 += P.power[2 * (size_t)P.n + idx] * w;
                }
            }
        }
        res0 = wave_sum_f32(res0);
        res1 = wave_sum_f32(res1);
        res2 = wave_sum_f32(res2);
        if (lane == 0) {
            float coef = 1.f;
            if (m > 0) coef = __fdiv_rn(1.f, __fmul_rn(__fmul_rn(pi_f, __fmul_rn(rmax, rmax)), 1.f));
            P.rgb[q] = m > 0 ? res0 * coef : 0.f;
            P.rgb[P.nq + q] = m > 0 ? res1 * coef : 0.f;
            P.rgb[2 * (size_t)P.nq + q] = m > 0 ? res2 * coef : 0.f;
        }
    }
}

template <int CAP>
__global__ __launch_bounds__(64) void k_knn_large(KnnParams P) {
    __shared__ WaveLds<CAP> L;
    const uint32_t blk = P.remap ? pmd::xcd_remap(blockIdx.x, gridDim.x) : blockIdx.x;
    if (blk >= P.nq) return;
    large_one<CAP>(P, L, threadIdx.x, P.order ? P.order[blk] : blk);
}

// The queries a k_gather_wide launch handed over (list[0, *count)), one wave
// per workgroup over a fixed grid.
template <int CAP>
__global__ __launch_bounds__(64) void k_knn_large_list(KnnParams P, const uint32_t* __restrict__ list,
                                                       const uint32_t* __restrict__ count) {
    __shared__ WaveLds<CAP> L;
    const uint32_t n = *count;
    for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {
        large_one<CAP>(P, L, threadIdx.x, list[i]);
        wave_sync();
    }
}

// Radiance for 512 < k <= 2048 without a k-key buffer (the kernel behind the
// reference frame's k = 2000 gather), set up and walked as the streaming
// gather, over a query's candidates up to four times:
//   1. when its rows hold few enough candidates that at most k are expected
//      within the radius: count them and keep the largest d2. That is all
//      when at most k are: they are all kept;
//   2. otherwise count them into 256 bins linear in d2 (even on surfaces);
//   3. collect the keys (d2, slot) of the bin holding the k-th smallest, at
//      most 64 (a fuller bin is split 256 ways by a walk first), and rank them
//      against each other: the (k - below)-th there is the k-th key K*;
//   4. sum the estimate over the photons with key <= K* (or all of them), the
//      filter radius being the largest kept distance.
// The kept set is exactly the k smallest (d2, slot) keys, as in the buffered
// kernels; the radiance sum runs in walk order. A query whose split bin still
// holds more than 64 keys is appended to `ovf_list` for k_knn_large_list.
// Bound by the VALU (85% of its issue). The reference frame's ~740k queries
// (1M photons, k = 2000, r = 0.05): 6.56 ms with a set-up and three walks a
// query, a 512-key register sort and the reference's FP32 weights, 5.12 ms
// now. Listing the slots in walk 1 for the sum to run over, instead of walking
// again, saved 9% of the instructions and lost as much to the LDS (8 KB a
// wave: 5 waves per SIMD).
constexpr uint32_t kWideList = 64;
constexpr uint32_t kWideRing = 256;
struct WideLds {
    union {
        uint32_t hist[256];
        uint64_t list[kWideList];
        uint64_t ring[kWideRing];  // kept keys waiting for their batch of 64
    };
};

// The crossing of the k-th count in L.hist (ascending bins): its bin, that
// bin's count, and the count in the bins before it.
__device__ __forceinline__ void wide_crossing(const WideLds& L, uint32_t lane, uint32_t k, uint32_t& bin,
                                              uint32_t& c, uint32_t& below) {
    // lane l holds bins 4 l .. 4 l + 3
    const uint32_t h0 = L.hist[4 * lane], h1 = L.hist[4 * lane + 1], h2 = L.hist[4 * lane + 2],
                   h3 = L.hist[4 * lane + 3];
    const uint32_t incl = wave_incl_scan(h0 + h1 + h2 + h3, lane);
    const int ls = __builtin_ctzll(wballot(incl >= k));
    const uint32_t c0 = __builtin_amdgcn_readlane(h0, ls), c1 = __builtin_amdgcn_readlane(h1, ls),
                   c2 = __builtin_amdgcn_readlane(h2, ls), c3 = __builtin_amdgcn_readlane(h3, ls);
    below = __builtin_amdgcn_readlane(incl, ls) - (c0 + c1 + c2 + c3);
    bin = 4u * (uint32_t)ls;
    c = c0;
    if (below + c < k) below += c, ++bin, c = c1;
    if (below + c < k) below += c, ++bin, c = c2;
    if (below + c < k) below += c, ++bin, c = c3;
}

constexpr float kBinTop = 0x1.fffffep+7f;  // the largest float below 256

// One query (lb: its first lane); false: handed to the overflow list.
__device__ __forceinline__ bool wide_query(ParamsPtr kp0, const WaveQueries& W, uint32_t lb, uint32_t lane,
                                           WideLds& L) {
    uint32_t found, hi, m;
    bool batch;
    uint64_t kstar = ~0ull;
    float rmax2;
    {
        ParamsPtr kp = opaque(kp0);
        const uint32_t k = (uint32_t)kp->k, hit = __float_as_uint(kp->T) + 1u;
        batch = kp->nr > 0;
        hi = __builtin_amdgcn_readlane(W.hib, lb);
        bool part = hi < hit, binned = true;
        if (batch && !part) {
            const uint32_t all = __builtin_amdgcn_readlane(W.end, lb + (uint32_t)kp->nr - 1u);
            binned = (float)all * kp->within > 0.9f * (float)k;
        }
        float dmax = 0.f, scale = 0.f;
        for (;;) {
            found = 0;
            dmax = 0.f;
            if (!binned) {
                walk_query<false>(kp0, lane, W, lb, batch, false, hi,
                           [&](uint64_t am, uint32_t sa, float d2a, uint64_t bm, uint32_t sb, float d2b) {
                               const uint64_t ba = am & wballot(__float_as_uint(d2a) < hi),
                                              bb = bm & wballot(__float_as_uint(d2b) < hi);
                               found += (uint32_t)(__popcll(ba) + __popcll(bb));
                               dmax = fmaxf(dmax, __builtin_amdgcn_inverse_ballot_w64(ba) ? d2a : 0.f);
                               dmax = fmaxf(dmax, __builtin_amdgcn_inverse_ballot_w64(bb) ? d2b : 0.f);
                           });
                if (found <= k) break;
                binned = true;
                continue;
            }
            for (uint32_t e = lane; e < 256; e += 64) L.hist[e] = 0;
            wave_sync();
            // (a NaN product, when hi is 0 or denormal, gives bin 255)
            scale = 256.f * __builtin_amdgcn_rcpf(__uint_as_float(hi));
            walk_query<false>(kp0, lane, W, lb, batch, false, hi,
                       [&](uint64_t am, uint32_t, float d2a, uint64_t bm, uint32_t, float d2b) {
                           const uint64_t ba = am & wballot(__float_as_uint(d2a) < hi),
                                          bb = bm & wballot(__float_as_uint(d2b) < hi);
                           found += (uint32_t)(__popcll(ba) + __popcll(bb));
                           if (__builtin_amdgcn_inverse_ballot_w64(ba)) {
                               atomicAdd(&L.hist[(uint32_t)fminf(d2a * scale, kBinTop)], 1u);
                               dmax = fmaxf(dmax, d2a);
                           }
                           if (__builtin_amdgcn_inverse_ballot_w64(bb)) {
                               atomicAdd(&L.hist[(uint32_t)fminf(d2b * scale, kBinTop)], 1u);
                               dmax = fmaxf(dmax, d2b);
                           }
                       });
            wave_sync();
            if (!part || found >= k) break;
            // fewer than k below the guessed bound: the whole box
            part = batch = false;
            hi = hit;
        }
        m = found < k ? found : k;
        if (found > k) {
            uint32_t bin, c, below;
            wide_crossing(L, lane, k, bin, c, below);
            wave_sync();  // the bins are read before they are written again
            uint32_t sub = 0;
            const bool split = c > kWideList;
            if (split) {
                // the bin's keys by the next eight bits (the difference is
                // exact, so the order is kept)
                for (uint32_t e = lane; e < 256; e += 64) L.hist[e] = 0;
                wave_sync();
                walk_query<false>(kp0, lane, W, lb, batch, false, hi,
                           [&](uint64_t am, uint32_t, float d2a, uint64_t bm, uint32_t, float d2b) {
                               const float fa = fminf(d2a * scale, kBinTop), fb = fminf(d2b * scale, kBinTop);
                               const uint64_t ba = am & wballot(__float_as_uint(d2a) < hi) & wballot((uint32_t)fa == bin),
                                              bb = bm & wballot(__float_as_uint(d2b) < hi) & wballot((uint32_t)fb == bin);
                               if (__builtin_amdgcn_inverse_ballot_w64(ba))
                                   atomicAdd(&L.hist[(uint32_t)((fa - (float)bin) * 256.f)], 1u);
                               if (__builtin_amdgcn_inverse_ballot_w64(bb))
                                   atomicAdd(&L.hist[(uint32_t)((fb - (float)bin) * 256.f)], 1u);
                           });
                wave_sync();
                uint32_t b2;
                wide_crossing(L, lane, k - below, sub, c, b2);
                below += b2;
                wave_sync();
                if (c > kWideList) return false;
            }
            uint32_t cnt = 0;
            walk_query<false>(kp0, lane, W, lb, batch, false, hi,
                       [&](uint64_t am, uint32_t sa, float d2a, uint64_t bm, uint32_t sb, float d2b) {
                           const float fa = fminf(d2a * scale, kBinTop), fb = fminf(d2b * scale, kBinTop);
                           uint64_t ba = am & wballot(__float_as_uint(d2a) < hi) & wballot((uint32_t)fa == bin),
                                    bb = bm & wballot(__float_as_uint(d2b) < hi) & wballot((uint32_t)fb == bin);
                           if (split) {
                               ba &= wballot((uint32_t)((fa - (float)bin) * 256.f) == sub);
                               bb &= wballot((uint32_t)((fb - (float)bin) * 256.f) == sub);
                           }
                           const uint32_t cb = __builtin_amdgcn_readfirstlane(cnt + (uint32_t)__popcll(ba));
                           if (__builtin_amdgcn_inverse_ballot_w64(ba)) L.list[cnt + mbcnt(ba)] = make_key(d2a, sa);
                           if (__builtin_amdgcn_inverse_ballot_w64(bb)) L.list[cb + mbcnt(bb)] = make_key(d2b, sb);
                           cnt = cb + (uint32_t)__popcll(bb);
                       });
            wave_sync();
            const uint64_t kk = lane < c ? L.list[lane] : ~0ull;
            uint32_t rank = 0;
            for (uint32_t j = 0; j < c; ++j) {
                const uint64_t kj = ((uint64_t)__builtin_amdgcn_readlane((uint32_t)(kk >> 32), j) << 32) |
                                    (uint32_t)__builtin_amdgcn_readlane((uint32_t)kk, j);
                rank += kj < kk ? 1u : 0u;
            }
            const int at = __builtin_ctzll(wballot(lane < c && rank == k - below - 1u));
            const uint32_t kh = __builtin_amdgcn_readlane((uint32_t)(kk >> 32), at);
            kstar = ((uint64_t)kh << 32) | (uint32_t)__builtin_amdgcn_readlane((uint32_t)kk, at);
            rmax2 = __uint_as_float(kh);
        } else {
            rmax2 = wave_max_nonneg_f32(dmax);
        }
    }
    const uint32_t q = __builtin_amdgcn_readlane(W.q, lb);
    ParamsPtr kp = opaque(kp0);
    if (kp->out_count && lane == 0) kp->out_count[q] = m;

    // Raytracer.cuh:110-138 over the kept photons, 64 at a time in walk order,
    // one lane each, with the weights of radiance_buffer. Their keys queue in
    // the wave's LDS ring; a batch's direction and power are consumed only when
    // the next batch is taken, some walk steps later, so the walk does not wait
    // on them.
    const float alpha = 1.818f, beta = 1.953f;
    const float pi_f = 3.141592654f;
    const float inv_denom = 1.16529458f, log2e = 1.44269504f;
    float res0 = 0.f, res1 = 0.f, res2 = 0.f;
    const float rmax = __builtin_amdgcn_sqrtf(rmax2);
    const float filter_r = __fmul_rn(rmax, rmax);
    const uint32_t nq = kp->nq;
    if (m > 0) {
        const float s = -beta * __builtin_amdgcn_rcpf(2.f * filter_r) * log2e;
        const float wa = alpha * (1.f - inv_denom), wb = alpha * inv_denom;
        const float* nrm = kp->nrm;
        const float nx = nrm[q], ny = nrm[nq + q], nz = nrm[2 * (size_t)nq + q];
        bool bv = false;
        float bd2 = 0.f, bx = 0.f, by = 0.f, bz = 0.f, br = 0.f, bg = 0.f, bb = 0.f;
        auto consume = [&]() {
            const float cosNL = __fadd_rn(__fadd_rn(__fmul_rn(nx, -bx), __fmul_rn(ny, -by)), __fmul_rn(nz, -bz));
            if (bv && cosNL > 0.f) {
                const float w = wa + wb * __builtin_amdgcn_exp2f(bd2 * s);
                res0 += br * w;
                res1 += bg * w;
                res2 += bb * w;
            }
        };
        auto fetch = [&](ParamsPtr kt, uint32_t off) {
            const uint32_t n = kt->n;
            const float *dir = kt->dir, *pow = kt->power;
            bx = bload(plane_rsrc(dir, n), off);
            by = bload(plane_rsrc(dir + n, n), off);
            bz = bload(plane_rsrc(dir + 2 * (size_t)n, n), off);
            br = bload(plane_rsrc(pow, n), off);
            bg = bload(plane_rsrc(pow + n, n), off);
            bb = bload(plane_rsrc(pow + 2 * (size_t)n, n), off);
        };
        uint32_t head = 0, qn = 0;  // ring: entries head ... head + qn - 1 (mod its size)
        auto take = [&](uint32_t avail) {  // lanes < avail take the first entries
            bv = lane < avail;
            if (bv) {
                const uint64_t key = L.ring[(head + lane) & (kWideRing - 1u)];
                bd2 = __uint_as_float((uint32_t)(key >> 32));
                fetch(opaque(kp0), (uint32_t)key * 4u);
            }
        };
        wave_sync();  // the list is read before the ring is written
        walk_query<false>(kp0, lane, W, lb, batch, false, hi,
                   [&](uint64_t am, uint32_t sa, float d2a, uint64_t bm, uint32_t sb, float d2b) {
                       const uint64_t ka = make_key(d2a, sa), kb = make_key(d2b, sb);
                       const uint64_t ba = am & wballot(__float_as_uint(d2a) < hi) & wballot(ka <= kstar),
                                      bbal = bm & wballot(__float_as_uint(d2b) < hi) & wballot(kb <= kstar);
                       const uint32_t at = __builtin_amdgcn_readfirstlane(head + qn),
                                      bt = __builtin_amdgcn_readfirstlane(at + (uint32_t)__popcll(ba));
                       if (__builtin_amdgcn_inverse_ballot_w64(ba))
                           L.ring[(at + mbcnt(ba)) & (kWideRing - 1u)] = ka;
                       if (__builtin_amdgcn_inverse_ballot_w64(bbal))
                           L.ring[(bt + mbcnt(bbal)) & (kWideRing - 1u)] = kb;
                       // (fewer than 64 + 128: the ring holds fewer than 64 between steps)
                       qn = bt - head + (uint32_t)__popcll(bbal);
                       while (qn >= 64) {
                           wave_sync();
                           consume();
                           take(64);
                           wave_sync();
                           head = __builtin_amdgcn_readfirstlane(head + 64u);
                           qn -= 64;
                       }
                   });
        wave_sync();
        consume();
        take(qn);
        consume();
    }
    const float tot = wave_sum3_f32(res0, res1, res2);
    if ((lane & 15) == 15 && lane < 63) {
        const float coef = __builtin_amdgcn_rcpf(__fmul_rn(pi_f, __fmul_rn(rmax, rmax)));
        const uint32_t plane = lane == 15 ? 0u : lane == 31 ? 2u : 1u;
        kp->rgb[(size_t)plane * nq + q] = m > 0 ? tot * coef : 0.f;
    }
    return true;
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6))) void k_gather_wide(
    KnnParams P, uint32_t* __restrict__ ovf_list, uint32_t* __restrict__ ovf_count) {
    __shared__ WideLds lds[kWaves];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t blk = P.remap == 2 ? xcd_chunked(blockIdx.x, P.xcd_shift)
                         : P.remap   ? pmd::xcd_remap(blockIdx.x, gridDim.x)
                                     : blockIdx.x;
    const uint32_t nq = P.nq_dev ? min(P.nq, *P.nq_dev) : P.nq;
    const uint32_t u = blk * kWaves + wave;
    if (u >= nq || u >= P.n_waves) return;  // wave-uniform; no workgroup barriers below
    ParamsPtr kp0 = (ParamsPtr)__builtin_amdgcn_kernarg_segment_ptr();
    const uint32_t nqw = wave_queries(u, P.n_waves, (uint32_t)P.gq, nq);
    WaveQueries W;
    setup_queries(kp0, lane, P.order, u, P.n_waves, 0u, nqw, W);
    for (uint32_t i = 0; i < nqw; ++i) {
        const uint32_t lb = i * (uint32_t)opaque(kp0)->nr;
        if (!wide_query(kp0, W, lb, lane, lds[wave]) && lane == 0)
            ovf_list[atomicAdd(ovf_count, 1u)] = __builtin_amdgcn_readlane(W.q, lb);
        wave_sync();
    }
}

// Batched forms: the queries of many jobs (grids, radii, k) in one launch.
// The launch's waves are numbered job by job: job j's are wbase[j] ... ,
// gq_j queries each, so a wave's queries are all of one job (positions
// qbase[j] + ... of the flattened order, which is sorted by job).
__device__ __forceinline__ uint32_t job_of(const uint32_t* __restrict__ base, uint32_t n_jobs, uint32_t g) {
    uint32_t lo = 0, hi = n_jobs;
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (base[mid] <= g)
            lo = mid;
        else
            hi = mid;
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

template <bool kLists>
__device__ __forceinline__ void batch_wave(const KnnParams* __restrict__ jobs, const uint32_t* __restrict__ qbase,
                                           const uint32_t* __restrict__ wbase, uint32_t n_jobs,
                                           const uint32_t* __restrict__ order, uint32_t u, WaveLds<512>& L) {
    const uint32_t j = job_of(wbase, n_jobs, u);
    ParamsPtr kp = (ParamsPtr)(jobs + j);
    const uint32_t n_waves = kp->n_waves;
    const uint32_t qb = __builtin_amdgcn_readfirstlane(qbase[j]);
    const uint32_t first = __builtin_amdgcn_readfirstlane(u - wbase[j]);
    stream_wave<512, kLists, false>(kp, L, threadIdx.x & 63, order, qb + first, n_waves, qb,
                             wave_queries(first, n_waves, (uint32_t)kp->gq, kp->nq));
}

// Workgroups go to the 8 XCDs round-robin; the linear workgroup id is
// remapped so that XCD x takes chunks x, x + 8, ... of 2^shift consecutive
// workgroups: each XCD's L2 still sees runs of neighbouring cells, while at
// any moment all XCDs work inside the same region of the (job, cell) order
// and share the photon blocks in the MALL (a contiguous eighth per XCD would
// put eight different jobs in flight). The 2-D grid keeps every dimension's
// work-item count below 2^32; the workgroups past the rounded-up count exit
// at once.
template <bool kLists>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(7))) void k_knn_batch_grid(
    const KnnParams* __restrict__ jobs, const uint32_t* __restrict__ qbase, const uint32_t* __restrict__ wbase,
    uint32_t n_jobs, const uint32_t* __restrict__ order, uint32_t n_waves, uint32_t n_blocks, uint32_t shift) {
    __shared__ WaveLds<512> lds[kWaves];
    const uint32_t b = blockIdx.y * gridDim.x + blockIdx.x;
    if (b >= n_blocks) return;  // n_blocks is a multiple of 8 << shift
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t u = xcd_chunked(b, shift) * kWaves + wave;
    if (u >= n_waves) return;  // wave-uniform
    batch_wave<kLists>(jobs, qbase, wbase, n_jobs, order, u, lds[wave]);
}

// Persistent form: workgroups stay resident and their waves take wave units
// from a device work counter until it passes the total.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6))) void k_knn_batch(
    const KnnParams* __restrict__ jobs, const uint32_t* __restrict__ qbase, const uint32_t* __restrict__ wbase,
    uint32_t n_jobs, const uint32_t* __restrict__ order, uint32_t n_waves, uint32_t* __restrict__ counter) {
    __shared__ WaveLds<512> lds[kWaves];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (;;) {
        uint32_t u = 0;
        if (lane == 0) u = atomicAdd(counter, 1u);
        u = __builtin_amdgcn_readfirstlane(u);
        if (u >= n_waves) break;
        batch_wave<true>(jobs, qbase, wbase, n_jobs, order, u, lds[wave]);
        wave_sync();
    }
}

// Two passes: histogram of in-radius d2 over the float-bit bins, then the
// keys below the bin edge that keeps >= k are compacted into the buffer.
__global__ __launch_bounds__(256) void k_knn_two_pass(KnnParams P) {
    constexpr int CAP = 512;
    __shared__ WaveLds<CAP> lds[kWaves];
    const uint32_t lane = threadIdx.x & 63;
    uint32_t q;
    Box B;
    float qx, qy, qz;
    if (!query_of_wave(P, q)) return;
    box_of(P, q, B, qx, qy, qz);
    WaveLds<CAP>& L = lds[threadIdx.x >> 6];
    const float T = P.T;
    const uint32_t bT = P.bT, k = (uint32_t)P.k;
    L.hist[lane] = 0;
    wave_sync();
    walk(P, lane, B, qx, qy, qz, [&](bool valid, uint32_t, float d2) {
        if (valid && d2 <= T) {
            uint32_t h = bT - (__float_as_uint(d2) >> 22);
            atomicAdd(&L.hist[h < 63u ? h : 63u], 1u);
        }
    });
    wave_sync();
    uint32_t cum = wave_incl_scan(L.hist[63 - lane], lane);
    const uint32_t found = __shfl(cum, 63, 64);
    uint64_t khi = ~0ull;
    if (found > k) {
        int ls = __builtin_ctzll(wballot(cum >= k));
        khi = (uint64_t)(bT - (63u - (uint32_t)ls) + 1u) << 54;
    }
    // collect; if the bin edge keeps more than CAP keys, tighten on the fly
    uint32_t cnt = 0;
    walk(P, lane, B, qx, qy, qz, [&](bool valid, uint32_t slot, float d2) {
        uint64_t key = make_key(d2, slot);
        bool acc = valid && d2 <= T && key < khi;
        uint64_t bal = wballot(acc);
        uint32_t na = (uint32_t)__popcll(bal);
        if (cnt + na > (uint32_t)CAP) {
            wave_sync();
            cnt = buf_select<CAP>(L, lane, cnt, k, CAP / 2, bT, khi);
            acc = acc && key < khi;
            bal = wballot(acc);
            na = (uint32_t)__popcll(bal);
        }
        if (acc) L.buf[cnt + mbcnt(bal)] = key;
        cnt += na;
    });
    wave_sync();
    // (khi <= (bits(T) + 1) << 32 once narrowed, else every key is within T)
    const uint32_t top = __float_as_uint(T) + 1u;
    const uint64_t up = khi >= (uint64_t)top << 32 ? top : (khi + 0xffffffffull) >> 32;
    finish<CAP, true>(P, L, lane, q, cnt, (uint32_t)up);
}

// Radiance from a stored kNN result (pm_radiance): one wave per query.
__global__ __launch_bounds__(256) void k_radiance(KnnParams P) {
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t q = blockIdx.x * kWaves + wave;
    if (q >= P.nq) return;
    const uint32_t m = min(P.out_count[q], (uint32_t)P.k);
    const float alpha = 1.818f, beta = 1.953f;
    const float pi_f = 3.141592654f;
    float res0 = 0.f, res1 = 0.f, res2 = 0.f;
    float rmax = m > 0 ? P.out_dist[(size_t)q * P.k + (m - 1)] : 0.f;
    if (m > 0) {
        const float filter_r = __fmul_rn(rmax, rmax);
        const float denom = 1.f - expf(-beta);
        const float nx = P.nrm[q], ny = P.nrm[P.nq + q], nz = P.nrm[2 * (size_t)P.nq + q];
        for (uint32_t e = lane; e < m; e += 64) {
            uint32_t idx = P.out_idx[(size_t)q * P.k + e];
            float dx = P.dir[idx], dy = P.dir[P.n + idx], dz = P.dir[2 * (size_t)P.n + idx];
            float cosNL = __fadd_rn(__fadd_rn(__fmul_rn(nx, -dx), __fmul_rn(ny, -dy)), __fmul_rn(nz, -dz));
            if (cosNL > 0.f) {
                float d = P.out_dist[(size_t)q * P.k + e];
                float x = __fdiv_rn(__fmul_rn(__fmul_rn(-beta, d), d), __fmul_rn(2.f, filter_r));
                float w = __fmul_rn(alpha, 1.f - __fdiv_rn(1.f - expf(x), denom));
                res0 += P.power[idx] * w;
                res1 += P.power[P.n + idx] * w;
                res2 += P.power[2 * (size_t)P.n + idx] * w;
            }
        }
    }
    res0 = wave_sum_f32(res0);
    res1 = wave_sum_f32(res1);
    res2 = wave_sum_f32(res2);
    if (lane == 0) {
        float coef = m > 0 ? __fdiv_rn(1.f, __fmul_rn(__fmul_rn(pi_f, __fmul_rn(rmax, rmax)), 1.f)) : 0.f;
        P.rgb[q] = res0 * coef;
        P.rgb[P.nq + q] = res1 * coef;
        P.rgb[2 * (size_t)P.nq + q] = res2 * coef;
    }
}

// Batch processing order keys: flattened query g of job j gets
// cell_base[j] + its cell, so one sort orders jobs, then cells within a job.
__global__ __launch_bounds__(256) void k_batch_query_keys(const KnnParams* __restrict__ jobs,
                                                         const uint32_t* __restrict__ qbase,
                                                         const uint32_t* __restrict__ cell_base, uint32_t n_jobs,
                                                         uint32_t total, uint32_t* __restrict__ keys) {
    uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= total) return;
    uint32_t lo = 0, hi = n_jobs;
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (qbase[mid] <= g)
            lo = mid;
        else
            hi = mid;
    }
    const KnnParams& P = jobs[lo];
    const uint32_t q = g - qbase[lo];
    int x = pmd::cell_coord(P.qx[q], P.G.mn[0], P.G.cell, P.G.g[0]);
    int y = pmd::cell_coord(P.qy[q], P.G.mn[1], P.G.cell, P.G.g[1]);
    int z = pmd::cell_coord(P.qz[q], P.G.mn[2], P.G.cell, P.G.g[2]);
    keys[g] = cell_base[lo] + pmd::cell_index(P.G, x, y, z);
}

// Cell key of each query for the optional cell-ordered processing.
__global__ __launch_bounds__(256) void k_query_keys(GridGeom G, const float* __restrict__ qx,
                                                   const float* __restrict__ qy, const float* __restrict__ qz,
                                                   uint32_t nq, uint32_t* __restrict__ keys,
                                                   const uint32_t* __restrict__ nq_dev) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nq || (nq_dev && i >= *nq_dev)) return;
    int x = pmd::cell_coord(qx[i], G.mn[0], G.cell, G.g[0]);
    int y = pmd::cell_coord(qy[i], G.mn[1], G.cell, G.g[1]);
    int z = pmd::cell_coord(qz[i], G.mn[2], G.cell, G.g[2]);
    keys[i] = pmd::cell_index(G, x, y, z);
}

// Sum over queries of C_q (cells in the box) and P_q (photons in them).
__global__ __launch_bounds__(256) void k_box_stats(GridGeom G, const uint32_t* __restrict__ starts,
                                                  const uint32_t* __restrict__ sizes, const float* __restrict__ qx,
                                                  const float* __restrict__ qy, const float* __restrict__ qz,
                                                  uint32_t nq, int rc, float T, int reference,
                                                  unsigned long long* __restrict__ out) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    unsigned long long cells = 0, cands = 0;
    if (i < nq) {
        const float qv[3] = {qx[i], qy[i], qz[i]};
        Box B;
        for (int a = 0; a < 3; ++a) {
            int c = pmd::cell_coord(qv[a], G.mn[a], G.cell, G.g[a]);
            B.lo[a] = max(0, c - rc);
            B.hi[a] = min(G.g[a] - 1, c + rc);
        }
        // the runs the gather walks (row_span): cells and photons visited
        const int nx = B.hi[0] - B.lo[0] + 1, ny = B.hi[1] - B.lo[1] + 1, nz = B.hi[2] - B.lo[2] + 1;
        const int nseg = G.layout == PM_LAYOUT_LINEAR ? ny * nz : nx * ny * nz;
        // (C_q stays the box's cell count in the linear layout, an upper
        // bound of the start / size words its row spans read)
        if (reference) {
            // the reference's whole box (PhotonGrid.cu:262-272)
            cells = (unsigned long long)nx * ny * nz;
            for (int z = B.lo[2]; z <= B.hi[2]; ++z)
                for (int y = B.lo[1]; y <= B.hi[1]; ++y) {
                    if (G.layout == PM_LAYOUT_LINEAR) {
                        const uint32_t c0 = pmd::cell_index(G, B.lo[0], y, z), c1 = c0 + (uint32_t)(nx - 1);
                        cands += starts[c1] + sizes[c1] - starts[c0];
                    } else {
                        for (int x = B.lo[0]; x <= B.hi[0]; ++x) cands += sizes[pmd::cell_index(G, x, y, z)];
                    }
                }
        } else {
            for (int s = 0; s < nseg; ++s) {
                uint32_t b, len;
                const bool kept = row_span(G, starts, sizes, B, s, qv[0], qv[1], qv[2], T, b, len);
                cands += len;
                if (G.layout != PM_LAYOUT_LINEAR) cells += kept;
            }
            if (G.layout == PM_LAYOUT_LINEAR) cells = (unsigned long long)nx * ny * nz;
        }
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        cells += __shfl_xor(cells, d, 64);
        cands += __shfl_xor(cands, d, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&out[0], cells);
        atomicAdd(&out[1], cands);
    }
}

__global__ void k_zero2(unsigned long long* p) {
    p[0] = 0;
    p[1] = 0;
}

pm_status setup(pm_ctx* ctx, const pm_grid* grid, const float* d_q, uint32_t nq, float radius, int32_t k,
                uint32_t flags, KnnParams& P, const char* who) {
    if (!grid) return pm::fail(ctx, PM_ERR_INVALID, "%s: null grid", who);
    if (nq > 0 && !d_q) return pm::fail(ctx, PM_ERR_INVALID, "%s: null queries", who);
    if (!(radius >= 0.f) || !std::isfinite(radius)) return pm::fail(ctx, PM_ERR_INVALID, "%s: bad radius", who);
    if (k < 1 || k > kMaxK) return pm::fail(ctx, PM_ERR_UNSUPPORTED, "%s: k=%d outside [1, %d]", who, k, kMaxK);
    const pm_grid_desc& D = grid->desc;
    // candidate positions are read through raw buffers with 32-bit byte offsets
    if (D.n_photons >= (1u << 30))
        return pm::fail(ctx, PM_ERR_UNSUPPORTED, "%s: grid of %u photons (the gather takes < 2^30)", who, D.n_photons);
    P = KnnParams{};
    for (int a = 0; a < 3; ++a) {
        P.G.mn[a] = D.aabb[a];
        P.G.g[a] = D.dims[a];
    }
    P.G.cell = D.cell_size;
    P.G.layout = D.layout;
    P.starts = D.d_cell_starts;
    P.sizes = D.d_cell_sizes;
    P.n = D.n_photons;
    P.px = D.d_photons;
    P.py = D.d_photons + P.n;
    P.pz = D.d_photons + 2 * (size_t)P.n;
    P.power = D.d_photons + 3 * (size_t)P.n;
    P.dir = D.d_photons + 6 * (size_t)P.n;
    P.qx = d_q;
    P.qy = d_q + nq;
    P.qz = d_q + 2 * (size_t)nq;
    P.nq = nq;
    P.r = radius;
    P.T = radius_threshold(radius);
    uint32_t tb;
    std::memcpy(&tb, &P.T, 4);
    P.bT = tb >> 22;
    // PhotonGrid.cu:266: radius_cells = (int)ceilf(radius / cell_size)
    float rcf = std::ceil(radius / D.cell_size);
    if (!(rcf < 4096.f)) return pm::fail(ctx, PM_ERR_UNSUPPORTED, "%s: radius/cell ratio too large", who);
    P.rc = (int)rcf;
    P.k = k;
    P.remap = (flags & PM_KNN_NO_XCD_REMAP) ? 0 : (flags & PM_KNN_XCD_CONTIGUOUS) ? 1 : 2;
    P.h = (flags & PM_KNN_INNER_BOX) ? P.rc / 2 : 0;
    P.gq = 1;
    return PM_OK;
}

// The streaming gather's queries per wave, for a launch of `total` queries:
// as many as their rows fit the wave's 64 lanes, while at least kFillWaves
// waves remain (16 a SIMD's worth: below that the chip is not full and a
// wave's queries would only run one after the other), and not so that a few waves
// are left over after two full rounds (8192 waves are resident).
//
// Estimates keep kFillUneven waves where several queries a wave give less than the
// longest wave costs: with the inner box (no guessed bound; 131k queries in 16M
// photons 376 us at 16384 waves, 318 at 49152, 351 with a set-up each), in
// sorted launches on crowded maps (thousands of candidates, several such queries
// end up in one wave: 65k queries in 3.78M photons, r = 0.047, 1107 and 705 us; in
// 1M, r = 0.05, 315 and 265), and in unsorted ones where the guess saves little
// (33k in 2M photons, r = 0.01, k = 100, 99 and 87; k = 32 in 16M, r = 0.005, 57 %
// of the time at 16384). Lists, whose second bound is close, do not lose there.
//
// Above k = 256 a query's walk dwarfs its set-up and the buffer leaves fewer waves,
// so the last round of long waves costs more than shared set-ups give: 60k queries,
// k = 500 920 -> 706 us at 65536 waves instead of 16384, k = 1000 1888 -> 1635, a
// 1024x768 frame's k = 2000 the same.
constexpr uint32_t kFillWaves = 16384, kFillUneven = 49152, kFillWavesLarge = 65536;
void split_waves(KnnParams& P, uint64_t total, bool sorted) {
    P.w = P.h > 0 ? P.h : P.rc;
    const int64_t side = 2 * (int64_t)P.w + 1, rows = side * side;
    P.nr = P.G.layout == PM_LAYOUT_LINEAR && rows <= 64 ? (int)rows : 0;
    const uint64_t fit = P.nr > 0 ? 64 / (uint64_t)P.nr : 1;
    uint64_t fill = kFillWaves;
    if (P.k > 256) {
        fill = kFillWavesLarge;
    } else if (!P.out_idx) {
        // photons expected within the radius, were they even on the box's faces
        const float e[3] = {(float)P.G.g[0] * P.G.cell, (float)P.G.g[1] * P.G.cell, (float)P.G.g[2] * P.G.cell};
        const float within = 3.14f * P.r * P.r * (float)P.n / (2.f * (e[0] * e[1] + e[1] * e[2] + e[2] * e[0]));
        if (P.h > 0 || (sorted ? fit > 2 && within > 900.f : within < 6.f * (float)P.k)) fill = kFillUneven;
    }
    uint64_t gq = std::min(fit, total / fill);
    if (P.k <= 256 && total > gq * fill && 16 * total < 17 * gq * fill) gq = gq == 2 ? 1 : gq + 1 == fit ? fit : gq;
    P.gq = (int)std::max<uint64_t>(1, gq);
    P.n_waves = pm::div_up(P.nq, (uint32_t)P.gq);
    // (a single query's wave would only wait for the second look-up of its
    // rows, 2000 queries 13 -> 18 us, but for long lists, whose second bound
    // makes up for a guess that fell short: 2482 lists of k = 400 279 -> 194
    // us, 10k estimates 304 -> 398; and the inner box is about the guess already)
    const float cr = 1.f + 0.6f * P.G.cell / std::max(P.r, 1e-30f);
    P.within = 1.f / (cr * cr);
    const bool guess = (P.gq > 1 || (P.k > 256 && P.out_idx)) && P.h == 0;
    // (lists, whose next bound is close, do without the fifth: k = 50 959 -> 937
    // us, k = 100 595 -> 540; from k = 200 on, 794 -> 799, it is worth having)
    const float spare = P.out_idx && P.k <= 128 ? 1.f : 1.2f;
    P.guess = guess ? spare * ((float)P.k + 3.f * std::sqrt((float)P.k) + 2.f) : INFINITY;
}

pm_status query_order(pm_ctx* ctx, const pm_grid* grid, const KnnParams& P, uint32_t* order_out) {
    size_t rs = pm::radix_sort_scratch_bytes(P.nq);
    void* work = nullptr;
    pm_status st = pm::scratch_reserve(ctx, pm::carve_size({(size_t)P.nq * 4, (size_t)P.nq * 4, (size_t)P.nq * 4, rs}),
                                       &work);
    if (st != PM_OK) return st;
    pm::Carve cv{static_cast<char*>(work)};
    uint32_t* keys = cv.take<uint32_t>(P.nq);
    uint32_t* skeys = cv.take<uint32_t>(P.nq);
    uint32_t* own = cv.take<uint32_t>(P.nq);
    uint32_t* order = order_out ? order_out : own;
    void* rw = cv.take<char>(rs);
    hipLaunchKernelGGL(k_query_keys, dim3(pm::div_up(P.nq, 256)), dim3(256), 0, ctx->stream, P.G, P.qx, P.qy, P.qz,
                       P.nq, keys, P.nq_dev);
    PM_CHECK_LAUNCH(ctx, "k_query_keys");
    int bits = 1;
    while (bits < 32 && (1ull << bits) < (uint64_t)grid->desc.n_cells) ++bits;
    return pm::radix_sort_pairs_auto(ctx, keys, nullptr, skeys, order, P.nq, bits, rw, P.nq_dev);
}

pm_status launch(pm_ctx* ctx, const pm_grid* grid, KnnParams& P, uint32_t flags) {
    if (P.nq == 0) return PM_OK;
    // radiance (and counts) without neighbour lists for k > 512: k_gather_wide
    // (up to four walks, no key buffer), with an overflow list behind it
    // (256 < k <= 512: one walk with the 768-key buffer)
    const bool mid = P.k > 256 && P.k <= 512 && (P.out_idx || P.rgb);
    const bool wide = P.k > 512 && !P.out_idx && P.rgb;
    const bool sort = (flags & PM_KNN_SORT_QUERIES) != 0;
    uint32_t* ovf_list = nullptr;
    uint32_t* ovf_count = nullptr;
    if (sort || wide) {
        // the order lives in the scratch block carved by query_order; the
        // overflow list follows it
        const size_t rs = sort ? pm::radix_sort_scratch_bytes(P.nq) : 0;
        const size_t a = sort ? (size_t)P.nq * 4 : 0;
        void* work = nullptr;
        pm_status st = pm::scratch_reserve(
            ctx, pm::carve_size({a, a, a, rs, wide ? (size_t)P.nq * 4 : 0, wide ? (size_t)64 : 0}), &work);
        if (st != PM_OK) return st;
        pm::Carve cv{static_cast<char*>(work)};
        cv.take<uint32_t>(a / 4);
        cv.take<uint32_t>(a / 4);
        uint32_t* order = cv.take<uint32_t>(a / 4);
        cv.take<char>(rs);
        if (wide) {
            ovf_list = cv.take<uint32_t>(P.nq);
            ovf_count = cv.take<uint32_t>(16);
        }
        if (sort) {
            if ((st = query_order(ctx, grid, P, order)) != PM_OK) return st;
            P.order = order;
        }
    }
    if (wide) {
        pm_status st = pm::fill_u32(ctx, ovf_count, 0u, 1);
        if (st != PM_OK) return st;
        P.h = 0;  // (the inner box is the k <= 256 gathers')
        split_waves(P, P.nq, sort);
        uint32_t nblk = pm::div_up(P.n_waves, kWaves);
        P.xcd_shift = xcd_shift_for(nblk, (uint32_t)P.gq);
        if (P.remap == 2) nblk = xcd_round(nblk, P.xcd_shift);
        hipLaunchKernelGGL(k_gather_wide, dim3(nblk), dim3(256), 0,
                           ctx->stream, P, ovf_list, ovf_count);
        PM_CHECK_LAUNCH(ctx, "k_gather_wide");
        const uint32_t lblocks = std::min<uint32_t>(P.nq, (uint32_t)std::max(ctx->cu_count, 1) * 8u);
        if (P.k > 1024)
            hipLaunchKernelGGL(k_knn_large_list<4096>, dim3(lblocks), dim3(64), 0, ctx->stream, P, ovf_list, ovf_count);
        else
            hipLaunchKernelGGL(k_knn_large_list<2048>, dim3(lblocks), dim3(64), 0, ctx->stream, P, ovf_list, ovf_count);
        PM_CHECK_LAUNCH(ctx, "k_knn_large_list");
        return PM_OK;
    }
    if (P.k > 1024) {
        hipLaunchKernelGGL(k_knn_large<4096>, dim3(P.nq), dim3(64), 0, ctx->stream, P);
        PM_CHECK_LAUNCH(ctx, "k_knn_large");
        return PM_OK;
    }
    if (P.k > 256 && !mid) {
        hipLaunchKernelGGL(k_knn_large<2048>, dim3(P.nq), dim3(64), 0, ctx->stream, P);
        PM_CHECK_LAUNCH(ctx, "k_knn_large");
        return PM_OK;
    }
    const bool two_pass = !mid && (flags & PM_KNN_TWO_PASS);
    if (!two_pass) split_waves(P, P.nq, sort);
    uint32_t nblk = pm::div_up(two_pass ? P.nq : P.n_waves, kWaves);
    P.xcd_shift = xcd_shift_for(nblk, (uint32_t)P.gq);
    if (P.remap == 2) nblk = xcd_round(nblk, P.xcd_shift);
    const dim3 grid_dim(nblk), block(256);
    const bool lists = P.out_idx != nullptr;
    if (two_pass)
        hipLaunchKernelGGL(k_knn_two_pass, grid_dim, block, 0, ctx->stream, P);
    else if (mid && lists)
        hipLaunchKernelGGL((k_knn_stream<768, true>), grid_dim, block, 0, ctx->stream, P);
    else if (mid)
        hipLaunchKernelGGL((k_knn_stream<768, false>), grid_dim, block, 0, ctx->stream, P);
    else if ((flags & PM_KNN_LARGE_BUFFER) && !lists)
        hipLaunchKernelGGL((k_knn_stream<1024, false>), grid_dim, block, 0, ctx->stream, P);
    else if (flags & PM_KNN_LARGE_BUFFER)
        hipLaunchKernelGGL((k_knn_stream<1024, true>), grid_dim, block, 0, ctx->stream, P);
    else if (P.gq == 1)
        hipLaunchKernelGGL((lists ? k_knn_stream<512, true, true> : k_knn_stream<512, false, true>), grid_dim, block, 0,
                           ctx->stream, P);
    else
        hipLaunchKernelGGL((lists ? k_knn_stream<512, true> : k_knn_stream<512, false>), grid_dim, block, 0,
                           ctx->stream, P);
    PM_CHECK_LAUNCH(ctx, "k_knn");
    return PM_OK;
}

}  // namespace

extern "C" pm_status pm_grid_knn(pm_ctx* ctx, const pm_grid* grid, const float* d_queries3, uint32_t nq, float radius,
                                 int32_t k, uint32_t flags, uint32_t* d_idx, float* d_dist, uint32_t* d_count) {
    if (!ctx) return PM_ERR_INVALID;
    flags = pm::tuned_flags(ctx, grid, radius, k, flags);
    KnnParams P;
    pm_status st = setup(ctx, grid, d_queries3, nq, radius, k, flags, P, "pm_grid_knn");
    if (st != PM_OK) return st;
    if (nq > 0 && (!d_idx || !d_dist || !d_count)) return pm::fail(ctx, PM_ERR_INVALID, "pm_grid_knn: null output");
    P.out_idx = d_idx;
    P.out_dist = d_dist;
    P.out_count = d_count;
    return launch(ctx, grid, P, flags);
}

extern "C" pm_status pm_grid_gather_radiance(pm_ctx* ctx, const pm_grid* grid, const float* d_queries3,
                                             const float* d_normals3, uint32_t nq, float radius, int32_t k,
                                             uint32_t flags, float* d_rgb3, uint32_t* d_count) {
    if (!ctx) return PM_ERR_INVALID;
    flags = pm::tuned_flags(ctx, grid, radius, k, flags);
    KnnParams P;
    pm_status st = setup(ctx, grid, d_queries3, nq, radius, k, flags, P, "pm_grid_gather_radiance");
    if (st != PM_OK) return st;
    if (nq > 0 && (!d_normals3 || !d_rgb3))
        return pm::fail(ctx, PM_ERR_INVALID, "pm_grid_gather_radiance: null normals/output");
    P.nrm = d_normals3;
    P.rgb = d_rgb3;
    P.out_count = d_count;
    return launch(ctx, grid, P, flags);
}

namespace pm {
pm_status gather_radiance_counted(pm_ctx* ctx, const pm_grid* grid, const float* d_queries3, const float* d_normals3,
                                  uint32_t cap, const uint32_t* d_nq, float radius, int32_t k, uint32_t flags,
                                  float* d_rgb3, uint32_t* d_count) {
    KnnParams P;
    pm_status st = setup(ctx, grid, d_queries3, cap, radius, k, flags, P, "gather (device count)");
    if (st != PM_OK) return st;
    P.nq_dev = d_nq;
    P.nrm = d_normals3;
    P.rgb = d_rgb3;
    P.out_count = d_count;
    return launch(ctx, grid, P, flags);
}
}  // namespace pm

extern "C" pm_status pm_radiance(pm_ctx* ctx, const pm_grid* grid, const uint32_t* d_idx, const float* d_dist,
                                 const uint32_t* d_count, const float* d_normals3, uint32_t nq, int32_t k,
                                 float* d_rgb3) {
    if (!ctx) return PM_ERR_INVALID;
    if (!grid) return pm::fail(ctx, PM_ERR_INVALID, "pm_radiance: null grid");
    if (k < 1) return pm::fail(ctx, PM_ERR_INVALID, "pm_radiance: k < 1");
    if (nq == 0) return PM_OK;
    if (!d_idx || !d_dist || !d_count || !d_normals3 || !d_rgb3)
        return pm::fail(ctx, PM_ERR_INVALID, "pm_radiance: null buffer");
    const pm_grid_desc& D = grid->desc;
    KnnParams P{};
    P.n = D.n_photons;
    P.power = D.d_photons + 3 * (size_t)P.n;
    P.dir = D.d_photons + 6 * (size_t)P.n;
    P.nq = nq;
    P.k = k;
    P.out_idx = const_cast<uint32_t*>(d_idx);
    P.out_dist = const_cast<float*>(d_dist);
    P.out_count = const_cast<uint32_t*>(d_count);
    P.nrm = d_normals3;
    P.rgb = d_rgb3;
    hipLaunchKernelGGL(k_radiance, dim3(pm::div_up(nq, kWaves)), dim3(256), 0, ctx->stream, P);
    PM_CHECK_LAUNCH(ctx, "k_radiance");
    return PM_OK;
}

extern "C" pm_status pm_grid_box_stats(pm_ctx* ctx, const pm_grid* grid, const float* d_queries3, uint32_t nq,
                                       float radius, uint32_t flags, uint64_t* h_sum_cells, uint64_t* h_sum_cands) {
    if (!ctx) return PM_ERR_INVALID;
    KnnParams P;
    pm_status st = setup(ctx, grid, d_queries3, nq, radius, 1, 0, P, "pm_grid_box_stats");
    if (st != PM_OK) return st;
    void* work = nullptr;
    if ((st = pm::scratch_reserve(ctx, 256, &work)) != PM_OK) return st;
    unsigned long long* acc = static_cast<unsigned long long*>(work);
    hipLaunchKernelGGL(k_zero2, dim3(1), dim3(1), 0, ctx->stream, acc);
    if (nq > 0)
        hipLaunchKernelGGL(k_box_stats, dim3(pm::div_up(nq, 256)), dim3(256), 0, ctx->stream, P.G, P.starts, P.sizes,
                           P.qx, P.qy, P.qz, nq, P.rc, P.T, (flags & PM_BOX_REFERENCE) ? 1 : 0, acc);
    PM_CHECK_LAUNCH(ctx, "k_box_stats");
    unsigned long long h[2] = {0, 0};
    PM_HIP(ctx, hipMemcpyAsync(h, acc, sizeof h, hipMemcpyDeviceToHost, ctx->stream));
    PM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (h_sum_cells) *h_sum_cells = h[0];
    if (h_sum_cands) *h_sum_cands = h[1];
    return PM_OK;
}

extern "C" pm_status pm_grid_query_order(pm_ctx* ctx, const pm_grid* grid, const float* d_queries3, uint32_t nq,
                                         uint32_t* d_order) {
    if (!ctx) return PM_ERR_INVALID;
    KnnParams P;
    pm_status st = setup(ctx, grid, d_queries3, nq, 0.f, 1, 0, P, "pm_grid_query_order");
    if (st != PM_OK) return st;
    if (nq == 0) return PM_OK;
    if (!d_order) return pm::fail(ctx, PM_ERR_INVALID, "pm_grid_query_order: null output");
    return query_order(ctx, grid, P, d_order);
}

extern "C" pm_status pm_gather_batch(pm_ctx* ctx, const pm_gather_job* jobs, uint32_t n_jobs, uint32_t flags) {
    if (!ctx) return PM_ERR_INVALID;
    if (n_jobs == 0) return PM_OK;
    if (!jobs) return pm::fail(ctx, PM_ERR_INVALID, "pm_gather_batch: null job table");
    // Jobs with k <= 256 share one launch of the batch kernel; those of larger k
    // run as their own launches of the single-map kernels, first, on the same
    // stream.
    std::vector<KnnParams> hp;
    std::vector<std::pair<const pm_grid*, KnnParams>> large;
    std::vector<uint32_t> qbase, cell_base, wbase;
    hp.reserve(n_jobs);
    uint64_t total = 0, cells = 0;
    for (uint32_t j = 0; j < n_jobs; ++j) {
        const pm_gather_job& J = jobs[j];
        // this job's flags: the call's, its own, and its tuning
        const uint32_t jf = pm::tuned_flags(ctx, J.grid, J.radius, J.k, flags | J.flags);
        KnnParams P;
        pm_status st = setup(ctx, J.grid, J.d_queries3, J.nq, J.radius, J.k, jf, P, "pm_gather_batch");
        if (st != PM_OK) return st;
        if (J.nq > 0) {
            if ((J.d_idx == nullptr) != (J.d_dist == nullptr))
                return pm::fail(ctx, PM_ERR_INVALID, "pm_gather_batch: job %u needs both d_idx and d_dist", j);
            if (J.d_rgb3 && !J.d_normals3)
                return pm::fail(ctx, PM_ERR_INVALID, "pm_gather_batch: job %u radiance without normals", j);
            if (!J.d_idx && !J.d_count && !J.d_rgb3)
                return pm::fail(ctx, PM_ERR_INVALID, "pm_gather_batch: job %u has no output", j);
        }
        P.out_idx = J.d_idx;
        P.out_dist = J.d_dist;
        P.out_count = J.d_count;
        P.nrm = J.d_rgb3 ? J.d_normals3 : nullptr;
        P.rgb = J.d_rgb3;
        P.order = nullptr;
        if (J.k > 256) {
            if (J.nq > 0) large.emplace_back(J.grid, P);
            continue;
        }
        qbase.push_back((uint32_t)total);
        cell_base.push_back((uint32_t)cells);
        hp.push_back(P);
        total += J.nq;
        cells += J.grid->desc.n_cells;
        if (total > 0xFFFFFFFFull) return pm::fail(ctx, PM_ERR_UNSUPPORTED, "pm_gather_batch: over 2^32 queries");
    }
    for (auto& L : large) {
        pm_status st = launch(ctx, L.first, L.second, flags & PM_KNN_SORT_QUERIES);
        if (st != PM_OK) return st;
    }
    if (total == 0) return PM_OK;
    n_jobs = (uint32_t)hp.size();
    uint64_t waves = 0;
    bool lists = false;
    for (KnnParams& P : hp) {
        split_waves(P, total, (flags & PM_KNN_SORT_QUERIES) != 0);
        wbase.push_back((uint32_t)waves);
        waves += P.n_waves;
        lists |= P.out_idx != nullptr;
    }
    const uint32_t n_waves = (uint32_t)waves;  // (at most total)
    const bool sorted = (flags & PM_KNN_SORT_QUERIES) && cells <= 0xFFFFFFFFull;
    const uint32_t nt = (uint32_t)total;
    const size_t rs = sorted ? pm::radix_sort_scratch_bytes(nt) : 0;
    const size_t bytes = pm::carve_size({(size_t)n_jobs * sizeof(KnnParams), (size_t)n_jobs * 4, (size_t)n_jobs * 4,
                                         (size_t)n_jobs * 4, 64, sorted ? (size_t)nt * 4 : 0, sorted ? (size_t)nt * 4 : 0,
                                         sorted ? (size_t)nt * 4 : 0, rs});
    void* work = nullptr;
    pm_status st = pm::scratch_reserve(ctx, bytes, &work);
    if (st != PM_OK) return st;
    pm::Carve cv{static_cast<char*>(work)};
    KnnParams* d_jobs = cv.take<KnnParams>(n_jobs);
    uint32_t* d_qbase = cv.take<uint32_t>(n_jobs);
    uint32_t* d_cbase = cv.take<uint32_t>(n_jobs);
    uint32_t* d_wbase = cv.take<uint32_t>(n_jobs);
    uint32_t* d_counter = cv.take<uint32_t>(16);
    // the four tables lie side by side in the carve
    std::vector<char> tables(reinterpret_cast<char*>(d_wbase + n_jobs) - reinterpret_cast<char*>(d_jobs));
    auto place = [&](void* at, const void* src, size_t len) {
        std::memcpy(tables.data() + (static_cast<char*>(at) - reinterpret_cast<char*>(d_jobs)), src, len);
    };
    place(d_jobs, hp.data(), hp.size() * sizeof(KnnParams));
    place(d_qbase, qbase.data(), qbase.size() * 4);
    place(d_cbase, cell_base.data(), cell_base.size() * 4);
    place(d_wbase, wbase.data(), wbase.size() * 4);
    if ((st = pm::put(ctx, d_jobs, tables.data(), tables.size())) != PM_OK) return st;
    const uint32_t* order = nullptr;
    if (sorted) {
        uint32_t* keys = cv.take<uint32_t>(nt);
        uint32_t* skeys = cv.take<uint32_t>(nt);
        uint32_t* ord = cv.take<uint32_t>(nt);
        void* rw = cv.take<char>(rs);
        hipLaunchKernelGGL(k_batch_query_keys, dim3(pm::div_up(nt, 256)), dim3(256), 0, ctx->stream, d_jobs, d_qbase,
                           d_cbase, n_jobs, nt, keys);
        PM_CHECK_LAUNCH(ctx, "k_batch_query_keys");
        int bits = 1;
        while (bits < 32 && (1ull << bits) < cells) ++bits;
        if ((st = pm::radix_sort_pairs_auto(ctx, keys, nullptr, skeys, ord, nt, bits, rw)) != PM_OK) return st;
        order = ord;
    }
    if (flags & PM_KNN_BATCH_QUEUE) {
        if ((st = pm::fill_u32(ctx, d_counter, 0u, 1)) != PM_OK) return st;
        const uint32_t blocks =
            std::min<uint32_t>(pm::div_up(n_waves, kWaves), (uint32_t)std::max(ctx->cu_count, 1) * 8u);
        hipLaunchKernelGGL(k_knn_batch, dim3(blocks), dim3(256), 0, ctx->stream, d_jobs, d_qbase, d_wbase, n_jobs,
                           order, n_waves, d_counter);
    } else {
        const uint32_t nblk = pm::div_up(n_waves, kWaves);
        const uint32_t shift = xcd_shift_for(nblk, std::max(1u, nt / n_waves));
        const uint32_t blocks = xcd_round(nblk, shift);
        const uint32_t gx = std::min<uint32_t>(blocks, 65536u);
        const dim3 gd(gx, pm::div_up(blocks, gx));
        if (lists)
            hipLaunchKernelGGL(k_knn_batch_grid<true>, gd, dim3(256), 0, ctx->stream, d_jobs, d_qbase, d_wbase, n_jobs,
                               order, n_waves, blocks, shift);
        else
            hipLaunchKernelGGL(k_knn_batch_grid<false>, gd, dim3(256), 0, ctx->stream, d_jobs, d_qbase, d_wbase,
                               n_jobs, order, n_waves, blocks, shift);
    }
    PM_CHECK_LAUNCH(ctx, "k_knn_batch");
    return PM_OK;
}
