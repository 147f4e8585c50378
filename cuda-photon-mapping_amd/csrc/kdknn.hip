// k nearest photons on the photon kd-tree (cpm::PhotonMap query).
//
// The reference's PhotonMap::locate_q (PhotonMap.cuh:289-371) is a debug
// search (priority queue of nodes, a 10000 sentinel, printf) used only by its
// tests; this is a standard kd search with the same answer as the grid
// gather: the k smallest (d2, photon index) among photons within r.
//
// A query searches a ball of a guessed squared radius: when that holds at
// least k photons, they are the k nearest overall (every photon outside it is
// farther than every photon inside). Otherwise the count c it found sizes the
// next ball, 1.5 (k / c) times as large (the growth of a surface density),
// searched from an empty buffer when it is below 0.7 of the full threshold,
// and the full ball comes last. The first guess is 0.16 of the threshold for
// a wave's first queries, then a running mean of 1.4 times the squared
// distances its earlier queries needed, at least 0.01 of the threshold (500k
// queries, k = 50: 813 -> 740 us; k = 200: 3.6 -> 2.8 ms), and the full ball where
// that mean is above 0.4 of it (50k queries beside the photons' reach 5.2 -> 3.75
// ms: nearly all of them walked two balls). The kept set is the k smallest keys whatever balls
// were tried. A full key buffer keeps its k smallest, and the search goes on
// below the k-th, photons and half-spaces alike.
//
// A query has a group of 32 lanes, two share a wave, and a group that is done
// takes the wave's next query. Each step a group pops the top 32 entries of
// its LIFO stack of node ids in LDS, visits one node a lane and pushes the
// children whose half-spaces meet the query ball, the near ones on top. A
// lone entry (the way down to the ball, and back) is instead visited with the
// four levels below it, each lane one node of that subtree: what is not
// reached from above it through the ball is dropped. The node's record is one
// 16-byte load, and the step has no lane branch but the stores: predicates are
// wave masks combined in SGPRs.
//
// What bounds it is VALU issue (about 65 instructions a step). With 64 lanes
// to a query, a node a step on the way down and two dependent loads a node,
// eight lanes of 64 were at work on average: 1M photons, 500k queries, k = 50
// within 330 photons' reach 2464 us, now 667; 1000 queries 31 us both ways
// (the longest query alone). 16 lanes to a query: 808 us instead of 690 (and k = 200
// 2.5 -> 4.2 ms, LDS for fewer waves).
//
// A launch of few queries (kFew) waits for its longest, and 32 lanes take longer
// over that than 64 do. There a query that has its wave to itself is walked by all
// lanes, with the idle group's memory for its stack (walk_alone): 1000 queries of
// k = 200 in 16M photons 151 -> 70 us (79 with 64 lanes to every query), of k = 100
// in 10k photons 41 -> 23 (26), 20k queries off the surfaces of 16M photons 10.5 ->
// 3.8 ms (3.6).
//
// A subtree is skipped only when the squared distance from the query to its
// splitting plane exceeds the threshold by a relative 1e-5, so no photon
// within it is ever missed.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "pm_select.hpp"

namespace {

using namespace pms;

constexpr int kWaves = 2;
constexpr uint32_t kGroup = 32;  // lanes of a query
constexpr uint32_t kGroups = 2;  // queries that a wave searches side by side
constexpr uint32_t kMaxLevels = 40;

struct KdParams {
    // per node {x, y, z, photon index | split plane << 30}; w = 0xFFFFFFFF
    // for an empty slot
    const float4* nodes;
    uint32_t cap;
    const float* qx;
    const float* qy;
    const float* qz;
    uint32_t nq;
    float T;
    float T_in;  // the first search's threshold, 0.16 T
    uint32_t bT;
    uint32_t per_wave;  // queries
    int k;
    uint32_t* out_idx;
    float* out_dist;
    uint32_t* out_count;
};

// A group's node stack. A step pops n entries (n <= 32) and pushes at most two
// children for each, so it grows the stack by at most n; n is cut to what is
// free above kMaxLevels, and to 1 at last (a depth-first walk from any state
// grows the stack by at most the tree's depth, at most kMaxLevels by the
// host's check), so the stack never overflows. 288 entries hold the usual
// walks (224: 5 % slower) and leave LDS for seven waves per SIMD (512: 740 us
// instead of 690).
constexpr uint32_t kStackCap = 288;

// The parameters in the kernel's argument segment; opaque() keeps what is read
// through it from being held in registers across the search.
typedef const __attribute__((address_space(4))) KdParams* KdPtr;
__device__ __forceinline__ KdPtr opaque(KdPtr p) {
    asm volatile("" : "+s"(p));
    return p;
}

// CAP: the key buffer, 128 keys for k <= 64, 256 for k <= 128, else 384 (k and
// a step's 32 fit).
template <int CAP>
struct KdLds {
    WaveLds<CAP> sel;
    uint32_t stk[kStackCap];
};

__device__ __forceinline__ float kd_dist2(float px, float py, float pz, float qx, float qy, float qz) {
    float dx = px - qx, dy = py - qy, dz = pz - qz;
    float xx = __fmul_rn(dx, dx), yy = __fmul_rn(dy, dy), zz = __fmul_rn(dz, dz);
    return __fadd_rn(__fadd_rn(xx, yy), zz);
}

// The squared distance of the k-th sorted key.
template <int R>
__device__ __forceinline__ float kth(const uint64_t (&v)[R], uint32_t k) {
    const uint32_t j = (k - 1u) / 64u;
    uint32_t d = (uint32_t)(v[0] >> 32);
#pragma unroll
    for (int r = 1; r < R; ++r)
        if (j == (uint32_t)r) d = (uint32_t)(v[r] >> 32);
    return __uint_as_float(__builtin_amdgcn_readlane(d, (k - 1u) % 64u));
}

// A search's cnt keys, all with d2 bits below hi, hold the k nearest: the
// sorted row of query q. Returns the squared distance that the query needed.
template <int CAP>
__device__ __forceinline__ float finish_query(KdPtr kp, WaveLds<CAP>& L, uint32_t lane, uint32_t q,
                                             uint32_t cnt, uint32_t hi) {
    const uint32_t k = (uint32_t)kp->k, m = cnt < k ? cnt : k;
    uint32_t* irow = kp->out_idx + (size_t)q * k;
    float* drow = kp->out_dist + (size_t)q * k;
    float dk;
    if constexpr (CAP > 256) {
        if (cnt > 256u) {
            hi = __float_as_uint(lin_select<CAP>(L, lane, cnt, k, hi, kp->bT)) + 1u;
            cnt = k;
            wave_sync();
        }
    }
    if (cnt <= 64) {
        uint64_t v[1];
        sort_keys<1, CAP>(L, lane, cnt, hi, v);
        write_rows<1>(v, lane, m, (int)k, irow, drow);
        dk = kth<1>(v, k);
    } else if (CAP <= 128 || cnt <= 128) {
        uint64_t v[2];
        sort_keys<2, CAP>(L, lane, cnt, hi, v);
        write_rows<2>(v, lane, m, (int)k, irow, drow);
        dk = kth<2>(v, k);
    } else {
        uint64_t v[4];
        sort_keys<4, CAP>(L, lane, cnt, hi, v);
        write_rows<4>(v, lane, m, (int)k, irow, drow);
        dk = kth<4>(v, k);
    }
    if (lane == 0) kp->out_count[q] = m;
    return m < k ? kp->T : dk;
}

// A query that the wave has no other beside: the walk of its ball by all 64
// lanes, with `stk`, the idle group's memory, for its stack (top entries). From
// half the stack on it takes subtrees of five levels off its top, each one entry
// for up to 32, while these leave the depth-first walk its kMaxLevels. All
// else as in k_kd_knn, where a group walks; cnt and T are the query's, wave-uniform.
template <int CAP>
__device__ __forceinline__ void walk_alone(KdPtr kp0, WaveLds<CAP>& B, uint32_t* stk, uint32_t lane, uint32_t lev,
                                           uint32_t via_l, uint32_t via_r, uint64_t bottom, float q0, float q1,
                                           float q2, uint32_t top, uint32_t& cnt, float& T) {
    constexpr uint32_t kAll = sizeof(KdLds<CAP>) / 4;
    const float4* __restrict__ nodes = kp0->nodes;
    const uint32_t cap = kp0->cap, k = (uint32_t)kp0->k;
    float prune = T * (1.0f + 1e-5f) + 1e-30f;
    while (top > 0) {
        if (cnt > CAP - 64u) {
            T = lin_select<CAP>(B, lane, cnt, k, __float_as_uint(T) + 1u, opaque(kp0)->bT);
            wave_sync();
            cnt = k;
            prune = T * (1.0f + 1e-5f) + 1e-30f;
        }
        uint32_t node = stk[lane < top ? top - 1u - lane : 0u];
        bool sub = top == 1;
        if (top > kAll / 2 && top + kGroup - 1u <= kAll - kMaxLevels)
            sub = __builtin_amdgcn_readfirstlane(node) < cap >> 4;
        const uint32_t n = sub ? 1u : min(min(top, 64u), (uint32_t)max((int)(kAll - kMaxLevels - top), 1));
        if (sub) node = (__builtin_amdgcn_readfirstlane(node) << lev) + (lane & 31u);
        const uint64_t has = wballot(lane < (sub ? kGroup - 1u : n)) & wballot(node < cap);
        wave_sync();  // every pop is read before the pushes reuse the slots
        top -= n;
        const float4 rec = nodes[min(node, cap - 1u)];
        const uint32_t w = __float_as_uint(rec.w);
        const float d2 = kd_dist2(rec.x, rec.y, rec.z, q0, q1, q2);
        const bool py = (w >> 30) == 1u, px = (w >> 30) == 0u;
        const float diff = (px ? q0 : py ? q1 : q2) - (px ? rec.x : py ? rec.y : rec.z);
        const uint64_t ok = has & wballot(w != 0xFFFFFFFFu), inner = ok & wballot(node < cap >> 1);
        const uint64_t out = wballot(diff * diff > prune), right = wballot(diff > 0.f);
        uint64_t go_l = inner & ~(out & right), go_r = inner & ~(out & wballot(diff < 0.f));
        uint64_t in = ok & wballot(d2 <= T);
        if (sub) {
            const float num = q0 + q1 + q2;
            const uint64_t reached =
                num == num ? wballot(((via_l & ~(uint32_t)go_l) | (via_r & ~(uint32_t)go_r)) == 0u) : 0ull;
            in &= reached;
            go_l &= reached & bottom;
            go_r &= reached & bottom;
        }
        if (__builtin_amdgcn_inverse_ballot_w64(in)) B.buf[cnt + mbcnt(in)] = make_key(d2, w & 0x3FFFFFFFu);
        cnt += (uint32_t)__popcll(in);
        const uint64_t both = go_l & go_r, any = go_l | go_r;
        const uint32_t nf = top + (uint32_t)__popcll(both);
        const uint64_t nr = (both & right) | (go_r & ~go_l);
        const uint32_t near = 2u * node + (__builtin_amdgcn_inverse_ballot_w64(nr) ? 2u : 1u);
        if (__builtin_amdgcn_inverse_ballot_w64(both)) stk[top + mbcnt(both)] = 4u * node + 3u - near;
        if (__builtin_amdgcn_inverse_ballot_w64(any)) stk[nf + mbcnt(any)] = near;
        top = nf + (uint32_t)__popcll(any);
        wave_sync();
    }
}

// The half of a wave mask that holds this lane.
__device__ __forceinline__ uint32_t half_of(uint64_t m, uint32_t lane) {
    return lane >= 32 ? (uint32_t)(m >> 32) : (uint32_t)m;
}

template <int CAP, bool kFew>
__global__ __launch_bounds__(64 * kWaves)
__attribute__((amdgpu_waves_per_eu(CAP == 128 && !kFew ? 7 : 5))) void k_kd_knn(KdParams P0) {
    __shared__ KdLds<CAP> lds[kWaves][kGroups];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t gl = lane % kGroup, grp = lane / kGroup, below = (1u << gl) - 1u;
    // this lane's node of a subtree of five levels, in heap order (the last
    // lane has none): its level, and the subtree's nodes whose left / right
    // child the path to it takes
    const uint32_t lev = 31u - (uint32_t)__builtin_clz(gl + 1u);
    uint32_t via_l = 0, via_r = 0;
    for (uint32_t i = gl; i > 0; i = (i - 1u) >> 1) {
        const uint32_t bit = 1u << ((i - 1u) >> 1);
        if (i & 1u)
            via_l |= bit;
        else
            via_r |= bit;
    }
    const uint64_t bottom = wballot(gl < kGroup - 1u && gl >= kGroup / 2u - 1u);
    KdPtr kp0 = (KdPtr)__builtin_amdgcn_kernarg_segment_ptr();
    uint32_t next = (blockIdx.x * kWaves + wave) * kp0->per_wave;
    const uint32_t end = min(kp0->nq, next + kp0->per_wave);
    if (next >= end) return;  // wave-uniform
    KdLds<CAP>* W = lds[wave];
    KdLds<CAP>& L = W[grp];
    const float4* __restrict__ nodes = kp0->nodes;
    const uint32_t cap = kp0->cap;
    const uint32_t k = (uint32_t)kp0->k;

    // the group's query and search: its ball, the acceptance threshold (the
    // ball's or the k-th kept key's) and the plane bound of that
    float first = kp0->T_in;
    uint32_t q, cnt, top;
    float q0 = 0.f, q1 = 0.f, q2 = 0.f, ball = 0.f, T = 0.f, prune = 0.f;
    auto bound = [&](float t) {
        T = t;
        prune = t * (1.0f + 1e-5f) + 1e-30f;
    };
    auto start = [&](float t) {
        ball = t;
        bound(t);
        cnt = 0;
        top = 1;
        if (gl == 0) L.stk[0] = 0;
    };
    auto take = [&](uint32_t i) {
        KdPtr kp = opaque(kp0);
        q = i;
        cnt = top = 0;  // (an idle group's buffer is not looked at again)
        if (q < end) {
            q0 = kp->qx[q];
            q1 = kp->qy[q];
            q2 = kp->qz[q];
            // (a ball of nearly the radius would mostly be walked a second time)
            start(first < 0.4f * kp->T ? first : kp->T);
        }
    };
    take(next + grp);
    next += kGroups;
    wave_sync();
    uint64_t live = wballot(q < end);  // (kFew; wave-uniform)
    while (kFew ? live != 0 : wballot(q < end) != 0) {
        if (kFew && live != ~0ull) {
            const uint32_t l0 = (uint32_t)__builtin_ctzll(live), g = l0 / kGroup;
            const auto of = [&](float v) {
                return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), l0));
            };
            const uint32_t n = __builtin_amdgcn_readlane(top, l0);
            uint32_t* stk = reinterpret_cast<uint32_t*>(&W[1u - g]);
            for (uint32_t i = lane; i < n; i += 64) stk[i] = W[g].stk[i];
            wave_sync();
            uint32_t c = __builtin_amdgcn_readlane(cnt, l0);
            float t = of(T);
            walk_alone<CAP>(kp0, W[g].sel, stk, lane, lev, via_l, via_r, bottom, of(q0), of(q1), of(q2), n, c, t);
            cnt = c;
            top = 0;
            T = t;
        } else {
            // a full buffer keeps its k smallest keys, and the search goes on below the k-th
            for (uint64_t full = wballot(cnt > CAP - kGroup); full;) {
                const uint32_t l0 = (uint32_t)__builtin_ctzll(full), g = l0 / kGroup;
                const float d = lin_select<CAP>(W[g].sel, lane, __builtin_amdgcn_readlane(cnt, l0), k,
                                                __builtin_amdgcn_readlane(__float_as_uint(T), l0) + 1u, opaque(kp0)->bT);
                wave_sync();
                if (grp == g) {
                    cnt = k;
                    bound(d);
                }
                full &= ~(0xffffffffull << l0);
            }
            const uint32_t n = min(min(top, kGroup), (uint32_t)max((int)(kStackCap - kMaxLevels - top), 1));
            const uint64_t sub = wballot(top == 1);
            const uint32_t e = top - (top == 1 ? 1u : gl + 1u);
            uint32_t node = L.stk[e < kStackCap ? e : 0u];
            if (top == 1) node = (node << lev) + gl;
            const uint64_t has = wballot(gl < (top == 1 ? kGroup - 1u : n)) & wballot(node < cap);
            wave_sync();  // every pop is read before the pushes reuse the slots
            top -= n;
            const float4 rec = nodes[min(node, cap - 1u)];
            const uint32_t w = __float_as_uint(rec.w);
            const float d2 = kd_dist2(rec.x, rec.y, rec.z, q0, q1, q2);
            const bool py = (w >> 30) == 1u, px = (w >> 30) == 0u;
            const float diff = (px ? q0 : py ? q1 : q2) - (px ? rec.x : py ? rec.y : rec.z);
            const uint64_t ok = has & wballot(w != 0xFFFFFFFFu), inner = ok & wballot(node < cap >> 1);
            // left subtree: coordinate <= median; right: >= median
            const uint64_t out = wballot(diff * diff > prune), right = wballot(diff > 0.f);
            uint64_t go_l = inner & ~(out & right), go_r = inner & ~(out & wballot(diff < 0.f));
            uint64_t in = ok & wballot(d2 <= T);
            if (sub) {
                // the nodes that the steps above them lead to; the bottom ones' children go on the stack
                // (every walk begins so: nothing is reached from a position that is not a number)
                const float num = q0 + q1 + q2;
                const uint64_t reached =
                    ~sub | (wballot(((via_l & ~half_of(go_l, lane)) | (via_r & ~half_of(go_r, lane))) == 0u) &
                            wballot(num == num));
                in &= reached;
                go_l &= reached & (bottom | ~sub);
                go_r &= reached & (bottom | ~sub);
            }
            const uint32_t hin = half_of(in, lane);
            if (__builtin_amdgcn_inverse_ballot_w64(in))
                L.sel.buf[cnt + __popc(hin & below)] = make_key(d2, w & 0x3FFFFFFFu);
            cnt += __popc(hin);
            // far children below the near ones, which are popped first: a full
            // buffer's k-th key then soon cuts off the rest
            const uint64_t both = go_l & go_r, any = go_l | go_r;
            if (any) {
                const uint32_t hb = half_of(both, lane), ha = half_of(any, lane);
                const uint32_t nf = top + __popc(hb);
                const uint64_t nr = (both & right) | (go_r & ~go_l);
                const uint32_t near = 2u * node + (__builtin_amdgcn_inverse_ballot_w64(nr) ? 2u : 1u);
                if (__builtin_amdgcn_inverse_ballot_w64(both)) L.stk[top + __popc(hb & below)] = 4u * node + 3u - near;
                if (__builtin_amdgcn_inverse_ballot_w64(any)) L.stk[nf + __popc(ha & below)] = near;
                top = nf + __popc(ha);
            }
            wave_sync();
        }
        if (wballot(top == 0) & wballot(q < end)) {
            KdPtr kp = opaque(kp0);
            const float Tr = kp->T;
            const bool mine = top == 0 && q < end;
            // the last ball holds the k nearest, or it was the full one
            const bool fin = mine && (cnt >= k || !(ball < Tr));
            uint64_t done = wballot(fin);
            if (mine && !fin) {
                float t = Tr;
                const float est = ball * fmaxf(1.5f * (float)k / (float)max(cnt, 1u), cnt > 0 ? 0.f : 8.f);
                if (est > ball && est < 0.7f * Tr) t = est;  // (ball: 0 where the radius is denormal)
                start(t);
            }
            while (done) {
                const uint32_t l0 = (uint32_t)__builtin_ctzll(done), g = l0 / kGroup;
                const float dk = finish_query<CAP>(opaque(kp0), W[g].sel, lane, __builtin_amdgcn_readlane(q, l0),
                                                   __builtin_amdgcn_readlane(cnt, l0),
                                                   __builtin_amdgcn_readlane(__float_as_uint(T), l0) + 1u);
                wave_sync();
                first = 0.7f * first + 0.3f * fminf(fmaxf(1.4f * dk, 0.01f * Tr), Tr);
                if (grp == g) take(next);
                ++next;
                done &= ~(0xffffffffull << l0);
            }
            if (kFew) live = wballot(q < end);
            wave_sync();
        }
    }
}

}  // namespace

extern "C" pm_status pm_kdtree_knn(pm_ctx* ctx, const pm_kdtree* tree, const float* d_queries3, uint32_t nq,
                                   float radius, int32_t k, uint32_t* d_idx, float* d_dist, uint32_t* d_count) {
    if (!ctx) return PM_ERR_INVALID;
    if (!tree) return pm::fail(ctx, PM_ERR_INVALID, "pm_kdtree_knn: null tree");
    if (!(radius >= 0.f) || !std::isfinite(radius)) return pm::fail(ctx, PM_ERR_INVALID, "pm_kdtree_knn: bad radius");
    if (k < 1 || k > 256) return pm::fail(ctx, PM_ERR_UNSUPPORTED, "pm_kdtree_knn: k=%d outside [1, 256]", k);
    if (tree->levels > kMaxLevels) return pm::fail(ctx, PM_ERR_UNSUPPORTED, "pm_kdtree_knn: tree too deep");
    if (nq == 0) return PM_OK;
    if (!d_queries3 || !d_idx || !d_dist || !d_count) return pm::fail(ctx, PM_ERR_INVALID, "pm_kdtree_knn: null buffer");
    KdParams P{};
    P.nodes = tree->nodes;
    P.cap = tree->cap;
    P.qx = d_queries3;
    P.qy = d_queries3 + nq;
    P.qz = d_queries3 + 2 * (size_t)nq;
    P.nq = nq;
    P.T = radius_threshold(radius);
    P.T_in = P.T * 0.16f;
    uint32_t tb;
    std::memcpy(&tb, &P.T, 4);
    P.bT = tb >> 22;
    P.k = k;
    P.out_idx = d_idx;
    P.out_dist = d_dist;
    P.out_count = d_count;
    // Queries a wave: one for each group while the launch has fewer than
    // 12288 waves that way, and up to eight where it has more (the ball learned
    // from the wave's own queries: 500k queries 962 -> 690 us; 100k: 230 us at
    // one, 203 at four, 230 at eight, which leaves 6k waves).
    // Few queries: while a wave takes fewer than eight, each with a wave of its own
    // up to 6144. The buffer then leaves room for 64 keys a step; where that doubles
    // it, the bound is half (90k queries of k = 64 in 300k photons 312 us with it, 265
    // with groups alone). 10k to 4M photons, groups alone against it: 20k queries of
    // k = 200 13 % slower, of k = 64 10 %, 90k of k = 100 9 %; a search of k < 8 is a
    // few steps long, and from 3072 queries on their number counts (6000 of k = 1:
    // 17.2 us, with it 18.6).
    const uint32_t most = (k > 32 && k <= 64 ? 4u : 8u) * 12288u;
    const bool few = nq < most && (k >= 8 || nq <= 3072u);
    P.per_wave = few && nq <= 6144u ? 1u : kGroups * std::min(8u, std::max(1u, nq / (kGroups * 12288u)));
    const auto kernel = few ? (k <= 32 ? k_kd_knn<128, true> : k <= 128 ? k_kd_knn<256, true> : k_kd_knn<384, true>)
                            : (k <= 64 ? k_kd_knn<128, false> : k <= 128 ? k_kd_knn<256, false> : k_kd_knn<384, false>);
    hipLaunchKernelGGL(kernel, dim3(pm::div_up(nq, kWaves * P.per_wave)), dim3(64 * kWaves), 0, ctx->stream, P);
    PM_CHECK_LAUNCH(ctx, "k_kd_knn");
    return PM_OK;
}
