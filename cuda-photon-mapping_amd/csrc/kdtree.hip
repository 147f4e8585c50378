// Photon kd-tree build (cpm::PhotonMap, PhotonMap.cuh:189-283) and the
// per-model AABB of create_kd_tree (KdTree.cu:395-464).
//
// Photon kd-tree, level by level instead of the reference's sequential LIFO
// of quicksorts:
//   * three presorted orders, one per axis, each a stable radix sort of the
//     coordinate (so ties are ordered by photon index, the total order the
//     tree is defined on); a photon's rank on an axis is its position in
//     that sort, and its record in an axis's order holds its ranks on the two
//     other axes (8 bytes): comparing ranks compares (coordinate, index), and
//     in the split axis's own order the side is the position;
//   * at every level each node's segment [from, to) has its median at
//     mid = from + (to - from)/2 in the order of the node's split axis;
//     the other two orders are stable-partitioned around that median in one
//     pass (counts with decoupled look-back), so every order stays
//     sorted inside every child segment; subtrees of at most 1024 photons
//     are finished in LDS by one workgroup each;
//   * a child's split plane is the argmax extent of its points, read from
//     the first and last record of its segment in each axis order.
// The implicit heap (children 2i+1, 2i+2) is stored with 2^L - 1 slots so no
// node is dropped (the reference's Tree drops indices >= n, Tree.cuh:10-13).
#include <cfloat>
#include <cmath>

#include "pm_internal.hpp"

namespace {

// A photon's record in the order of axis a: its ranks on the two other axes,
// other_axis(a, 0) < other_axis(a, 1).
struct Rk {
    uint32_t r[2];
};

__host__ __device__ __forceinline__ int other_axis(int a, int i) {
    return i == 0 ? (a == 0 ? 1 : 0) : (a == 2 ? 1 : 2);
}

// The level phase's arrays: the three orders (A[a][j]: the record at
// position j of axis a's order), each axis's sorted photon indices
// (order[a n + r]: the photon of rank r) and ranks (rank4[4 id + a]), and
// the input planes (coordinates by photon index).
struct Orders {
    const Rk* A[3];
    const uint32_t* order;
    const uint32_t* rank4;
    const float* ph9;
    uint32_t n;
};

// the photon at position j of axis a's order
__device__ __forceinline__ uint32_t id_at(const Orders& O, int a, uint32_t j) {
    return O.order[(size_t)other_axis(a, 0) * O.n + O.A[a][j].r[0]];
}

constexpr uint32_t kFinal = 0xFFFFFFFFu;
constexpr uint32_t kTicket = 32;  // words between the axes' tile counters (a line each)

__device__ __forceinline__ uint32_t orderable(float f) {
    f = f + 0.0f;  // -0 -> +0 so that equal coordinates tie on the index
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__global__ __launch_bounds__(256) void k_axis_keys(const float* __restrict__ p, uint32_t n, uint32_t* __restrict__ keys) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) keys[i] = orderable(p[i]);
}

// Each photon as one 48-byte record (three float4: pos + power.r, power.gb +
// dir.xy, dir.z): the gathers by sort order and by node read one record
// instead of up to nine scattered 4-byte values.
__global__ __launch_bounds__(256) void k_photon_records(const float* __restrict__ in9, uint32_t n,
                                                       float4* __restrict__ rec) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float v[9];
#pragma unroll
    for (int p = 0; p < 9; ++p) v[p] = in9[(size_t)p * n + i];
    rec[3 * (size_t)i + 0] = make_float4(v[0], v[1], v[2], v[3]);
    rec[3 * (size_t)i + 1] = make_float4(v[4], v[5], v[6], v[7]);
    rec[3 * (size_t)i + 2] = make_float4(v[8], 0.f, 0.f, 0.f);
}

// rank4[order[a n + r]].a = r (blockIdx.y = axis a): each photon's three
// ranks in one 16-byte entry, so a record is one gather
__global__ __launch_bounds__(256) void k_ranks(const uint32_t* __restrict__ order, uint32_t n,
                                              uint32_t* __restrict__ rank4) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x, a = blockIdx.y;
    if (r >= n) return;
    rank4[4 * (size_t)order[(size_t)a * n + r] + a] = r;
}

// the records of axis a's order (blockIdx.y = a): ranks on the other axes
__global__ __launch_bounds__(256) void k_rank_recs(const uint32_t* __restrict__ order,
                                                  const uint4* __restrict__ rank4, uint32_t n,
                                                  Rk* __restrict__ out0, Rk* __restrict__ out1,
                                                  Rk* __restrict__ out2) {
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x, a = blockIdx.y;
    if (j >= n) return;
    const uint4 rk = rank4[order[(size_t)a * n + j]];
    Rk r;
    r.r[0] = a == 0 ? rk.y : rk.x;
    r.r[1] = a == 2 ? rk.y : rk.z;
    (a == 0 ? out0 : a == 1 ? out1 : out2)[j] = r;
}

// PhotonMap::find_largest_plane (PhotonMap.cuh:161-178) from the extreme
// photons of a non-empty segment in each axis order.
__device__ __forceinline__ int8_t plane_of(const Orders& O, uint32_t f, uint32_t t) {
    float d[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float* c = O.ph9 + (size_t)a * O.n;
        d[a] = fabsf(c[id_at(O, a, t - 1)] - c[id_at(O, a, f)]);
    }
    int8_t p = 0;
    float mx = d[0];
    if (d[1] > mx) {
        mx = d[1];
        p = 1;
    }
    if (d[2] > mx) p = 2;
    return p;
}

// Per node of a level: its split plane (the argmax extent of its segment,
// PhotonMap.cuh:252-273: an empty node keeps +-FLT_MAX corners -> plane 0)
// and, when `medians`, its median, the median's key and the children's
// segments (med = {the median's rank on the plane, the plane}). root_n > 0:
// the level is the root's, whose segment is [0, root_n). lookback_counter
// (nullable): the level partition before this launch has completed, so its
// look-back epoch is advanced here; the axes' tile counters start at 0 again.
__global__ __launch_bounds__(256) void k_level_nodes(Orders O, uint32_t first, uint32_t count,
                                                    uint32_t cap, uint32_t root_n, bool medians, uint2* __restrict__ seg,
                                                    int8_t* __restrict__ plane, uint32_t* __restrict__ node_idx,
                                                    int8_t* __restrict__ node_plane, uint2* __restrict__ med,
                                                    uint32_t* __restrict__ lookback_counter,
                                                    uint32_t* __restrict__ tickets) {
    uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < 3) tickets[t * kTicket] = 0;
    if (t == 0 && lookback_counter) pm::lookback_advance(lookback_counter, pm::lookback_epoch(lookback_counter));
    if (t >= count) return;
    uint32_t node = first + t;
    if (root_n > 0) seg[node] = make_uint2(0, root_n);
    const uint2 s = root_n > 0 ? make_uint2(0, root_n) : seg[node];
    const int8_t p = s.y > s.x ? plane_of(O, s.x, s.y) : (int8_t)0;
    plane[node] = p;
    if (!medians) return;
    uint32_t l = 2 * node + 1, r = 2 * node + 2;
    if (s.y <= s.x) {  // empty
        if (l < cap) seg[l] = make_uint2(0, 0);
        if (r < cap) seg[r] = make_uint2(0, 0);
        return;
    }
    uint32_t mid = s.x + (s.y - s.x) / 2;
    const uint32_t id = id_at(O, p, mid);
    node_idx[node] = id;
    node_plane[node] = p;
    med[node] = make_uint2(O.rank4[4 * (size_t)id + p], (uint32_t)p);
    if (s.y - s.x == 1) {
        if (l < cap) seg[l] = make_uint2(0, 0);
        if (r < cap) seg[r] = make_uint2(0, 0);
    } else {
        if (l < cap) seg[l] = make_uint2(s.x, mid);
        if (r < cap) seg[r] = make_uint2(mid + 1, s.y);
    }
}

// ---- one level's stable partition in one pass --------------------------------
// The three axis orders are three streams of n positions. A record
// goes left, is its node's median or goes right; with the left records (lb) and
// the median (mb) counted from its node's `from` up to it, its destination is
//   left: from + lb,   median: mid,   right: mid + 1 + (j - from - lb - mb).
// Both counts are differences of plain counts over a stream, whose values at
// every node's start and end are known without counting: the nodes of a level
// hold v or v + 1 records, adjacent ones are one finished median apart, and a
// node of size s has s / 2 left records. So a row of 64 positions takes two
// ballots, and a tile that holds any node's first or last position knows its
// place in the stream; only a tile inside one node (the upper levels) takes
// it from the tiles before it by decoupled look-back (epoch-tagged tile words,
// as in the u32 scan; kLook), and the lower levels' tiles wait for nothing.
// The axes' tiles are apart, each axis with its own ordered tile ids (a tile
// waits for lower ids of its axis only, which have all started): one counter
// hands out an id in about 22 ns, 16 us a level.
// 2M photons, a level: 52 us with a segmented scan of flag words over each row
// (171 VALU instructions for 64 positions, and one tile counter), now 39.6 where
// tiles wait and 31.6 where they do not (25 is the copying at 5.1 TB/s).
constexpr int kPThreads = 1024;
constexpr int kPItems = 8;                        // rows of kPThreads positions per tile
constexpr uint32_t kPTile = kPThreads * kPItems;  // 8192
constexpr int kPRows = kPItems * (kPThreads / 64);  // wave rows, two a lane of the wave that scans them
static_assert(kPRows == 128, "the wave rows of a tile are scanned by one wave, two a lane");
// counts up to a position inside a tile: left records in bits 0-14, medians
// from bit 15; and its record's side
constexpr uint32_t kCntM = 1u << 15, kCnt = (1u << 30) - 1, kIsL = 1u << 30, kIsM = 1u << 31;
// counts up to a tile: left records mod 2^30, the parity of the medians
constexpr uint32_t kAbsL = (1u << 30) - 1, kAbsM = 1u << 30;
constexpr uint64_t kStAgg = 1, kStIncl = 2;

// A level's nodes: from `first` on, each of v or v + 1 records.
struct Level {
    uint32_t first, v;
};

__device__ __forceinline__ uint32_t abs_add(uint32_t x, uint32_t y) {
    return ((x + y) & kAbsL) | ((x ^ y) & kAbsM);
}
// a count inside a tile as one up to a tile
__device__ __forceinline__ uint32_t abs_of(uint32_t cnt) {
    return (cnt & (kCntM - 1u)) | ((cnt & kCntM) ? kAbsM : 0u);
}
// the counts at the start of the level's node i, `from` its first position: c of
// the nodes before it hold v + 1 records
__device__ __forceinline__ uint32_t abs_at(const Level& V, uint32_t i, uint32_t from) {
    const uint32_t c = from - i * (V.v + 1u);
    const uint32_t l = i * (V.v >> 1) + ((V.v & 1u) ? c : 0u);
    return (l & kAbsL) | ((i & 1u) ? kAbsM : 0u);
}
__device__ __forceinline__ uint32_t abs_sub(uint32_t x, uint32_t y) {
    return ((x - y) & kAbsL) | ((x ^ y) & kAbsM);
}

__device__ __forceinline__ uint64_t seg_state(uint32_t epoch, uint64_t status, uint32_t value) {
    return ((uint64_t)epoch << 34) | (status << 32) | value;
}

template <bool kLook>
__global__ __launch_bounds__(kPThreads) __attribute__((amdgpu_waves_per_eu(8))) void k_level_partition(
    const Rk* __restrict__ A0, const Rk* __restrict__ A1, const Rk* __restrict__ A2, Rk* __restrict__ B0,
    Rk* __restrict__ B1, Rk* __restrict__ B2, uint32_t n, const uint32_t* __restrict__ node_in,
    uint32_t* __restrict__ node_out, const uint2* __restrict__ seg, const uint2* __restrict__ med, Level V,
    uint64_t* __restrict__ state, const uint32_t* __restrict__ counter, uint32_t* __restrict__ tickets) {
    __shared__ uint32_t s_tile, s_epoch, s_known, s_at;
    __shared__ uint32_t s_row[kPRows];
    const uint32_t t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const uint32_t a = blockIdx.x % 3u, n_tiles = gridDim.x / 3u;  // the axis, and its tiles
    if (t == 0) {
        s_known = 0;
        s_tile = blockIdx.x / 3u;
        if (kLook) {
            // the epoch is advanced, and the tickets taken back, by
            // k_level_nodes, the next launch: a tile here may finish its
            // look-back before earlier tiles have read it
            s_epoch = pm::lookback_epoch(counter);
            s_tile = atomicAdd(&tickets[a * kTicket], 1u);
        }
    }
    __syncthreads();
    const uint32_t tile = s_tile, j0 = tile * kPTile + t;  // n <= 2^30
    const Rk* __restrict__ A = a == 0 ? A0 : a == 1 ? A1 : A2;
    Rk* __restrict__ B = a == 0 ? B0 : a == 1 ? B1 : B2;
    const uint32_t lo = (uint32_t)other_axis((int)a, 0);

    // position of item k: tile row k, wave, lane (rows of kPThreads consecutive
    // positions). All loads of the tile's items are issued before any item
    // is counted: positions, then their nodes' segments, planes and medians.
    uint32_t node[kPItems], cnt[kPItems];
    Rk rec[kPItems];
#pragma unroll
    for (int k = 0; k < kPItems; ++k) {
        const uint32_t j = j0 + (uint32_t)k * kPThreads;
        node[k] = kFinal;
        if (j < n) {
            node[k] = node_in[j];
            rec[k] = A[j];
        }
    }
    // (this thread's latest position that is a node's first or last, and the
    // counts before it)
    int mark = -1;
    uint32_t mark_abs = 0;
#pragma unroll
    for (int k = 0; k < kPItems; ++k) {
        const uint32_t j = j0 + (uint32_t)k * kPThreads;
        bool is_l = false, is_m = false;
        if (node[k] != kFinal) {
            const uint2 sg = seg[node[k]], md = med[node[k]];
            const uint32_t half = (sg.y - sg.x) / 2;
            // the split axis's own order: the position decides; another
            // order: the record's rank on the split axis against the median's
            const bool own = md.y == a;
            const uint32_t x = own ? j : rec[k].r[md.y == lo ? 0 : 1];
            const uint32_t m = own ? sg.x + half : md.x;
            is_l = x < m;
            is_m = x == m;
            if (j == sg.x || j + 1u == sg.y) {
                mark = k;
                mark_abs = abs_at(V, node[k] - V.first, sg.x);
                if (j != sg.x)  // (after the last position: all the node's, less its own side)
                    mark_abs = abs_add(mark_abs, (half - (is_l ? 1u : 0u)) | (is_m ? 0u : kAbsM));
            }
        }
        const uint64_t bl = __ballot(is_l), bm = __ballot(is_m);
        cnt[k] = __builtin_amdgcn_mbcnt_hi((uint32_t)(bl >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bl, 0u)) +
                 kCntM * __builtin_amdgcn_mbcnt_hi((uint32_t)(bm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bm, 0u)) +
                 (is_l ? kIsL : 0u) + (is_m ? kIsM : 0u);
        if (lane == 0) s_row[k * (kPThreads / 64) + wave] = (uint32_t)__popcll(bl) + kCntM * (uint32_t)__popcll(bm);
    }
    __syncthreads();
    // exclusive counts of the wave rows, in tile order (row-major)
    uint32_t agg = 0;
    if (wave == 0) {
        const uint32_t a = s_row[2 * lane], b = s_row[2 * lane + 1];
        uint32_t x = a + b;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(x, d, 64);
            if (lane >= (uint32_t)d) x += y;
        }
        s_row[2 * lane] = x - a - b;
        s_row[2 * lane + 1] = x - b;
        agg = abs_of(__builtin_amdgcn_readlane(x, 63));
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPItems; ++k) {
        cnt[k] += s_row[k * (kPThreads / 64) + wave];
        if (mark == k) {  // (every mark of the tile gives the same counts)
            s_at = abs_sub(mark_abs, abs_of(cnt[k] & kCnt));
            s_known = 1u;
        }
    }
    __syncthreads();
    if (kLook) {
        if (wave == 0) {
            uint32_t at = s_at;
            const uint32_t epoch = s_epoch;
            if (!s_known) {
                // inside one node: the counts of the tiles before, back to one that knows its own
                if (lane == 0)
                    __hip_atomic_store(&state[a * n_tiles + tile], seg_state(epoch, kStAgg, agg), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                at = 0;
                for (int64_t jt = (int64_t)tile - 1;; jt -= 64) {
                    const int64_t idx = jt - (int64_t)lane;
                    uint64_t w, stop_mask, upto;
                    for (;;) {
                        uint32_t status = (uint32_t)kStIncl;
                        w = 0;
                        if (idx >= 0) {
                            w = __hip_atomic_load(&state[a * n_tiles + (uint32_t)idx], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            status = ((uint32_t)(w >> 34) == epoch) ? (uint32_t)((w >> 32) & 3) : 0u;
                        }
                        stop_mask = __ballot(status == kStIncl);
                        const uint64_t inval_mask = __ballot(status == 0);
                        const int first = stop_mask ? __builtin_ctzll(stop_mask) : 63;
                        upto = (first == 63) ? ~0ull : ((2ull << first) - 1);
                        if ((inval_mask & upto) == 0) break;
                        __builtin_amdgcn_s_sleep(1);
                    }
                    uint32_t win = ((upto >> lane) & 1ull) ? (uint32_t)w : 0u;
#pragma unroll
                    for (int d = 32; d >= 1; d >>= 1) win = abs_add(win, (uint32_t)__shfl_xor(win, d, 64));
                    at = abs_add(at, win);
                    if (stop_mask & upto) break;
                }
            }
            if (lane == 0) {
                __hip_atomic_store(&state[a * n_tiles + tile], seg_state(epoch, kStIncl, abs_add(at, agg)), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
                s_at = at;
            }
        }
        __syncthreads();
    }
    const uint32_t at = s_at;
#pragma unroll
    for (int k = 0; k < kPItems; ++k) {
        const uint32_t j = j0 + (uint32_t)k * kPThreads;
        if (j >= n) continue;
        const uint32_t s = node[k];
        uint32_t dst = j, nn = kFinal;
        if (s != kFinal) {
            const uint2 sg = seg[s];
            const uint32_t mid = sg.x + (sg.y - sg.x) / 2;
            const uint32_t b = abs_sub(abs_add(at, abs_of(cnt[k] & kCnt)), abs_at(V, s - V.first, sg.x));
            const uint32_t lb = b & kAbsL, mb = b >> 30;
            if (cnt[k] & kIsL)
                dst = sg.x + lb;
            else if (cnt[k] & kIsM)
                dst = mid;
            else
                dst = mid + 1 + ((j - sg.x) - lb - mb);
            if (!(sg.y - sg.x <= 1 || j == mid)) nn = j < mid ? 2 * s + 1 : 2 * s + 2;
        }
        if (dst < n) B[dst] = rec[k];  // always true for a consistent tree
        if (a == 0) node_out[j] = nn;
    }
}

// ---- bottom levels in LDS ---------------------------------------------------
// Once every segment holds at most kLocal records, one workgroup finishes a
// whole subtree in LDS: the same median / stable-partition / child-plane
// steps as the level loop above, on the subtree's slice of the three axis
// orders. The orders are permutations of 16-bit local indices (positions in
// the axis-0 order); a thread keeps its four positions' nodes and segments in
// registers (they depend on the positions alone). A depth takes four
// barriers: each record's side is marked from its node's split axis, all three
// orders count their left records and medians by ballots from the known node
// starts (as above), move, and each new segment's first position works out its
// plane. 31 KB of LDS, five workgroups a CU. The time goes into the barriers and
// the dependent LDS reads between them: 2M photons 338 us, and 79 for a kernel that
// prepared the axis-0 positions, with one axis after the other (fifteen barriers,
// a scan of 0/1 flags and 46 KB of LDS), now 171.
constexpr int kLocal = 1024;
constexpr int kLocalThreads = 256;
constexpr int kLocalPer = kLocal / kLocalThreads;
constexpr int kLocalRows = kLocal / 64;  // wave rows of an axis
static_assert(kLocalRows == 16, "an axis's wave rows are one DPP row");

struct LocalLds {
    float c[kLocal][3];  // by local index
    uint32_t id[kLocal];
    union {
        uint16_t ord[2][3][kLocal];  // per axis: the local index at each position, this depth's and the next's
        struct {
            uint16_t first[3][kLocal];
            uint32_t r0[kLocal];  // the axis-0 ranks, ascending (while the orders are set up)
        };
    };
    uint8_t side[kLocal];   // by local index: 1 left, 2 median, 0 right
    uint8_t plane[kLocal];  // by a segment's first position
    uint32_t row[3 * kLocalRows];
};
static_assert(sizeof(uint16_t) * 3 * kLocal >= sizeof(uint32_t) * kLocal, "the ranks fit the next depth's orders");

// find_largest_plane over local segment [f, t) (PhotonMap.cuh:161-178)
__device__ __forceinline__ uint8_t local_plane(const LocalLds& L, const uint16_t (&o)[3][kLocal], uint32_t f,
                                               uint32_t t) {
    const float d0 = fabsf(L.c[o[0][t - 1]][0] - L.c[o[0][f]][0]);
    const float d1 = fabsf(L.c[o[1][t - 1]][1] - L.c[o[1][f]][1]);
    const float d2 = fabsf(L.c[o[2][t - 1]][2] - L.c[o[2][f]][2]);
    uint8_t p = 0;
    float mx = d0;
    if (d1 > mx) {
        mx = d1;
        p = 1;
    }
    if (d2 > mx) p = 2;
    return p;
}

// Inclusive sum over each row of 16 lanes.
template <int kCtrl>
__device__ __forceinline__ uint32_t dpp_row_add(uint32_t v) {
    return v + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kCtrl, 0xf, 0xf, false);
}
__device__ __forceinline__ uint32_t row_incl_scan(uint32_t v) {
    v = dpp_row_add<0x111>(v);  // row_shr:1
    v = dpp_row_add<0x112>(v);
    v = dpp_row_add<0x114>(v);
    return dpp_row_add<0x118>(v);
}

__global__ __launch_bounds__(kLocalThreads) void k_local_subtrees(Orders O, const float4* __restrict__ prec,
                                                                 uint32_t first, const uint2* __restrict__ gseg,
                                                                 const int8_t* __restrict__ gplane,
                                                                 uint32_t* __restrict__ node_idx,
                                                                 int8_t* __restrict__ node_plane) {
    __shared__ LocalLds L;
    const uint32_t root = first + blockIdx.x, t = threadIdx.x, lane = t & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint2 rs = gseg[root];
    if (rs.y <= rs.x || rs.y - rs.x > (uint32_t)kLocal) return;  // empty subtree; larger ones never reach here
    const uint32_t m = rs.y - rs.x;
    // the segment holds the same photons in each order: the photons of the
    // axis-0 order with their coordinates and axis-0 ranks
    uint32_t id[kLocalPer], a1[kLocalPer], a2[kLocalPer];
#pragma unroll
    for (int k = 0; k < kLocalPer; ++k) {
        const uint32_t j = (uint32_t)k * kLocalThreads + t;
        if (j < m) {
            id[k] = id_at(O, 0, rs.x + j);
            a1[k] = O.A[1][rs.x + j].r[0];
            a2[k] = O.A[2][rs.x + j].r[0];
        }
    }
#pragma unroll
    for (int k = 0; k < kLocalPer; ++k) {
        const uint32_t j = (uint32_t)k * kLocalThreads + t;
        L.r0[j] = 0xFFFFFFFFu;
        if (j < m) {
            const float4 c = prec[3 * (size_t)id[k]];
            L.r0[j] = O.rank4[4 * (size_t)id[k]];
            L.id[j] = id[k];
            L.c[j][0] = c.x;
            L.c[j][1] = c.y;
            L.c[j][2] = c.z;
        }
    }
    __syncthreads();
    // axes 1 and 2 mapped to axis-0 positions by their records' axis-0 ranks
#pragma unroll
    for (int k = 0; k < kLocalPer; ++k) {
        const uint32_t j = (uint32_t)k * kLocalThreads + t;
        if (j < m) {
            uint32_t x = 0, y = 0;
#pragma unroll
            for (uint32_t d = kLocal / 2; d > 0; d >>= 1) {
                if (L.r0[x + d] <= a1[k]) x += d;
                if (L.r0[y + d] <= a2[k]) y += d;
            }
            L.first[0][j] = (uint16_t)j;
            L.first[1][j] = (uint16_t)x;
            L.first[2][j] = (uint16_t)y;
        }
    }
    if (t == 0) L.plane[0] = (uint8_t)gplane[root];
    __syncthreads();

    // a position's node at this depth and its segment (from | to << 16); to = 0: finished
    uint32_t node[kLocalPer], sg[kLocalPer];
#pragma unroll
    for (int k = 0; k < kLocalPer; ++k) {
        node[k] = 0;
        sg[k] = (uint32_t)k * kLocalThreads + t < m ? m << 16 : 0u;
    }
    uint32_t smin = m, smax = m;  // the node sizes of the depth
    for (uint32_t d = 0;; ++d) {
        const uint16_t(&ord)[3][kLocal] = L.ord[d & 1u];
        uint16_t(&out)[3][kLocal] = L.ord[(d & 1u) ^ 1u];
        const uint32_t gfirst = ((root + 1u) << d) - 1u;  // global index of local node 0 at this depth
#pragma unroll
        for (int k = 0; k < kLocalPer; ++k) {
            const uint32_t j = (uint32_t)k * kLocalThreads + t, from = sg[k] & 0xffffu, to = sg[k] >> 16;
            if (to == 0) continue;
            const uint32_t mid = (from + to) >> 1;
            const uint8_t p = L.plane[from];
            const uint32_t x = ord[p][j];
            L.side[x] = j < mid ? 1 : j == mid ? 2 : 0;
            if (j == mid) {
                node_idx[gfirst + node[k]] = L.id[x];
                node_plane[gfirst + node[k]] = (int8_t)p;
            }
        }
        if (smax <= 1) break;
        __syncthreads();
        // per position and axis: local index, side, counts in its wave row
        uint32_t e[3][kLocalPer];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
#pragma unroll
            for (int k = 0; k < kLocalPer; ++k) {
                const bool on = sg[k] != 0;
                const uint32_t x = on ? ord[a][(uint32_t)k * kLocalThreads + t] : 0u;
                const uint32_t s = on ? L.side[x] : 0u;
                const uint64_t bl = __ballot(s == 1), bm = __ballot(s == 2);
                e[a][k] = x | s << 10 |
                          __builtin_amdgcn_mbcnt_hi((uint32_t)(bl >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bl, 0u)) << 12 |
                          __builtin_amdgcn_mbcnt_hi((uint32_t)(bm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bm, 0u)) << 20;
                if (lane == 0)
                    L.row[a * kLocalRows + k * (kLocalThreads / 64) + wave] =
                        (uint32_t)__popcll(bl) | (uint32_t)__popcll(bm) << 16;
            }
        }
        __syncthreads();
        const uint32_t rows = lane < 3u * kLocalRows ? L.row[lane] : 0u, before = row_incl_scan(rows) - rows;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
#pragma unroll
            for (int k = 0; k < kLocalPer; ++k) {
                const uint32_t b = __builtin_amdgcn_readlane(before, a * kLocalRows + k * (kLocalThreads / 64) + wave);
                if (sg[k] == 0) continue;
                const uint32_t j = (uint32_t)k * kLocalThreads + t, from = sg[k] & 0xffffu, to = sg[k] >> 16;
                const uint32_t mid = (from + to) >> 1, i = node[k];
                // the left records of the nodes before (abs_at), and their medians
                const uint32_t bl = i * (smin >> 1) + ((smin & 1u) ? from - i * (smin + 1u) : 0u);
                const uint32_t lb = (b & 0xffffu) + (e[a][k] >> 12 & 0x7fu) - bl;
                const uint32_t mb = (b >> 16) + (e[a][k] >> 20) - i, s = e[a][k] >> 10 & 3u;
                const uint32_t dst = s == 1 ? from + lb : s == 2 ? mid : mid + 1 + ((j - from) - lb - mb);
                out[a][dst & (kLocal - 1)] = (uint16_t)(e[a][k] & 0x3ffu);
            }
        }
#pragma unroll
        for (int k = 0; k < kLocalPer; ++k) {
            const uint32_t j = (uint32_t)k * kLocalThreads + t, from = sg[k] & 0xffffu, to = sg[k] >> 16;
            const uint32_t mid = (from + to) >> 1;
            if (to == 0) continue;
            node[k] = 2 * node[k] + (j > mid ? 1u : 0u);
            sg[k] = j == mid ? 0u : j < mid ? (from | mid << 16) : ((mid + 1u) | to << 16);
        }
        smin = (smin - 1u) / 2u;
        smax /= 2u;
        __syncthreads();
        // the new segments' planes (as k_level_nodes), by their first positions
#pragma unroll
        for (int k = 0; k < kLocalPer; ++k) {
            const uint32_t j = (uint32_t)k * kLocalThreads + t, from = sg[k] & 0xffffu, to = sg[k] >> 16;
            if (to > 0 && j == from) L.plane[from] = local_plane(L, out, from, to);
        }
        __syncthreads();
    }
}

// The tree's photons in node order (nine planes), and each node's 16-byte
// descent record {x, y, z, photon index | plane << 30} (w = 0xFFFFFFFF for
// an empty slot): the kNN reads one record per visited node.
__global__ __launch_bounds__(256) void k_tree_photons(const float4* __restrict__ prec,
                                                     const uint32_t* __restrict__ node_idx,
                                                     const int8_t* __restrict__ node_plane, uint32_t cap,
                                                     float* __restrict__ out9, float4* __restrict__ nodes) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= cap) return;
    uint32_t id = node_idx[i];
    float v[9];
    if (id != kFinal) {
        const float4 a = prec[3 * (size_t)id], b = prec[3 * (size_t)id + 1], c = prec[3 * (size_t)id + 2];
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w; v[8] = c.x;
    } else {
#pragma unroll
        for (int p = 0; p < 9; ++p) v[p] = p < 3 ? __builtin_inff() : 0.f;
    }
#pragma unroll
    for (int p = 0; p < 9; ++p) out9[(size_t)p * cap + i] = v[p];
    const uint32_t w = id != kFinal ? id | ((uint32_t)node_plane[i] << 30) : kFinal;
    nodes[i] = make_float4(v[0], v[1], v[2], __uint_as_float(w));
}

// ---- model AABB (the live effect of create_kd_tree, KdTree.cu:395-464) ----
// One workgroup per model: min/max over the model's vertices with wave
// reductions. Replaces per-triangle AABBs -> 32-triangle chunks -> pairwise
// segmented reduction (KdTree.cu:82-327).
__global__ __launch_bounds__(256) void k_model_aabb(const float* __restrict__ tris9, const uint32_t* __restrict__ tb,
                                                   float* __restrict__ out) {
    __shared__ float s[4][6];
    const uint32_t m = blockIdx.x, t = threadIdx.x, lane = t & 63, wave = t >> 6;
    uint32_t v0 = tb[m] * 3, v1 = tb[m + 1] * 3;  // vertex range
    float mn[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, mx[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    for (uint32_t v = v0 + t; v < v1; v += blockDim.x) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            float p = tris9[(size_t)v * 3 + a];
            mn[a] = fminf(mn[a], p);
            mx[a] = fmaxf(mx[a], p);
        }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) {
            mn[a] = fminf(mn[a], __shfl_xor(mn[a], d, 64));
            mx[a] = fmaxf(mx[a], __shfl_xor(mx[a], d, 64));
        }
    }
    if (lane == 0)
        for (int a = 0; a < 3; ++a) {
            s[wave][a] = mn[a];
            s[wave][a + 3] = mx[a];
        }
    __syncthreads();
    if (t < 6) {
        float r = s[0][t];
        for (int w = 1; w < 4; ++w) r = t < 3 ? fminf(r, s[w][t]) : fmaxf(r, s[w][t]);
        out[(size_t)m * 6 + t] = r;
    }
}

}  // namespace

extern "C" pm_status pm_kdtree_build(pm_ctx* ctx, const float* d_photons9, uint32_t n, pm_kdtree** out) {
    if (!ctx || !out) return PM_ERR_INVALID;
    *out = nullptr;
    if (n == 0 || !d_photons9) return pm::fail(ctx, PM_ERR_INVALID, "pm_kdtree_build: no photons");
    if (n > (1u << 30)) return pm::fail(ctx, PM_ERR_UNSUPPORTED, "pm_kdtree_build: n too large");
    uint32_t L = 0;
    while (((1ull << L) - 1) < (uint64_t)n) ++L;
    const uint32_t cap = (uint32_t)((1ull << L) - 1);

    pm_kdtree* T = new pm_kdtree();
    T->n = n;
    T->cap = cap;
    T->levels = L;
    size_t bytes = pm::carve_size({(size_t)cap * 4, (size_t)cap, (size_t)cap * 36, (size_t)cap * 16});
    // (a block of the context's cache when one fits, as for grids)
    hipError_t e = pm::block_take(ctx, bytes, &T->mem, &T->mem_bytes);
    if (e != hipSuccess) {
        delete T;
        return pm::hip_fail(ctx, e, "hipMalloc(kdtree)");
    }
    T->owner = ctx;
    pm::Carve tc{static_cast<char*>(T->mem)};
    T->node_idx = tc.take<uint32_t>(cap);
    T->node_plane = tc.take<int8_t>(cap);
    T->photons = tc.take<float>((size_t)cap * 9);
    T->nodes = tc.take<float4>(cap);
    auto bail = [&](pm_status s) {
        pm_kdtree_destroy(T);
        return s;
    };

    // the three axis sorts run as one segmented sort of 3n keys
    size_t rs = pm::radix_sort_scratch_bytes(n, 3);
    const size_t rb = (size_t)n * sizeof(Rk), n3 = 3 * (size_t)n;
    size_t need = pm::carve_size({rb, rb, rb, rb, rb, rb, (size_t)n * 4, (size_t)n * 4, (size_t)cap * 8, (size_t)cap,
                                  (size_t)cap * 8, n3 * 4, n3 * 4, n3 * 4, (size_t)n * 16, rs, (size_t)n * 48,
                                  3 * kTicket * 4});
    void* work = nullptr;
    pm_status st = pm::scratch_reserve(ctx, need, &work);
    if (st != PM_OK) return bail(st);
    pm::Carve cv{static_cast<char*>(work)};
    Rk* A[3];
    Rk* B[3];
    for (int a = 0; a < 3; ++a) A[a] = cv.take<Rk>(n);
    for (int a = 0; a < 3; ++a) B[a] = cv.take<Rk>(n);
    uint32_t* node_of = cv.take<uint32_t>(n);
    uint32_t* node_of2 = cv.take<uint32_t>(n);
    uint2* seg = cv.take<uint2>(cap);
    int8_t* plane = cv.take<int8_t>(cap);
    uint2* med = cv.take<uint2>(cap);
    uint32_t* keys = cv.take<uint32_t>(n3);   // sort keys
    uint32_t* skeys = cv.take<uint32_t>(n3);  // sorted keys
    uint32_t* order = cv.take<uint32_t>(n3);  // each axis's photons in rank order
    uint32_t* rank4 = cv.take<uint32_t>(4 * (size_t)n);  // each photon's three ranks
    void* rw = cv.take<char>(rs);
    float4* prec = cv.take<float4>((size_t)n * 3);
    uint32_t* tickets = cv.take<uint32_t>(3 * kTicket);

    const uint32_t nb = pm::div_up(n, 256);
    hipStream_t s = ctx->stream;
    hipLaunchKernelGGL(k_photon_records, dim3(nb), dim3(256), 0, s, d_photons9, n, prec);
    // planes 0-2 of the block are the three coordinates, back to back
    hipLaunchKernelGGL(k_axis_keys, dim3(pm::div_up((uint32_t)n3, 256)), dim3(256), 0, s, d_photons9, (uint32_t)n3,
                       keys);
    if ((st = pm::radix_sort_pairs_auto(ctx, keys, nullptr, skeys, order, n, 32, rw, nullptr, 3)) != PM_OK)
        return bail(st);
    hipLaunchKernelGGL(k_ranks, dim3(nb, 3), dim3(256), 0, s, order, n, rank4);
    hipLaunchKernelGGL(k_rank_recs, dim3(nb, 3), dim3(256), 0, s, order, reinterpret_cast<const uint4*>(rank4), n,
                       A[0], A[1], A[2]);
    auto orders = [&] {
        Orders O;
        for (int a = 0; a < 3; ++a) O.A[a] = A[a];
        O.order = order;
        O.rank4 = rank4;
        O.ph9 = d_photons9;
        O.n = n;
        return O;
    };
    if ((st = pm::fill_u32(ctx, T->node_idx, kFinal, cap)) != PM_OK) return bail(st);
    // node_plane = -1; the carve pads every block to 256 bytes, so whole
    // words past cap stay inside the allocation.
    if ((st = pm::fill_u32(ctx, reinterpret_cast<uint32_t*>(T->node_plane), 0xFFFFFFFFu, (cap + 3) / 4)) != PM_OK)
        return bail(st);
    if ((st = pm::fill_u32(ctx, node_of, 0u, n)) != PM_OK) return bail(st);

    // Levels [0, Lg) run on the whole arrays; from level Lg every segment
    // holds at most kLocal records (a node of size s has children of at most
    // s / 2) and each subtree is finished by one workgroup in LDS.
    uint32_t Lg = 0;
    for (uint32_t smax = n; smax > (uint32_t)kLocal; smax /= 2) ++Lg;
    // a segment of at most 1024 records spans at most 11 levels (node arrays of kLocal)
    if (L - Lg > 11) return bail(pm::fail(ctx, PM_ERR_INVALID, "pm_kdtree_build: internal level split"));
    // the root's plane (and, above the LDS levels, its median)
    hipLaunchKernelGGL(k_level_nodes, dim3(1), dim3(256), 0, s, orders(), 0u, 1u, cap, n, Lg > 0, seg, plane,
                       T->node_idx, T->node_plane, med, nullptr, tickets);
    uint32_t smin = n;  // the smallest node of the level (those above the LDS levels are not empty)
    for (uint32_t lvl = 0; lvl < L; ++lvl) {
        uint32_t first = (1u << lvl) - 1, count = 1u << lvl;
        if (lvl == Lg) {
            hipLaunchKernelGGL(k_local_subtrees, dim3(count), dim3(kLocalThreads), 0, s, orders(), prec, first, seg,
                               plane, T->node_idx, T->node_plane);
            break;
        }
        if (lvl + 1 == L) break;  // every segment of the last level has size <= 1
        const uint32_t tiles = 3u * pm::div_up(n, kPTile);
        uint64_t* lstate = nullptr;
        uint32_t* lcounter = nullptr;
        const Level V{first, smin};
        // (a tile strictly inside a node knows its place from the tiles before)
        if (smin + 1u >= kPTile + 2u) {
            if ((st = pm::lookback_begin(ctx, tiles, &lstate, &lcounter)) != PM_OK) return bail(st);
            hipLaunchKernelGGL(k_level_partition<true>, dim3(tiles), dim3(kPThreads), 0, s, A[0], A[1], A[2], B[0],
                               B[1], B[2], n, node_of, node_of2, seg, med, V, lstate, lcounter, tickets);
        } else {
            hipLaunchKernelGGL(k_level_partition<false>, dim3(tiles), dim3(kPThreads), 0, s, A[0], A[1], A[2], B[0],
                               B[1], B[2], n, node_of, node_of2, seg, med, V, lstate, lcounter, tickets);
        }
        smin = (smin - 1u) / 2u;
        for (int a = 0; a < 3; ++a) std::swap(A[a], B[a]);
        std::swap(node_of, node_of2);
        // the children's planes, and their medians above the LDS levels
        uint32_t cf = (1u << (lvl + 1)) - 1, cc = 1u << (lvl + 1);
        hipLaunchKernelGGL(k_level_nodes, dim3(pm::div_up(cc, 256)), dim3(256), 0, s, orders(), cf, cc, cap, 0u,
                           lvl + 1 < Lg, seg, plane, T->node_idx, T->node_plane, med, lcounter, tickets);
    }
    hipLaunchKernelGGL(k_tree_photons, dim3(pm::div_up(cap, 256)), dim3(256), 0, s, prec, T->node_idx,
                       T->node_plane, cap, T->photons, T->nodes);
    if (hipGetLastError() != hipSuccess) return bail(pm::fail(ctx, PM_ERR_HIP, "pm_kdtree_build: launch failed"));
    *out = T;
    return PM_OK;
}

extern "C" pm_status pm_kdtree_describe(const pm_kdtree* t, pm_kdtree_desc* out) {
    if (!t || !out) return PM_ERR_INVALID;
    out->n_photons = t->n;
    out->n_slots = t->cap;
    out->levels = t->levels;
    out->d_node_idx = t->node_idx;
    out->d_node_plane = t->node_plane;
    out->d_photons = t->photons;
    return PM_OK;
}

extern "C" pm_status pm_kdtree_copy_to_host(pm_ctx* ctx, const pm_kdtree* t, uint32_t* h_node_idx,
                                            int8_t* h_node_plane) {
    if (!ctx || !t) return PM_ERR_INVALID;
    if (h_node_idx) PM_HIP(ctx, hipMemcpyAsync(h_node_idx, t->node_idx, (size_t)t->cap * 4, hipMemcpyDeviceToHost, ctx->stream));
    if (h_node_plane) PM_HIP(ctx, hipMemcpyAsync(h_node_plane, t->node_plane, t->cap, hipMemcpyDeviceToHost, ctx->stream));
    PM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return PM_OK;
}

extern "C" pm_status pm_kdtree_destroy(pm_kdtree* t) {
    if (!t) return PM_OK;
    if (t->mem && !pm::block_give(t->owner, t->mem, t->mem_bytes)) (void)hipFree(t->mem);
    delete t;
    return PM_OK;
}

namespace pm {
pm_status model_aabb_launch(pm_ctx* ctx, const float* tris9, const uint32_t* tb, int n_models, float* out6) {
    if (n_models <= 0) return PM_OK;
    hipLaunchKernelGGL(k_model_aabb, dim3(n_models), dim3(256), 0, ctx->stream, tris9, tb, out6);
    PM_CHECK_LAUNCH(ctx, "k_model_aabb");
    return PM_OK;
}
}  // namespace pm

extern "C" pm_status pm_model_aabb(pm_ctx* ctx, const float* d_tris9, const uint32_t* d_tri_begin, int32_t n_models,
                                   float* d_aabb6) {
    if (!ctx) return PM_ERR_INVALID;
    if (n_models < 0 || (n_models > 0 && (!d_tris9 || !d_tri_begin || !d_aabb6)))
        return pm::fail(ctx, PM_ERR_INVALID, "pm_model_aabb: bad arguments");
    if (n_models == 0) return PM_OK;
    hipLaunchKernelGGL(k_model_aabb, dim3(n_models), dim3(256), 0, ctx->stream, d_tris9, d_tri_begin, d_aabb6);
    PM_CHECK_LAUNCH(ctx, "k_model_aabb");
    return PM_OK;
}
