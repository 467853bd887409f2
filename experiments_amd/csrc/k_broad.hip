// k_broad.hip -- body setup and uniform-grid broadphase for gfx950.
//
//  k_setup      one pass over the body SoA: world AABB (initializeGpuAabbsFull,
//               opencl/broadphase_benchmark/broadphaseKernel.cl:293-331), cell key
//               (kCalcHashAABB, opencl/3dGridBroadphase/Shared/bt3dGridBroadphaseOCL.cl:26-47),
//               gravity and world inverse inertia (setupBodiesKernel,
//               broadphaseKernel.cl:163-212).  The reference runs these as three
//               launches with host syncs in between; here they share one read of
//               the body state.
//  k_cell_start first sorted index of every occupied cell (kFindCellStart,
//               bt3dGridBroadphaseOCL.cl:61-86).  The table is never cleared: a
//               lookup is valid only if it points at the first entry of that key
//               in the current sorted array, which a stale entry cannot.
//  k_find_pairs 27-cell stencil per small body (kFindOverlappingPairs /
//               findPairsInCell, bt3dGridBroadphaseOCL.cl:100-213), keeping the
//               overlapping bodies of lower index in a sorted per-body list in LDS.
//  k_large_pairs overflow list (kFindPairsLarge, :216-264): one workgroup per
//               large body tests its scene, in index order.
//  k_emit_pairs  int2 (x > y) pairs at scanned offsets (countOverlappingpairs /
//               squeezePairCaches, opencl/broadphase_benchmark/computeAabbKernelOCL.cl:40-111),
//               globally sorted by (x, y).
#include <float.h>
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>
#include <utility>

#include "dmath.h"
#include "rb_internal.h"

using namespace rb;

namespace {

constexpr uint32_t KEY_NONE = 0xffffffffu;

// LDS written by lanes of this wave, then read by others of it
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ void grid_pos(float4 mn, float4 mx, float inv_cell, const int *dims,
                                         int gp[3]) {
    float cx = (mn.x + mx.x) * 0.5f, cy = (mn.y + mx.y) * 0.5f, cz = (mn.z + mx.z) * 0.5f;
    gp[0] = ((int)floorf(cx * inv_cell)) & (dims[0] - 1);
    gp[1] = ((int)floorf(cy * inv_cell)) & (dims[1] - 1);
    gp[2] = ((int)floorf(cz * inv_cell)) & (dims[2] - 1);
}
__device__ __forceinline__ uint32_t pos_hash(int x, int y, int z, const int *dims) {
    x &= dims[0] - 1;
    y &= dims[1] - 1;
    z &= dims[2] - 1;
    return (uint32_t)(z * dims[1] * dims[0] + y * dims[0] + x);
}

// Stencil cells that can hold a member overlapping the AABB [mn, mx]: a
// member of cell k (unwrapped, along one axis) has its centre in
// [k c, (k+1) c) and a half-extent of at most c/2 (the grid's cell covers
// every member), so its AABB lies in [k c - c/2, (k+1) c + c/2].  Bit q of the
// result (q = 9 (dz+1) + 3 (dy+1) + (dx+1)) is set unless that cell is
// provably out of reach; wrapped aliases of a cell only hold members farther
// away, which the AABB test rejects anyway.  On an axis of two cells both
// neighbours are the same cell and on an axis of one cell all three are: the
// first of them stands for the others, so that no cell is searched twice.
__device__ __forceinline__ uint32_t reachable_cells(float4 mn, float4 mx, float inv_cell,
                                                    const int *dims) {
    const float c = 1.0f / inv_cell, h = 0.5f * c, eps = 1e-4f * c;
    const float lo[3] = {mn.x, mn.y, mn.z}, hi[3] = {mx.x, mx.y, mx.z};
    uint32_t ok[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const float ctr = (lo[k] + hi[k]) * 0.5f;
        const float g = floorf(ctr * inv_cell);
        ok[k] = 0;
#pragma unroll
        for (int d = -1; d <= 1; d++) {
            const float c0 = (g + (float)d) * c - h - eps, c1 = (g + (float)(d + 1)) * c + h + eps;
            if (hi[k] >= c0 && lo[k] <= c1) ok[k] |= 1u << (d + 1);
        }
        if (dims[k] == 2) ok[k] = (ok[k] & 2u) | (ok[k] & 5u ? 1u : 0u);
        if (dims[k] == 1) ok[k] = ok[k] ? 2u : 0u;
    }
    uint32_t m = 0;
#pragma unroll
    for (int q = 0; q < 27; q++)
        if (((ok[0] >> (q % 3)) & 1u) && ((ok[1] >> ((q / 3) % 3)) & 1u) && ((ok[2] >> (q / 9)) & 1u))
            m |= 1u << q;
    return m;
}

struct GridP {
    float inv_cell;
    int dims[3];
    int cell_bits;
};

__global__ __launch_bounds__(256) void k_setup(
    int n, const float4 *__restrict__ pos, const float4 *__restrict__ quat,
    float4 *__restrict__ linvel, float4 *__restrict__ angvel, const float *__restrict__ inv_mass,
    const int *__restrict__ shape, const int *__restrict__ scene, const int *__restrict__ is_large,
    const HullInfo *__restrict__ hulls, const float4 *__restrict__ inv_inertia_local,
    float4 *__restrict__ inv_inertia_world, float4 *__restrict__ aabb_min,
    float4 *__restrict__ aabb_max, uint2 *__restrict__ kv, GridP g, float gx, float gy, float gz,
    float dt, uint32_t *__restrict__ occ, int occ_words) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    // the cell occupancy bits of the previous step
    for (int w = i; w < occ_words; w += gridDim.x * blockDim.x) occ[w] = 0u;
    if (i >= n) return;
    float4 p = pos[i], q = quat[i];
    const HullInfo *h = hulls + shape[i];
    float4 hmn = h->aabb_min, hmx = h->aabb_max;
    float4 he = mk4((hmx.x - hmn.x) * 0.5f, (hmx.y - hmn.y) * 0.5f, (hmx.z - hmn.z) * 0.5f, 0.f);
    float4 lc = mk4((hmx.x + hmn.x) * 0.5f, (hmx.y + hmn.y) * 0.5f, (hmx.z + hmn.z) * 0.5f, 0.f);
    float4 wc = xform(lc, p, q);
    float4 m[3];
    abs_rot(q, m);
    float4 ext = mk4(dot3(m[0], he), dot3(m[1], he), dot3(m[2], he), 0.f);
    float4 mn = mk4(wc.x - ext.x, wc.y - ext.y, wc.z - ext.z, 0.f);
    float4 mx = mk4(wc.x + ext.x, wc.y + ext.y, wc.z + ext.z, 0.f);
    aabb_min[i] = mn;
    aabb_max[i] = mx;
    uint32_t key = KEY_NONE;
    if (!is_large[i]) {
        int gp[3];
        grid_pos(mn, mx, g.inv_cell, g.dims, gp);
        key = pos_hash(gp[0], gp[1], gp[2], g.dims) | ((uint32_t)scene[i] << g.cell_bits);
    }
    kv[i] = make_uint2(key, (uint32_t)i);
    float im = inv_mass[i];
    float4 *I = inv_inertia_world + 3 * i;
    if (im != 0.f) {
        float4 v = linvel[i];
        v.x = v.x + gx * dt;
        v.y = v.y + gy * dt;
        v.z = v.z + gz * dt;
        linvel[i] = v;
        float4 d = inv_inertia_local[i];
        float4 mt[3] = {mk4(m[0].x, m[1].x, m[2].x, 0.f), mk4(m[0].y, m[1].y, m[2].y, 0.f),
                        mk4(m[0].z, m[1].z, m[2].z, 0.f)};
        float4 loc[3] = {mk4(d.x, 0.f, 0.f, 0.f), mk4(0.f, d.y, 0.f, 0.f), mk4(0.f, 0.f, d.z, 0.f)};
        float4 tmp[3], out[3];
        // mtMul(a, b): ans[i][j] = dot3(a.row[i], b.col[j]) (broadphaseKernel.cl:130-148)
        for (int r = 0; r < 3; r++) {
            float4 c0 = mk4(loc[0].x, loc[1].x, loc[2].x, 0.f);
            float4 c1 = mk4(loc[0].y, loc[1].y, loc[2].y, 0.f);
            float4 c2 = mk4(loc[0].z, loc[1].z, loc[2].z, 0.f);
            tmp[r] = mk4(dot3(m[r], c0), dot3(m[r], c1), dot3(m[r], c2), 0.f);
        }
        for (int r = 0; r < 3; r++) {
            float4 c0 = mk4(mt[0].x, mt[1].x, mt[2].x, 0.f);
            float4 c1 = mk4(mt[0].y, mt[1].y, mt[2].y, 0.f);
            float4 c2 = mk4(mt[0].z, mt[1].z, mt[2].z, 0.f);
            out[r] = mk4(dot3(tmp[r], c0), dot3(tmp[r], c1), dot3(tmp[r], c2), 0.f);
        }
        I[0] = out[0];
        I[1] = out[1];
        I[2] = out[2];
    } else {
        float4 z = mk4(0.f, 0.f, 0.f, 0.f);
        linvel[i] = z;
        angvel[i] = z;
        I[0] = z;
        I[1] = z;
        I[2] = z;
    }
}

// First sorted index and occupancy bit of every occupied cell, and the AABBs
// in sorted order with their keys and indices (the pair search reads a cell
// member in one 32-byte piece).  occ[] was cleared by k_setup.
__global__ void k_cell_start(const uint2 *__restrict__ kv, int n,
                             const float4 *__restrict__ aabb_min,
                             const float4 *__restrict__ aabb_max, uint32_t *__restrict__ cell_start,
                             uint32_t *__restrict__ occ, float4 *__restrict__ boxes) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    uint2 e = kv[s];
    float4 mn = aabb_min[e.y], mx = aabb_max[e.y];
    mn.w = __uint_as_float(e.x);
    mx.w = __uint_as_float(e.y);
    boxes[2 * (size_t)s] = mn;
    boxes[2 * (size_t)s + 1] = mx;
    if (e.x == KEY_NONE) return;
    if (s == 0 || kv[s - 1].x != e.x) {
        cell_start[e.x] = (uint32_t)s;
        atomicOr(&occ[e.x >> 5], 1u << (e.x & 31u));
    }
}

// Stencil rows: the three cells of a row along x are one key range (z and y
// the outer strides of the key), so a wave that looks for the neighbours of
// OWN sorted boxes lists the rows that hold members and its lanes walk one
// listed row at a time, two members a read, taking the next one off the list
// when they are through.  (A lane per entry or a lane per few cells, which
// walked its own cells, left 64 lanes to wait for the longest of their chains
// of dependent reads.)
template <int OWN, int ROWS>
struct RowsLDS {
    float4 mn[OWN], mx[OWN];  // the wave's boxes, key and index in their w
    uint32_t first[ROWS];     // a row's first key
    uint32_t start[ROWS];     // its first member, 0: cell_start of the key
    uint8_t own[ROWS];        // the box and, from bit 6, the cells after the first
};
// boxes: the AABBs in sorted order, two float4 each with the key and the index
// in their w.  hits(m, c, o): the lanes of m hold a member, body c, that
// overlaps the wave's box o; it tells a lane of them to leave its row.  LOWER:
// only members of lower index than the box's.
template <bool LOWER, int OWN, int ROWS, class Hits>
__device__ __forceinline__ void walk_rows(int n, uint32_t total,
                                          const uint32_t *__restrict__ cell_start,
                                          const float4 *__restrict__ boxes,
                                          RowsLDS<OWN, ROWS> &S, Hits hits) {
    const uint32_t lane = threadIdx.x & 63;
    wave_fence();
    for (uint32_t p = lane; p < total; p += 64)
        if (S.start[p] == 0u) S.start[p] = cell_start[S.first[p]];
    wave_fence();
    uint32_t at = 64u, u = 0u, last = 0u;
    int o = 0, y = 0;
    float4 a = mk4(0.f, 0.f, 0.f, 0.f), b = a;
    bool walk = lane < total;
    auto take = [&](uint32_t p) {
        const uint32_t w = S.own[p];
        o = (int)(w & 63u);
        a = S.mn[o];
        b = S.mx[o];
        u = S.start[p];
        last = S.first[p] + (w >> 6);
        y = __float_as_int(b.w);
    };
    if (walk) take(lane);
    while (__ballot(walk)) {
        bool hit[2] = {false, false}, end = false;
        int c[2] = {0, 0};
        if (walk) {
            const uint32_t v = u + 1u < (uint32_t)n ? u + 1u : u;
            const float4 p0 = boxes[2 * (size_t)u], q0 = boxes[2 * (size_t)u + 1];
            const float4 p1 = boxes[2 * (size_t)v], q1 = boxes[2 * (size_t)v + 1];
            const bool in0 = __float_as_uint(p0.w) <= last;
            const bool in1 = in0 && v != u && __float_as_uint(p1.w) <= last;
            c[0] = __float_as_int(q0.w);
            c[1] = __float_as_int(q1.w);
            hit[0] = in0 && (!LOWER || c[0] < y) && aabb_overlap(a, b, p0, q0);
            hit[1] = in1 && (!LOWER || c[1] < y) && aabb_overlap(a, b, p1, q1);
            u += 2u;
            end = !in1 || u >= (uint32_t)n;
        }
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const uint64_t m = __ballot(hit[k]);
            if (m && hits(m, c[k], o)) end = true;
        }
        const uint64_t done = __ballot(end);
        if (done) {
            if (end) {
                const uint32_t p = __builtin_amdgcn_mbcnt_hi(
                    (uint32_t)(done >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)done, at));
                walk = p < total;
                if (walk) take(p);
            }
            at += (uint32_t)__popcll(done);
        }
    }
    wave_fence();
}
// Occupied cells among x - 1, x, x + 1 (bits 0 to 2) of the row at key b, from
// the occupancy words of the outer two.  (Rows of two or more cells start at
// even keys: at the grid's edge x still lies in the word of one of them.)
__device__ __forceinline__ uint32_t row_bits(uint32_t wl, uint32_t wr, uint32_t b, uint32_t xl,
                                             uint32_t x, uint32_t xr) {
    const uint32_t wc = ((b | x) >> 5) == ((b | xl) >> 5) ? wl : wr;
    return ((wl >> ((b | xl) & 31u)) & 1u) | ((wc >> ((b | x) & 31u)) & 1u) << 1 |
           ((wr >> ((b | xr) & 31u)) & 1u) << 2;
}
// List a row's cells m (not wrapped: adjacent keys) of the wave's box `own`
// behind the total rows before; every lane of the wave calls it.
template <int OWN, int ROWS>
__device__ __forceinline__ void list_row(RowsLDS<OWN, ROWS> &S, uint32_t &total, uint32_t m,
                                         uint32_t b, uint32_t x, uint32_t xmask, int own,
                                         uint32_t start) {
    const uint64_t has = __ballot(m != 0u);
    if (m) {
        const uint32_t p = __builtin_amdgcn_mbcnt_hi(
            (uint32_t)(has >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)has, total));
        const uint32_t lo = (uint32_t)__builtin_ctz(m), hi = 31u - (uint32_t)__builtin_clz(m);
        S.first[p] = b | ((x + lo - 1u) & xmask);
        S.start[p] = start;
        S.own[p] = (uint8_t)((uint32_t)own | (hi - lo) << 6);
    }
    total += (uint32_t)__popcll(has);
}

// The pair search: a wave per OWN sorted entries, 64 / OWN lanes an entry.  The
// lanes list the entry's stencil rows that hold members within reach, the wave
// walks them (walk_rows), and an entry's overlaps with bodies of lower index go
// to its list, the scene's large bodies after them, which is then ordered by
// rank.  An entry with more than K overlaps keeps the first K that a serial
// search meets (cells in stencil order, z then y then x, members in sorted
// order).  Bound by the latency of the member reads.  (A lane per entry,
// walking the occupied cells in turn: 276 us at 3.4M pairs of 4,096 scenes, now
// 183; 32 lanes an entry, a cell each: 113 us at 65,537 hulls, now 63.)
// Few bodies leave lanes idle, so there a wave takes 2 or 4 entries and lists
// each cell by itself, which shortens the longest walk (us; cubes in columns,
// then hulls in layers):
//   bodies                1,000   4,096 | 5,000  10,000  24,000  49,152  65,537
//   2 entries, cells        8.9     8.9 |  15.0    19.6    37.6    70.9    94.0
//   4 entries, cells       10.9    10.7 |  18.0    20.4    30.3    51.2    66.4
//   4 entries, rows        14.9    13.9 |  30.1    32.6    42.3            100
//   16 entries, rows       23.0    23.6 |  46.0    49.9    53.3    60.4    63.0
//   32 lanes, a cell each   7.9     8.4 |  20.3    25.2    47.2    84.9     113
constexpr int FP_WAVES = 4;
constexpr int FP_TWO = 1 << 13, FP_FOUR = 3 << 14;  // below: 2, 4 entries a wave
constexpr int FP_LIST = RB_MAX_BODY_PAIRS;  // K is no larger
template <int OWN>
struct FindLDS {
    static constexpr bool CELLS = OWN < 16;
    RowsLDS<OWN, OWN * (CELLS ? 27 : 9)> rows;
    uint32_t count[OWN];
    int list[OWN][FP_LIST | 1];
};

// Half a wave each for two entries (mn0, mx0; on: there is one): the first K
// overlaps in the order of a serial search.  The cells of a stencil row follow
// each other in the sorted order too, so a half reads a row 32 members at a
// time and stops at the K-th overlap.  Searches where many lists overflow, us:
// 60,000 cubes in a box of 16 and K = 64 460, K = 16 370, in one of 40 and K = 8
// 67, 12,000 in one of 10 and K = 64 112.  (A wave an entry, a cell a lane,
// counted and then stored, after a walk to the rows' ends: 1,293, 1,454, 93 and
// 308; 32 lanes an entry from the start, a cell each: 418, 424, 53 and 87.)
__device__ __forceinline__ void first_overlaps(bool on, int n,
                                               const uint32_t *__restrict__ cell_start,
                                               const uint32_t *__restrict__ occ,
                                               const float4 *__restrict__ boxes, const GridP &g,
                                               float4 mn0, float4 mx0, int *__restrict__ lst,
                                               int K) {
    const int q = threadIdx.x & 31, i = __float_as_int(mx0.w);
    const uint32_t half = threadIdx.x & 32;
    const uint32_t key = __float_as_uint(mn0.w), sk = key >> g.cell_bits << g.cell_bits;
    int gp[3];
    grid_pos(mn0, mx0, g.inv_cell, g.dims, gp);
    uint32_t nk = 0, u0 = 0;
    bool has = false;
    if (on && q < 27 && ((reachable_cells(mn0, mx0, g.inv_cell, g.dims) >> q) & 1u)) {
        nk = pos_hash(gp[0] + q % 3 - 1, gp[1] + (q / 3) % 3 - 1, gp[2] + q / 9 - 1, g.dims) | sk;
        has = (occ[nk >> 5] >> (nk & 31u)) & 1u;
        if (has) u0 = cell_start[nk];
    }
    // (below, every value but the member's is the same in a half's lanes)
    uint32_t cells = (uint32_t)(__ballot(has) >> half);
    uint32_t u = 0, last = 0;
    int c = 0;
    bool in_row = false;
    while (__ballot(c < K && (in_row || cells))) {
        // the row's cells from the first one left on, or that one alone where
        // they wrap round the grid's edge
        const int a = cells ? __builtin_ctz(cells) : 0;
        const uint32_t row = cells & (7u << (a - a % 3));
        const int z = row ? 31 - __builtin_clz(row) : 0;
        const uint32_t first = __shfl(nk, a, 32), end = __shfl(nk, z, 32);
        const uint32_t start = __shfl(u0, a, 32);
        if (!in_row) {
            const bool whole = end - first == (uint32_t)(z - a);
            last = whole ? end : first;
            u = start;
            in_row = cells != 0u;
            cells &= whole ? ~row : cells - 1u;
        }
        const uint32_t v = u + (uint32_t)q;
        bool in = in_row && c < K && v < (uint32_t)n, hit = false;
        int j = 0;
        if (in) {
            const float4 p = boxes[2 * (size_t)v], m = boxes[2 * (size_t)v + 1];
            j = __float_as_int(m.w);
            in = __float_as_uint(p.w) <= last;
            hit = in && j < i && aabb_overlap(mn0, mx0, p, m);
        }
        const uint32_t h = (uint32_t)(__ballot(hit) >> half);
        const int at = c + (int)__popc(h & ((1u << q) - 1u));
        if (hit && at < K) lst[at] = j;
        c += (int)__popc(h);
        in_row = (uint32_t)(__ballot(in) >> half) == 0xffffffffu;
        u += 32u;
    }
}

template <int OWN>
__global__ __launch_bounds__(64 * FP_WAVES) void k_find_pairs(
    int n, const uint32_t *__restrict__ cell_start, const uint32_t *__restrict__ occ,
    const float4 *__restrict__ boxes, const float4 *__restrict__ aabb_min,
    const float4 *__restrict__ aabb_max, const int *__restrict__ large_list,
    const int *__restrict__ large_first, const int *__restrict__ large_num, GridP g, int K,
    int *__restrict__ body_slots, uint32_t *__restrict__ pair_count, int *overflow) {
    constexpr int LANES = 64 / OWN;
    __shared__ FindLDS<OWN> s_find[FP_WAVES];
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    FindLDS<OWN> &S = s_find[w];
    const int t0 = ((int)blockIdx.x * FP_WAVES + w) * OWN;
    if (t0 >= n) return;
    const int own = lane / LANES, sub = lane & (LANES - 1);
    const int t = t0 + own;
    float4 mn0 = mk4(0.f, 0.f, 0.f, 0.f), mx0 = mn0;
    uint32_t key = KEY_NONE;  // (large bodies: k_large_count / k_large_write)
    if (t < n) {
        mn0 = boxes[2 * (size_t)t];
        mx0 = boxes[2 * (size_t)t + 1];
        key = __float_as_uint(mn0.w);
    }
    if (sub == 0) {
        S.rows.mn[own] = mn0;
        S.rows.mx[own] = mx0;
        S.count[own] = 0u;
    }
    const int i = __float_as_int(mx0.w);
    // the entry's rows sub, sub + LANES, ..: their cells that hold members
    // within reach (bit dx + 1)
    constexpr int R = (9 + LANES - 1) / LANES;
    const uint32_t xmask = (uint32_t)g.dims[0] - 1u;
    uint32_t bits[R], base[R], wrap0 = 0u, wrap2 = 0u;
    int gp[3] = {0, 0, 0};
    grid_pos(mn0, mx0, g.inv_cell, g.dims, gp);
    const uint32_t x = (uint32_t)gp[0], xl = (x - 1u) & xmask, xr = (x + 1u) & xmask;
    {
        const uint32_t reach = key != KEY_NONE ? reachable_cells(mn0, mx0, g.inv_cell, g.dims) : 0u;
        const uint32_t sk = key >> g.cell_bits << g.cell_bits;
        uint32_t wl[R], wr[R];
#pragma unroll
        for (int k = 0; k < R; k++) {
            const int r = sub + k * LANES;
            bits[k] = r < 9 ? (reach >> (3 * r)) & 7u : 0u;
            base[k] = sk | pos_hash(0, gp[1] + r % 3 - 1, gp[2] + r / 3 - 1, g.dims);
            wl[k] = bits[k] ? occ[(base[k] | xl) >> 5] : 0u;
            wr[k] = bits[k] ? occ[(base[k] | xr) >> 5] : 0u;
        }
#pragma unroll
        for (int k = 0; k < R; k++) bits[k] &= row_bits(wl[k], wr[k], base[k], xl, x, xr);
    }
    // (an entry with more than K overlaps is searched again: the rest of its
    // rows need not be walked)
    auto keep = [&](uint64_t m, int c, int o) {
        if (((m >> lane) & 1ull) == 0ull) return false;
        const uint32_t p = atomicAdd(&S.count[o], 1u);
        if (p < (uint32_t)K) S.list[o][p] = c;
        return p >= (uint32_t)K;
    };
    // by rows, round 0: the rows; rounds 1 and 2: their cells wrapped round the
    // grid's edge (x - 1 of cell 0, x + 1 of the last)
    for (int round = 0; round < 3; round++) {
        uint32_t total = 0;
        bool more = false;
#pragma unroll
        for (int k = 0; k < R; k++) {
            if constexpr (FindLDS<OWN>::CELLS) {
#pragma unroll
                for (int d = 0; d < 3; d++)
                    list_row(S.rows, total, bits[k] & (1u << d), base[k], x, xmask, own, 0u);
            } else {
                const uint32_t edge = (x == 0u ? 1u : 0u) | (x == xmask ? 4u : 0u);
                const uint32_t m =
                    bits[k] & (round == 0 ? ~edge : round == 1 ? edge & 1u : edge & 4u);
                more |= (bits[k] & edge) != 0u;
                list_row(S.rows, total, m, base[k], x, xmask, own, 0u);
            }
        }
        if (total) walk_rows<true>(n, total, cell_start, boxes, S.rows, keep);
        if (__ballot(more) == 0ull) break;
    }
    wave_fence();
    uint32_t c = S.count[own];
    for (uint64_t over = __ballot(sub == 0 && c > (uint32_t)K); over;) {
        const int o0 = __builtin_ctzll(over) / LANES;
        over &= over - 1ull;
        const bool two = over != 0ull;
        const int o = two && lane >= 32 ? __builtin_ctzll(over) / LANES : o0;
        over &= over - 1ull;  // (0 stays 0)
        first_overlaps(two || lane < 32, n, cell_start, occ, boxes, g, S.rows.mn[o], S.rows.mx[o],
                       S.list[o], K);
    }
    int *dst = body_slots + (size_t)i * K, *lst = S.list[own];
    if (large_num) {
        const int sc = key != KEY_NONE ? (int)(key >> g.cell_bits) : -1;
        const int l0 = sc >= 0 ? large_first[sc] : 0, nl = sc >= 0 ? large_num[sc] : 0;
        const uint64_t segmask = LANES == 64 ? ~0ull : ((1ull << LANES) - 1ull);
        for (int q0 = 0; q0 < nl; q0 += LANES) {
            const int q = q0 + sub;
            bool hit = false, stop = false;
            int L = 0;
            if (q < nl) {
                L = large_list[l0 + q];
                stop = L >= i;  // list sorted by index
                hit = !stop && aabb_overlap(mn0, mx0, aabb_min[L], aabb_max[L]);
            }
            const uint64_t hm = (__ballot(hit) >> (LANES * own)) & segmask;
            const uint64_t sm = (__ballot(stop) >> (LANES * own)) & segmask;
            if (hit) {
                const uint32_t p = c + (uint32_t)__popcll(hm & ((1ull << sub) - 1ull));
                if (p < (uint32_t)K) lst[p] = L;
            }
            c += (uint32_t)__popcll(hm);
            if (sm) break;
        }
    }
    if (c > (uint32_t)K) {
        if (sub == 0) atomicOr(overflow, (int)MI_RB_OVERFLOW_BODY_PAIRS);
        c = (uint32_t)K;
    }
    wave_fence();
    // ordered by rank (a large body's entry has none)
    for (uint32_t p = sub; p < c; p += LANES) {
        const int j = lst[p];
        uint32_t r = 0;
        for (uint32_t k = 0; k < c; k++) r += lst[k] < j ? 1u : 0u;
        dst[r] = j;
    }
    if (sub == 0 && key != KEY_NONE) pair_count[i] = c;
}

// Overflow list: pairs (x, j) of each large body x with every body j < x of
// its scene.  The scene range is split into chunks of LARGE_CHUNK bodies, one
// workgroup per (large body, chunk): a counting pass, then an ordered writing
// pass that places each chunk after the counts of the chunks before it.
constexpr int LARGE_CHUNK = RB_LARGE_CHUNK;

__device__ __forceinline__ int large_range(const int *large_list, const int *scene,
                                           const int *scene_start, int q, int c, int &x, int &j0,
                                           int &j1) {
    x = large_list[q];
    int s0 = scene ? scene_start[scene[x]] : 0;
    j0 = s0 + c * LARGE_CHUNK;
    j1 = j0 + LARGE_CHUNK < x ? j0 + LARGE_CHUNK : x;
    return j0 < j1;
}

__global__ __launch_bounds__(256) void k_large_count(
    const int *__restrict__ large_list, const int *__restrict__ scene,
    const int *__restrict__ scene_start, const float4 *__restrict__ aabb_min,
    const float4 *__restrict__ aabb_max, int nchunks, uint32_t *__restrict__ chunk_cnt) {
    __shared__ uint32_t s_n;
    const int q = blockIdx.x, c = blockIdx.y;
    int x, j0, j1;
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    if (large_range(large_list, scene, scene_start, q, c, x, j0, j1)) {
        float4 mn0 = aabb_min[x], mx0 = aabb_max[x];
        uint32_t cnt = 0;
        for (int j = j0 + threadIdx.x; j < j1; j += 256)
            cnt += aabb_overlap(mn0, mx0, aabb_min[j], aabb_max[j]) ? 1u : 0u;
        if (cnt) atomicAdd(&s_n, cnt);
    }
    __syncthreads();
    if (threadIdx.x == 0) chunk_cnt[q * nchunks + c] = s_n;
}

__global__ __launch_bounds__(256) void k_large_write(
    const int *__restrict__ large_list, const int *__restrict__ large_off,
    const int *__restrict__ scene, const int *__restrict__ scene_start,
    const float4 *__restrict__ aabb_min, const float4 *__restrict__ aabb_max, int nchunks,
    const uint32_t *__restrict__ chunk_cnt, int *__restrict__ large_slots,
    uint32_t *__restrict__ pair_count) {
    __shared__ uint32_t s_w[4];
    __shared__ uint32_t s_base;
    const int q = blockIdx.x, c = blockIdx.y;
    int x, j0, j1;
    int have = large_range(large_list, scene, scene_start, q, c, x, j0, j1);
    if (threadIdx.x == 0) {
        uint32_t base = 0, tot = 0;
        for (int k = 0; k < nchunks; k++) {
            uint32_t v = chunk_cnt[q * nchunks + k];
            if (k < c) base += v;
            tot += v;
        }
        s_base = base;
        if (c == 0) pair_count[large_list[q]] = tot;
    }
    __syncthreads();
    if (!have) return;
    int *dst = large_slots + large_off[q];
    float4 mn0 = aabb_min[x], mx0 = aabb_max[x];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int b0 = j0; b0 < j1; b0 += 256) {
        int j = b0 + threadIdx.x;
        bool hit = j < j1 && aabb_overlap(mn0, mx0, aabb_min[j], aabb_max[j]);
        uint64_t bal = __ballot(hit);
        uint32_t below = (uint32_t)__popcll(bal & lanemask_lt());
        if (lane == 0) s_w[wave] = (uint32_t)__popcll(bal);
        __syncthreads();
        uint32_t off = s_base, tot = 0;
        for (int w = 0; w < 4; w++) {
            if (w < wave) off += s_w[w];
            tot += s_w[w];
        }
        if (hit) dst[off + below] = j;
        __syncthreads();
        if (threadIdx.x == 0) s_base += tot;
        __syncthreads();
    }
}

// Lists into the pair array: EMIT_LANES lanes a body, whose list of a few
// partners they read and write as one run; then, for the overflow-list bodies,
// whose lists can hold a whole scene's worth, as many workgroups a body as its
// scene's size can use, up to 32.  (3.4M pairs of 4,096 scenes: a thread a body
// 88 us and 32 workgroups for each scene's ground 29 more, now 31; 16 for
// each ground, mostly idle, 52.)
constexpr int EMIT_LANES = 8;
__global__ __launch_bounds__(256) void k_emit_pairs(
    int n, int body_blocks, int large_blocks, const uint32_t *__restrict__ pair_count,
    const uint32_t *__restrict__ pair_off, const int *__restrict__ body_slots, int K,
    const int *__restrict__ is_large, const int *__restrict__ large_list,
    const int *__restrict__ large_off, const int *__restrict__ large_slots, int max_pairs,
    int2 *__restrict__ pairs, const uint32_t *total, int *num_pairs, int *overflow) {
    const int b = (int)blockIdx.x;
    int x;
    uint32_t k0, step;
    const int *src;
    if (b < body_blocks) {
        if (b == 0 && threadIdx.x == 0) {
            uint32_t tt = *total;
            if (tt > (uint32_t)max_pairs) {
                atomicOr(overflow, (int)MI_RB_OVERFLOW_PAIRS);
                tt = (uint32_t)max_pairs;
            }
            *num_pairs = (int)tt;
        }
        x = b * (256 / EMIT_LANES) + (int)threadIdx.x / EMIT_LANES;
        if (x >= n) return;
        if (is_large && is_large[x]) return;
        k0 = threadIdx.x % EMIT_LANES;
        step = EMIT_LANES;
        src = body_slots + (size_t)x * K;
    } else {
        const int q = (b - body_blocks) / large_blocks;
        x = large_list[q];
        k0 = (uint32_t)((b - body_blocks) % large_blocks) * blockDim.x + threadIdx.x;
        step = (uint32_t)large_blocks * blockDim.x;
        src = large_slots + large_off[q];
    }
    const uint32_t c = pair_count[x], off = pair_off[x];
    for (uint32_t k = k0; k < c; k += step) {
        const uint32_t o = off + k;
        if (o < (uint32_t)max_pairs) pairs[o] = make_int2(x, src[k]);
    }
}


// ---- hierarchical grid (stand-alone grid API) ----
// Level l has cells of cell0 * 2^l; an AABB lives on the lowest level whose
// cell is at least its largest extent, keyed (level << cell_bits) | cell of
// its centre.  Two overlapping AABBs on levels lx <= ly have centres within
// one level-ly cell per axis, so each pair is found exactly once, by the
// lower-level body: its 27 own-level neighbour cells (partners of lower index)
// and the 27 cells around its centre on every higher level (all partners).
struct HGridP {
    float inv_cell0;
    int dims[3];
    int cell_bits;
    int levels;
};

__device__ __forceinline__ int hg_level(float4 mn, float4 mx, float inv_cell0, int levels) {
    float ext = fmaxf(fmaxf(mx.x - mn.x, mx.y - mn.y), mx.z - mn.z) * inv_cell0;
    float c = 1.f;
    for (int l = 0; l < levels; l++, c *= 2.f)
        if (ext <= c) return l;
    return -1;
}
__device__ __forceinline__ void hg_cell(float4 mn, float4 mx, float inv_l, const int *dims,
                                        int gp[3]) {
    grid_pos(mn, mx, inv_l, dims, gp);
}

__global__ __launch_bounds__(256) void k_hg_hash(const float4 *__restrict__ mn,
                                                 const float4 *__restrict__ mx, int n, HGridP g,
                                                 uint2 *__restrict__ kv, uint32_t *__restrict__ counts,
                                                 uint32_t *__restrict__ cursor,
                                                 uint32_t *__restrict__ big_n, int *overflow,
                                                 float4 *__restrict__ raw) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) { big_n[0] = 0u; big_n[1] = 0u; }
    if (i >= n) return;
    counts[i] = 0u;
    cursor[i] = 0u;
    float4 a = mn[i], b = mx[i];
    // both halves in one line, for k_hg_cells to gather (1,048,576 boxes: 64 us
    // to 51 there for 8 more here)
    raw[2 * (size_t)i] = a;
    raw[2 * (size_t)i + 1] = b;
    int l = hg_level(a, b, g.inv_cell0, g.levels);
    uint32_t key = KEY_NONE;
    if (l < 0) {
        atomicOr(overflow, (int)MI_RB_OVERFLOW_LEVEL);
    } else {
        int gp[3];
        hg_cell(a, b, g.inv_cell0 * exp2f(-(float)l), g.dims, gp);
        key = ((uint32_t)l << g.cell_bits) | pos_hash(gp[0], gp[1], gp[2], g.dims);
    }
    kv[i] = make_uint2(key, (uint32_t)i);
}

// Cell starts of the sorted keys, the occupancy bit of every occupied cell,
// a flag per occupied level, and the AABBs in sorted order, two float4 each
// with the key and the index in their w (so that a cell member is one 32-byte
// read).  occ[] and the level flags after it are cleared before this kernel.
__global__ __launch_bounds__(256) void k_hg_cells(const uint2 *__restrict__ kv, int n,
                                                  const float4 *__restrict__ raw, HGridP g,
                                                  uint32_t *__restrict__ cell_start,
                                                  uint32_t *__restrict__ occ,
                                                  uint32_t *__restrict__ level_used,
                                                  float4 *__restrict__ boxes) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    uint2 e = kv[s];
    float4 mn = raw[2 * (size_t)e.y], mx = raw[2 * (size_t)e.y + 1];
    mn.w = __uint_as_float(e.x);
    mx.w = __uint_as_float(e.y);
    boxes[2 * (size_t)s] = mn;
    boxes[2 * (size_t)s + 1] = mx;
    if (e.x == KEY_NONE) return;
    if (s == 0 || kv[s - 1].x != e.x) {
        cell_start[e.x] = (uint32_t)s;
        atomicOr(&occ[e.x >> 5], 1u << (e.x & 31u));
        level_used[e.x >> g.cell_bits] = 1u;
    }
}

// The pair search: a wave per HG_OWN sorted entries.
//
// An entry looks for the members after it on its own level (the rest of its
// cell and the 13 cells after it in (z, y, x) order, so that each pair is met
// from one side) and for all members of the 27 cells around it on each coarser
// level.  The three cells of a stencil row are one key range, so a row is one
// walk over the sorted boxes; at the grid's edge the wrapped cell is a walk of
// its own.
//
// 1. Lane (entry, level) reads the occupancy bits of its rows and lists those
//    that hold a member within reach.  2. The lanes look the listed rows'
//    starts up.  3. Each lane walks one row at a time and takes the next one
//    of the list when it is through.
//
// What bounds it is the latency of dependent reads of single members.  With
// eight lanes an entry that each walked the occupied ones of their own four
// cells, level after level, 64 lanes waited for the longest walk of each step:
// 509 us at 1,048,576 bodies on four levels; listed rows keep the lanes on
// members: 199, and 166 with two members a read.  (The write pass read 24
// words an entry again, 87 us; it now streams the pairs that this pass left:
// 40.)
constexpr int HG_OWN = RB_HG_OWN, HG_REC = RB_HG_REC;
constexpr int HG_WAVES = 4;
// rows of an entry on the lowest of four levels: 5 of its own, 9 of each other
constexpr int HG_ROWS = HG_OWN * 32;
using HGLDS = RowsLDS<HG_OWN, HG_ROWS>;

// hits(m, c, y): the lanes of m hold a pair of bodies c and y
// (as walk_rows calls it)
template <class Hits>
__device__ __forceinline__ void hg_search(int n, const uint32_t *__restrict__ cell_start,
                                          const uint32_t *__restrict__ occ,
                                          const uint32_t *__restrict__ level_used,
                                          const float4 *__restrict__ boxes, const HGridP &g,
                                          int t0, HGLDS &S, Hits hits) {
    const int lane = threadIdx.x & 63;
    const int own = lane & (HG_OWN - 1), sub = lane / HG_OWN;
    const int t = t0 + own;
    const uint32_t xmask = (uint32_t)g.dims[0] - 1u;
    float4 mn0 = mk4(0, 0, 0, 0), mx0 = mn0;
    uint32_t key = KEY_NONE, next = KEY_NONE;
    if (t < n) {
        mn0 = boxes[2 * (size_t)t];
        mx0 = boxes[2 * (size_t)t + 1];
        key = __float_as_uint(mn0.w);
        if (t + 1 < n) next = __float_as_uint(boxes[2 * (size_t)t + 2].w);
    }
    if (sub == 0) {
        S.mn[own] = mn0;
        S.mx[own] = mx0;
    }
    const int lx = (int)(key >> g.cell_bits), l = lx + sub;
    // per row the cells that hold members within reach (bit dx + 1), three
    // bits a row
    uint32_t rows = 0u;
    int gp[3] = {0, 0, 0};
    if (key != KEY_NONE && l < g.levels && (sub == 0 || level_used[l])) {
        const float inv_l = g.inv_cell0 * exp2f(-(float)l);
        hg_cell(mn0, mx0, inv_l, g.dims, gp);
        const float c = 1.0f / inv_l, h = 0.5f * c;
        // (reachable_cells's rule, an axis at a time and with room for the
        // rounding of far coordinates: a pair is looked for from one side only)
        uint32_t ok[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const float lo = k == 0 ? mn0.x : k == 1 ? mn0.y : mn0.z;
            const float hi = k == 0 ? mx0.x : k == 1 ? mx0.y : mx0.z;
            const float ctr = (lo + hi) * 0.5f, eps = 1e-4f * c + 1e-6f * fabsf(ctr);
            const float f = floorf(ctr * inv_l);
            ok[k] = 0u;
#pragma unroll
            for (int d = -1; d <= 1; d++) {
                const float c0 = (f + (float)d) * c - h - eps;
                const float c1 = (f + (float)(d + 1)) * c + h + eps;
                if (!(hi < c0) && !(lo > c1)) ok[k] |= 1u << (d + 1);
            }
        }
        const uint32_t lk = (uint32_t)l << g.cell_bits, gx = (uint32_t)gp[0];
        uint32_t wl[9], wr[9];
#pragma unroll
        for (int r = 0; r < 9; r++) {
            const uint32_t b = lk | pos_hash(0, gp[1] + r % 3 - 1, gp[2] + r / 3 - 1, g.dims);
            const bool in = ((ok[1] >> (r % 3)) & 1u) && ((ok[2] >> (r / 3)) & 1u) &&
                            (sub > 0 || r >= 4);
            wl[r] = in ? occ[(b | ((gx - 1u) & xmask)) >> 5] : 0u;
            wr[r] = in ? occ[(b | ((gx + 1u) & xmask)) >> 5] : 0u;
        }
#pragma unroll
        for (int r = 0; r < 9; r++) {
            const uint32_t b = lk | pos_hash(0, gp[1] + r % 3 - 1, gp[2] + r / 3 - 1, g.dims);
            uint32_t m = row_bits(wl[r], wr[r], b, (gx - 1u) & xmask, gx, (gx + 1u) & xmask);
            m &= ok[0];
            if (sub == 0 && r == 4) m = (m & 4u) | (next == key ? 2u : 0u);
            rows |= m << (3 * r);
        }
    }
    // the wrapped cell of every row waits for the second round
    const uint32_t wrapped = gp[0] == 0 ? 0111111111u : (uint32_t)gp[0] == xmask ? 0444444444u : 0u;
    uint32_t rest = rows & wrapped;
    rows &= ~wrapped;
    const uint32_t lk = (uint32_t)l << g.cell_bits;
    for (int round = 0; round < 2; round++) {
        uint32_t total = 0;
#pragma unroll
        for (int r = 0; r < 9; r++)
            // (the own row starts after the entry itself)
            list_row(S, total, (rows >> (3 * r)) & 7u,
                     lk | pos_hash(0, gp[1] + r % 3 - 1, gp[2] + r / 3 - 1, g.dims),
                     (uint32_t)gp[0], xmask, own,
                     sub == 0 && r == 4 && round == 0 ? (uint32_t)t + 1u : 0u);
        if (total)
            walk_rows<false>(n, total, cell_start, boxes, S, [&](uint64_t m, int c, int o) {
                hits(m, c, __float_as_int(S.mx[o].w));
                return false;
            });
        rows = rest;
        if (__ballot(rest != 0u) == 0ull) break;
    }
}
// A pair (x, y), x > y, belongs to body x.  The count pass keeps its wave's
// pairs in LDS, counts them and leaves them in the wave's part of rec (HG_REC
// pairs; rec_n[wave] their number, or more when they did not fit) for the
// write pass, which searches again only where they did not fit (slot order
// within a body's range is that of the atomics; k_pairs_group orders it).
__global__ __launch_bounds__(64 * HG_WAVES) void k_hg_count(
    int n, const uint32_t *__restrict__ cell_start, const uint32_t *__restrict__ occ,
    const uint32_t *__restrict__ level_used, const float4 *__restrict__ boxes, HGridP g,
    uint32_t *__restrict__ counts, uint2 *__restrict__ rec, uint32_t *__restrict__ rec_n) {
    __shared__ HGLDS S[HG_WAVES];
    __shared__ uint2 s_rec[HG_WAVES][HG_REC];
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int wave = (int)blockIdx.x * HG_WAVES + w;
    if ((int64_t)wave * HG_OWN >= n) return;
    uint32_t found = 0;
    hg_search(n, cell_start, occ, level_used, boxes, g, wave * HG_OWN, S[w],
              [&](uint64_t m, int c, int y) {
                  if ((m >> lane) & 1ull) {
                      const uint32_t p = __builtin_amdgcn_mbcnt_hi(
                          (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, found));
                      const uint32_t hi = (uint32_t)(c > y ? c : y), lo = (uint32_t)(c > y ? y : c);
                      if (p < (uint32_t)HG_REC) s_rec[w][p] = make_uint2(hi, lo);
                      else atomicAdd(&counts[hi], 1u);
                  }
                  found += (uint32_t)__popcll(m);
              });
    wave_fence();
    const uint32_t kept = found < (uint32_t)HG_REC ? found : (uint32_t)HG_REC;
    for (uint32_t p = lane; p < kept; p += 64) {
        const uint2 e = s_rec[w][p];
        atomicAdd(&counts[e.x], 1u);
        rec[(size_t)wave * HG_REC + p] = e;
    }
    if (lane == 0) rec_n[wave] = found;
}
__global__ __launch_bounds__(64 * HG_WAVES) void k_hg_write(
    int n, const uint32_t *__restrict__ cell_start, const uint32_t *__restrict__ occ,
    const uint32_t *__restrict__ level_used, const float4 *__restrict__ boxes, HGridP g,
    const uint32_t *__restrict__ offsets, uint32_t *__restrict__ cursor, int max_pairs,
    uint32_t *__restrict__ ys, const uint2 *__restrict__ rec,
    const uint32_t *__restrict__ rec_n) {
    __shared__ HGLDS S[HG_WAVES];
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int wave = (int)blockIdx.x * HG_WAVES + w;
    if ((int64_t)wave * HG_OWN >= n) return;
    auto put = [&](uint32_t hi, uint32_t lo) {
        const uint32_t pos = offsets[hi] + atomicAdd(&cursor[hi], 1u);
        if (pos < (uint32_t)max_pairs) ys[pos] = lo;
    };
    const uint32_t found = rec_n[wave];
    if (found <= (uint32_t)HG_REC) {
        for (uint32_t p = lane; p < found; p += 64) {
            const uint2 e = rec[(size_t)wave * HG_REC + p];
            put(e.x, e.y);
        }
        return;
    }
    hg_search(n, cell_start, occ, level_used, boxes, g, wave * HG_OWN, S[w],
              [&](uint64_t m, int c, int y) {
                  if ((m >> lane) & 1ull)
                      put((uint32_t)(c > y ? c : y), (uint32_t)(c > y ? y : c));
              });
}

// The pair range of body x: [offsets[x], offsets[x] + counts[x]) clipped to
// the capacity.
__device__ __forceinline__ uint32_t pair_range(const uint32_t *counts, const uint32_t *offsets,
                                               int max_pairs, int x, uint32_t &off) {
    off = offsets[x];
    uint32_t len = counts[x];
    if (off >= (uint32_t)max_pairs) return 0u;
    if (off + len > (uint32_t)max_pairs) len = (uint32_t)max_pairs - off;
    return len;
}

// Batcher's merge-exchange network of N = 2^k keys, as a table for unrolling.
template <int N>
struct SortNet {
    static constexpr int count() {
        int c = 0;
        for (int p = 1; p < N; p *= 2)
            for (int k = p; k >= 1; k /= 2)
                for (int j = k % p; j + k < N; j += 2 * k)
                    for (int i = 0; i < k && i + j + k < N; i++)
                        if ((i + j) / (2 * p) == (i + j + k) / (2 * p)) c++;
        return c;
    }
    int a[count()], b[count()];
    constexpr SortNet() : a(), b() {
        int c = 0;
        for (int p = 1; p < N; p *= 2)
            for (int k = p; k >= 1; k /= 2)
                for (int j = k % p; j + k < N; j += 2 * k)
                    for (int i = 0; i < k && i + j + k < N; i++)
                        if ((i + j) / (2 * p) == (i + j + k) / (2 * p)) {
                            a[c] = i + j;
                            b[c] = i + j + k;
                            c++;
                        }
    }
};
template <int A, int B, int N>
__device__ __forceinline__ void compare_exchange(uint32_t (&v)[N]) {
    const uint32_t a = v[A], b = v[B];
    v[A] = a < b ? a : b;
    v[B] = a < b ? b : a;
}
template <int N, int... I>
__device__ __forceinline__ void sort_net(uint32_t (&v)[N], std::integer_sequence<int, I...>) {
    constexpr SortNet<N> net;
    (compare_exchange<net.a[I], net.b[I], N>(v), ...);
}
// One thread's range of at most N pairs of body x, ordered by y.
template <int N>
__device__ __forceinline__ void group_range(const uint32_t *__restrict__ ys, uint32_t off,
                                            uint32_t len, int x, int2 *__restrict__ pairs) {
    uint32_t v[N];
#pragma unroll
    for (int k = 0; k < N; k++) v[k] = (uint32_t)k < len ? ys[off + k] : 0xffffffffu;
    sort_net<N>(v, std::make_integer_sequence<int, SortNet<N>::count()>{});
#pragma unroll
    for (int k = 0; k < N; k++)
        if ((uint32_t)k < len) pairs[off + k] = make_int2(x, (int)v[k]);
}
constexpr int GROUP_SMALL = 32;

// One thread per body: its range sorted by y in registers (a network of 8, 16
// or 32 keys, by the longest range of the wave) and written as int2 (x, y).
// Longer ranges go to a list for k_pairs_group_big (from the front of big[]),
// those longer than huge_min to one for k_pairs_group_huge (from the back).
// Also the pair count and the capacity flag.  (With ranges of 9 and more left
// to a workgroup each, a third of the bodies of a layered scene of 65,537: 12
// us here and 37 there, against 7 and 5; 1M boxes on the grid: 23 -> 10 us.)
__global__ __launch_bounds__(256) void k_pairs_group(int n, const uint32_t *__restrict__ counts,
                                                     const uint32_t *__restrict__ offsets,
                                                     const uint32_t *__restrict__ total,
                                                     int max_pairs, const uint32_t *__restrict__ ys,
                                                     int2 *__restrict__ pairs, int *num_pairs,
                                                     int *overflow, uint32_t *__restrict__ big,
                                                     uint32_t *__restrict__ big_n, int huge_min) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x == 0) {
        uint32_t tt = *total;
        if (tt > (uint32_t)max_pairs) atomicOr(overflow, (int)MI_RB_OVERFLOW_PAIRS);
        *num_pairs = (int)(tt < (uint32_t)max_pairs ? tt : (uint32_t)max_pairs);
    }
    if (x >= n) return;
    uint32_t off;
    const uint32_t len = pair_range(counts, offsets, max_pairs, x, off);
    if (len == 0) return;
    if (len > (uint32_t)huge_min) {
        big[n - 1 - (int)atomicAdd(big_n + 1, 1u)] = (uint32_t)x;  // from the back
        return;
    }
    if (len > (uint32_t)GROUP_SMALL) {
        big[atomicAdd(big_n, 1u)] = (uint32_t)x;
        return;
    }
    if (!__ballot(len > 8u)) group_range<8>(ys, off, len, x, pairs);
    else if (!__ballot(len > 16u)) group_range<16>(ys, off, len, x, pairs);
    else group_range<32>(ys, off, len, x, pairs);
}

// Bodies with more than GROUP_SMALL pairs, one workgroup each: the rank of
// every y among its range (the y of one body are distinct) in LDS chunks.
constexpr int GROUP_CHUNK = 1024;
__global__ __launch_bounds__(256) void k_pairs_group_big(const uint32_t *__restrict__ counts,
                                                         const uint32_t *__restrict__ offsets,
                                                         int max_pairs,
                                                         const uint32_t *__restrict__ ys,
                                                         int2 *__restrict__ pairs,
                                                         const uint32_t *__restrict__ big,
                                                         const uint32_t *__restrict__ big_n) {
    __shared__ uint32_t sy[GROUP_CHUNK];
    const uint32_t nb = *big_n;
    for (uint32_t b = blockIdx.x; b < nb; b += gridDim.x) {
        const int x = (int)big[b];
        uint32_t off;
        const uint32_t len = pair_range(counts, offsets, max_pairs, x, off);
        for (uint32_t i0 = 0; i0 < len; i0 += 256) {
            const uint32_t i = i0 + threadIdx.x;
            const uint32_t yi = i < len ? ys[off + i] : 0u;
            uint32_t rank = 0;
            for (uint32_t j0 = 0; j0 < len; j0 += GROUP_CHUNK) {
                const uint32_t m = len - j0 < (uint32_t)GROUP_CHUNK ? len - j0 : GROUP_CHUNK;
                __syncthreads();
                for (uint32_t j = threadIdx.x; j < m; j += 256) sy[j] = ys[off + j0 + j];
                __syncthreads();
                for (uint32_t j = 0; j < m; j++) rank += sy[j] < yi ? 1u : 0u;
            }
            if (i < len) pairs[off + rank] = make_int2(x, (int)yi);
        }
    }
}

// Bodies with more than huge_min pairs (a ground touching thousands of
// bodies), one workgroup each: the y of the range are distinct indices below
// x, so one bit per index in LDS (cleared, set), per-thread chunk counts and
// their prefix give every y its rank.  Dynamic LDS: (n + 31) / 32 words.
constexpr int HUGE_BLOCK = 1024;
__global__ __launch_bounds__(HUGE_BLOCK) void k_pairs_group_huge(
    int n, const uint32_t *__restrict__ counts, const uint32_t *__restrict__ offsets,
    int max_pairs, const uint32_t *__restrict__ ys, int2 *__restrict__ pairs,
    const uint32_t *__restrict__ big, const uint32_t *__restrict__ big_n) {
    extern __shared__ uint32_t bm[];
    __shared__ uint32_t cbase[HUGE_BLOCK];
    const int tid = threadIdx.x;
    const uint32_t nh = big_n[1];
    for (uint32_t b = blockIdx.x; b < nh; b += gridDim.x) {
        const int x = (int)big[n - 1 - (int)b];
        uint32_t off;
        const uint32_t len = pair_range(counts, offsets, max_pairs, x, off);
        const int W = (x + 31) >> 5;
        const int chunk = (W + HUGE_BLOCK - 1) / HUGE_BLOCK;
        __syncthreads();
        for (int w = tid; w < W; w += HUGE_BLOCK) bm[w] = 0u;
        __syncthreads();
        for (uint32_t i = tid; i < len; i += HUGE_BLOCK) {
            const uint32_t y = ys[off + i];
            atomicOr(&bm[y >> 5], 1u << (y & 31u));
        }
        __syncthreads();
        uint32_t c = 0;
        for (int w = tid * chunk; w < (tid + 1) * chunk && w < W; w++) c += __popc(bm[w]);
        cbase[tid] = c;
        __syncthreads();
        // exclusive prefix of the chunk counts (Hillis-Steele in place)
        for (int o = 1; o < HUGE_BLOCK; o <<= 1) {
            const uint32_t v = tid >= o ? cbase[tid - o] : 0u;
            __syncthreads();
            cbase[tid] += v;
            __syncthreads();
        }
        const uint32_t excl = cbase[tid] - c;
        __syncthreads();
        cbase[tid] = excl;
        __syncthreads();
        for (uint32_t i = tid; i < len; i += HUGE_BLOCK) {
            const uint32_t y = ys[off + i];
            const int w = (int)(y >> 5), ck = w / chunk;
            uint32_t r = cbase[ck];
            for (int k = ck * chunk; k < w; k++) r += __popc(bm[k]);
            r += __popc(bm[w] & ((1u << (y & 31u)) - 1u));
            pairs[off + r] = make_int2(x, (int)y);
        }
    }
}

// ---- sweep and prune (btGpuSapBroadphase::calculateOverlappingPairs,
// opencl/gpu_rigidbody_pipeline2/btGpuSapBroadphase.cpp:91-434; kernels
// opencl/broadphase_benchmark/sap.cl:90-116, 290-320) ----

// order-preserving map of a float to uint32 (sap.cl FloatFlip: negative
// values have every bit flipped, others only the sign bit)
__device__ __forceinline__ uint32_t float_flip(float f) {
    const uint32_t u = __float_as_uint(f);
    return u ^ ((uint32_t)(-(int32_t)(u >> 31)) | 0x80000000u);
}
__device__ __forceinline__ float axis_of4(float4 v, int axis) {
    return axis == 0 ? v.x : (axis == 1 ? v.y : v.z);
}

// (FloatFlip(min[axis]), index) per AABB; large AABBs (is_large[i] != 0)
// sort last and go to a list of their own (lg, count lg_n, zero at launch).
// Zeroes the per-body pair counts.
__global__ __launch_bounds__(256) void k_sap_keys(const float4 *__restrict__ mn,
                                                  const int *__restrict__ is_large, int n, int axis,
                                                  uint2 *__restrict__ kv,
                                                  uint32_t *__restrict__ counts,
                                                  uint32_t *__restrict__ cursor,
                                                  uint32_t *__restrict__ big_n,
                                                  uint32_t *__restrict__ lg,
                                                  uint32_t *__restrict__ lg_n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) { big_n[0] = 0u; big_n[1] = 0u; }
    if (i >= n) return;
    const bool large = is_large && is_large[i] != 0;
    kv[i] = make_uint2(large ? 0xffffffffu : float_flip(axis_of4(mn[i], axis)), (uint32_t)i);
    if (large) lg[atomicAdd(lg_n, 1u)] = (uint32_t)i;
    counts[i] = 0u;
    cursor[i] = 0u;
}

// Pairs of the large AABBs (sap2Kernel's role, btGpuSapBroadphase.cpp:311-333):
// one thread per sorted AABB j tests it against every large AABB L; a pair
// of two large AABBs is taken by the one of lower index only.
template <int WRITE>
__global__ __launch_bounds__(256) void k_sap_large(int n, const float4 *__restrict__ mn,
                                                   const float4 *__restrict__ mx,
                                                   const float4 *__restrict__ smn,
                                                   const float4 *__restrict__ smx,
                                                   const uint32_t *__restrict__ lg,
                                                   const uint32_t *__restrict__ lg_n,
                                                   uint32_t *__restrict__ counts,
                                                   const uint32_t *__restrict__ offsets,
                                                   uint32_t *__restrict__ cursor, int max_pairs,
                                                   uint32_t *__restrict__ ys) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const int nl = (int)*lg_n;
    if (nl == 0) return;
    const int ns = n - nl;
    const float4 bmn = smn[j], bmx = smx[j];
    const int y = __float_as_int(bmn.w);
    for (int q = 0; q < nl; q++) {
        const int L = (int)lg[q];
        if (L == y || (j >= ns && y > L)) continue;
        if (!aabb_overlap(mn[L], mx[L], bmn, bmx)) continue;
        // (lanes whose pair belongs to L, all of them for a last ground, take
        // their places with one atomic per wave: 51 -> 13 us at 65,537 AABBs)
        const uint64_t own = __ballot(L > y);
        if (L > y) {
            const uint32_t rank = (uint32_t)__popcll(own & lanemask_lt()), m = (uint32_t)__popcll(own);
            uint32_t first = 0;
            if (rank == 0) first = atomicAdd(WRITE ? &cursor[L] : &counts[L], m);
            if (WRITE) {
                first = __shfl(first, __ffsll((long long)own) - 1);
                const uint32_t pos = offsets[L] + first + rank;
                if (pos < (uint32_t)max_pairs) ys[pos] = (uint32_t)y;
            }
        } else if (!WRITE) {
            atomicAdd(&counts[y], 1u);
        } else {
            const uint32_t pos = offsets[y] + atomicAdd(&cursor[y], 1u);
            if (pos < (uint32_t)max_pairs) ys[pos] = (uint32_t)L;
        }
    }
}

// AABBs in sorted order, the original index in min.w (as int bits)
__global__ __launch_bounds__(256) void k_sap_scatter(const uint2 *__restrict__ kv, int n,
                                                     const float4 *__restrict__ mn,
                                                     const float4 *__restrict__ mx,
                                                     float4 *__restrict__ smn,
                                                     float4 *__restrict__ smx) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t k = kv[i].y;
    float4 a = mn[k];
    a.w = __int_as_float((int)k);
    smn[i] = a;
    smx[i] = mx[k];
}

// The sweep over the sorted small AABBs (computePairsKernelOriginal): the
// pairs (i, j), i before j, that overlap on all three axes.  A wave owns 8
// consecutive AABBs, whose bounds it holds in scalar registers, and walks the
// candidates after them 64 at a time, one per lane: every compare tests 64
// pairs, and a candidate's load serves 8 of them.  It stops where the
// candidates' min passes the largest max of the 8 (no later j overlaps: the
// mins are sorted).  Bound by the compares and the pair counts' atomics.
// 65,537 AABBs in a layer, 470,000 pairs: 77 us to find and count, 27 to write.
// (One thread per AABB, each walking its own candidates, twice: 884 + 871 us at
// 65,537 AABBs in a layer; 64 owners in lanes and the candidates through the
// scalar cache, which a window of 60 KB does not fit: 97 us.)
constexpr int SAP_OWN = 8, SAP_BLOCK_OWN = 4 * SAP_OWN;
// hits(m, c, y): the lanes of m[k] hold a candidate (body c) that overlaps
// owner k (body y[k])
template <class Hits>
__device__ __forceinline__ void sap_sweep(int ns, int axis, const float4 *__restrict__ smn,
                                          const float4 *__restrict__ smx, Hits hits) {
    const int lane = threadIdx.x & 63;
    const int i0 = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * SAP_BLOCK_OWN +
                                                        (threadIdx.x >> 6) * SAP_OWN));
    if (i0 >= ns) return;
    float4 amn[SAP_OWN], amx[SAP_OWN];
    int y[SAP_OWN];
    float lim = -INFINITY;
#pragma unroll
    for (int k = 0; k < SAP_OWN; k++) {
        const int i = i0 + k < ns ? i0 + k : ns - 1;
        amn[k] = smn[i];
        amx[k] = smx[i];
        y[k] = __float_as_int(amn[k].w);
        lim = fmaxf(lim, axis_of4(amx[k], axis));
    }
    // (a lane past the end overlaps nothing: NaN)
    auto fetch = [&](int j, float4 &mn, float4 &mx) {
        mn = mx = mk4(NAN, NAN, NAN, 0.f);
        if (j < ns) {
            mn = smn[j];
            mx = smx[j];
        }
    };
    float4 bmn, bmx, nmn, nmx;
    fetch(i0 + 1 + lane, nmn, nmx);
    for (int j0 = i0 + 1; j0 < ns; j0 += 64) {
        bmn = nmn;
        bmx = nmx;
        if (__builtin_amdgcn_readfirstlane((int)(axis_of4(bmn, axis) > lim))) break;
        fetch(j0 + 64 + lane, nmn, nmx);
        uint64_t m[SAP_OWN], any = 0;
#pragma unroll
        for (int k = 0; k < SAP_OWN; k++) {
            m[k] = __ballot((amn[k].x <= bmx.x) & (bmn.x <= amx[k].x) & (amn[k].y <= bmx.y) &
                            (bmn.y <= amx[k].y) & (amn[k].z <= bmx.z) & (bmn.z <= amx[k].z));
            // (the first candidates are the owners themselves: those after k)
            if (j0 == i0 + 1) m[k] &= ~0ull << k;
            if (i0 + k >= ns) m[k] = 0ull;
            any |= m[k];
        }
        if (any) hits(m, __float_as_int(bmn.w), y);
    }
}
// A pair (x, y), x > y, belongs to body x.  The count pass keeps the pairs of
// its workgroup in LDS, counts them and leaves them in the workgroup's part of
// rec (SAP_REC pairs; rec_n[block] their number, or more when they did not
// fit) for the write pass, which sweeps again only where they did not fit.
constexpr int SAP_REC = RB_SAP_REC;
__global__ __launch_bounds__(256) void k_sap_count(int n, int axis, const float4 *__restrict__ smn,
                                                   const float4 *__restrict__ smx,
                                                   const uint32_t *__restrict__ lg_n,
                                                   uint32_t *__restrict__ counts,
                                                   uint2 *__restrict__ rec,
                                                   uint32_t *__restrict__ rec_n) {
    __shared__ uint2 s_rec[SAP_REC];
    __shared__ uint32_t s_n;
    n -= (int)*lg_n;  // the large AABBs sorted last do not sweep
    if (threadIdx.x == 0) s_n = 0u;
    __syncthreads();
    const uint64_t me = 1ull << (threadIdx.x & 63);
    sap_sweep(n, axis, smn, smx, [&](const uint64_t *m, int c, const int *y) {
        uint32_t total = 0, first = 0;
#pragma unroll
        for (int k = 0; k < SAP_OWN; k++) total += (uint32_t)__popcll(m[k]);
        if (me == 1ull) first = atomicAdd(&s_n, total);
        first = (uint32_t)__builtin_amdgcn_readfirstlane((int)first);
#pragma unroll
        for (int k = 0; k < SAP_OWN; k++) {
            if (m[k] == 0ull) continue;
            if (m[k] & me) {
                const uint32_t p = __builtin_amdgcn_mbcnt_hi(
                    (uint32_t)(m[k] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m[k], first));
                const uint32_t hi = (uint32_t)(c > y[k] ? c : y[k]),
                               lo = (uint32_t)(c > y[k] ? y[k] : c);
                if (p < (uint32_t)SAP_REC) s_rec[p] = make_uint2(hi, lo);
                else atomicAdd(&counts[hi], 1u);
            }
            first += (uint32_t)__popcll(m[k]);
        }
    });
    __syncthreads();
    const uint32_t kept = s_n < (uint32_t)SAP_REC ? s_n : (uint32_t)SAP_REC;
    for (uint32_t p = threadIdx.x; p < kept; p += 256) {
        const uint2 e = s_rec[p];
        atomicAdd(&counts[e.x], 1u);
        rec[(size_t)blockIdx.x * SAP_REC + p] = e;
    }
    if (threadIdx.x == 0) rec_n[blockIdx.x] = s_n;
}
__global__ __launch_bounds__(256) void k_sap_write(int n, int axis, const float4 *__restrict__ smn,
                                                   const float4 *__restrict__ smx,
                                                   const uint32_t *__restrict__ lg_n,
                                                   const uint32_t *__restrict__ offsets,
                                                   uint32_t *__restrict__ cursor, int max_pairs,
                                                   uint32_t *__restrict__ ys,
                                                   const uint2 *__restrict__ rec,
                                                   const uint32_t *__restrict__ rec_n) {
    auto put = [&](uint32_t hi, uint32_t lo) {
        const uint32_t pos = offsets[hi] + atomicAdd(&cursor[hi], 1u);
        if (pos < (uint32_t)max_pairs) ys[pos] = lo;
    };
    const uint32_t found = rec_n[blockIdx.x];
    if (found <= (uint32_t)SAP_REC) {
        for (uint32_t p = threadIdx.x; p < found; p += 256) {
            const uint2 e = rec[(size_t)blockIdx.x * SAP_REC + p];
            put(e.x, e.y);
        }
        return;
    }
    n -= (int)*lg_n;
    const uint64_t me = 1ull << (threadIdx.x & 63);
    sap_sweep(n, axis, smn, smx, [&](const uint64_t *m, int c, const int *y) {
#pragma unroll
        for (int k = 0; k < SAP_OWN; k++)
            if (m[k] & me) put((uint32_t)(c > y[k] ? c : y[k]), (uint32_t)(c > y[k] ? y[k] : c));
    });
}

}  // namespace

// ---------------------------------------------------------------- launchers
static GridP grid_of(const StepParams &p) {
    GridP g;
    g.inv_cell = p.inv_cell;
    g.dims[0] = p.dims[0];
    g.dims[1] = p.dims[1];
    g.dims[2] = p.dims[2];
    g.cell_bits = p.cell_bits;
    return g;
}

hipError_t launch_setup(const DeviceWorld &d, const StepParams &p, hipStream_t s) {
    if (p.n_bodies == 0) return hipSuccess;
    RB_LAUNCH(k_setup, dim3((p.n_bodies + 255) / 256), dim3(256), 0, s, p.n_bodies,
                       d.pos, d.quat, d.linvel, d.angvel, d.inv_mass, d.shape, d.scene, d.is_large,
                       d.hulls, d.inv_inertia_local, d.inv_inertia_world, d.aabb_min, d.aabb_max,
                       d.kv, grid_of(p), p.gravity[0], p.gravity[1], p.gravity[2], p.dt,
                       d.occ, d.occ_words);
    return rb_launch_status();
}

hipError_t launch_cell_start(const DeviceWorld &d, const StepParams &p, hipStream_t s) {
    const int n = p.n_bodies;
    if (n == 0) return hipSuccess;
    RB_LAUNCH(k_cell_start, dim3((n + 255) / 256), dim3(256), 0, s, d.kv, n, d.aabb_min,
                       d.aabb_max, d.cell_start, d.occ, d.boxes);
    return rb_launch_status();
}

hipError_t launch_find_pairs(const DeviceWorld &d, const StepParams &p, hipStream_t s) {
    int n = p.n_bodies;
    if (n == 0) return hipSuccess;
    int K = p.max_pairs_per_body;
    auto find = [&](auto kern, int own) {
        const int entries = FP_WAVES * own;
        RB_LAUNCH(kern, dim3((n + entries - 1) / entries), dim3(64 * FP_WAVES), 0, s, n,
                  d.cell_start, d.occ, d.boxes, d.aabb_min, d.aabb_max, d.large_list,
                  p.n_large ? d.large_first : nullptr, p.n_large ? d.large_num : nullptr,
                  grid_of(p), K, d.body_slots, d.pair_count, d.counters + RB_CNT_OVERFLOW);
    };
    if (n < FP_TWO) find(k_find_pairs<2>, 2);
    else if (n < FP_FOUR) find(k_find_pairs<4>, 4);
    else find(k_find_pairs<16>, 16);
    if (p.n_large > 0) {
        dim3 g(p.n_large, p.large_chunks);
        RB_LAUNCH(k_large_count, g, dim3(256), 0, s, d.large_list, d.scene,
                           d.scene_start, d.aabb_min, d.aabb_max, p.large_chunks, d.large_chunk_cnt);
        RB_LAUNCH(k_large_write, g, dim3(256), 0, s, d.large_list, d.large_off, d.scene,
                           d.scene_start, d.aabb_min, d.aabb_max, p.large_chunks,
                           d.large_chunk_cnt, d.large_slots, d.pair_count);
    }
    return rb_launch_status();
}

hipError_t launch_emit_pairs(const DeviceWorld &d, const StepParams &p, hipStream_t s) {
    int n = p.n_bodies;
    if (n == 0) return hipSuccess;
    const int body_blocks = (int)(((int64_t)n * EMIT_LANES + 255) / 256);
    const int large_blocks = std::max(1, std::min(32, p.max_scene / 256));
    RB_LAUNCH(k_emit_pairs, dim3(body_blocks + p.n_large * large_blocks), dim3(256), 0, s, n,
              body_blocks, large_blocks, d.pair_count, d.pair_off, d.body_slots, p.max_pairs_per_body,
              d.is_large, d.large_list, d.large_off, d.large_slots, p.max_pairs, d.pairs,
              (const uint32_t *)(d.counters + RB_CNT_SORT_TILE), d.counters + RB_CNT_PAIRS,
              d.counters + RB_CNT_OVERFLOW);
    return rb_launch_status();
}

// Each body's pair range ordered by y: ranges of up to GROUP_SMALL pairs in
// registers, up to HUGE_MIN by rank in LDS chunks, longer ones (a ground)
// through an LDS bitmap of the indices below the body when it fits.
constexpr int HUGE_MIN = 4096;
constexpr size_t HUGE_LDS_MAX = 60 * 1024;
static void launch_pairs_group(int n, uint32_t *counts, uint32_t *offsets, uint32_t *total,
                               int max_pairs, uint32_t *ys, int2 *pairs, int *num_pairs,
                               int *overflow, uint32_t *big, uint32_t *big_n, int blocks,
                               hipStream_t s) {
    const size_t bm_bytes = sizeof(uint32_t) * (((size_t)n + 31) / 32 + 1);
    const bool huge = bm_bytes <= HUGE_LDS_MAX;
    RB_LAUNCH(k_pairs_group, dim3(blocks), dim3(256), 0, s, n, counts, offsets, total,
                       max_pairs, ys, pairs, num_pairs, overflow, big, big_n,
                       huge ? HUGE_MIN : INT_MAX);
    if (n > 0) {
        RB_LAUNCH(k_pairs_group_big, dim3(1024), dim3(256), 0, s, counts, offsets,
                           max_pairs, ys, pairs, big, big_n);
        if (huge)
            RB_LAUNCH(k_pairs_group_huge, dim3(64), dim3(HUGE_BLOCK), bm_bytes, s, n,
                               counts, offsets, max_pairs, ys, pairs, big, big_n);
    }
}

// Hierarchical-grid pair search of n AABBs: hash, sort, cell starts, count
// per body, scan, write, then each body's pairs ordered by y.
hipError_t launch_hgrid_pairs(const float4 *mn, const float4 *mx, int n, float inv_cell0,
                              const int dims[3], int cell_bits, int levels, uint2 *kv,
                              uint32_t *cell_start, uint32_t *occ, float4 *boxes,
                              uint32_t *counts, uint32_t *offsets, uint32_t *cursor,
                              uint32_t *big, uint32_t *total, uint32_t *ys, int max_pairs,
                              int2 *pairs, int *num_pairs, int *overflow, const SortWork &sw,
                              uint32_t *scan_status, hipStream_t s, hipEvent_t *ev, uint2 *rec,
                              uint32_t *rec_n) {
    HGridP g;
    g.inv_cell0 = inv_cell0;
    g.dims[0] = dims[0]; g.dims[1] = dims[1]; g.dims[2] = dims[2];
    g.cell_bits = cell_bits;
    g.levels = levels;
    const int blocks = n > 0 ? (n + 255) / 256 : 1;
    const int hg_blocks = (n + HG_WAVES * HG_OWN - 1) / (HG_WAVES * HG_OWN);
    uint32_t *big_n = big + (n > 0 ? n : 0);
    // (the boxes as given, two float4 each: k_hg_cells has read them before the
    // count pass fills rec)
    static_assert(RB_HG_REC * sizeof(uint2) >= RB_HG_OWN * 2 * sizeof(float4));
    float4 *raw = (float4 *)rec;
    if (ev) hipEventRecord(ev[0], s);
    RB_LAUNCH(k_hg_hash, dim3(blocks), dim3(256), 0, s, mn, mx, n, g, kv, counts, cursor,
                       big_n, overflow, raw);
    if (ev) hipEventRecord(ev[1], s);
    hipError_t e = launch_radix_sort(kv, n, cell_bits + 2, 8, sw, s);
    if (e != hipSuccess) return e;
    if (ev) hipEventRecord(ev[2], s);
    // occupancy words of every level's cells, then one flag per level
    const size_t occ_words = ((size_t)1 << (cell_bits + 2)) / 32;
    uint32_t *level_used = occ + occ_words;
    if (n > 0) {
        e = launch_fill_u32(occ, 0u, occ_words + 4, s);
        if (e != hipSuccess) return e;
        RB_LAUNCH(k_hg_cells, dim3(blocks), dim3(256), 0, s, kv, n, raw, g, cell_start, occ,
                  level_used, boxes);
        RB_LAUNCH(k_hg_count, dim3(hg_blocks), dim3(64 * HG_WAVES), 0, s, n, cell_start, occ,
                  level_used, boxes, g, counts, rec, rec_n);
    }
    e = launch_exclusive_scan(counts, offsets, n, total, scan_status, s, nullptr, overflow);
    if (e != hipSuccess) return e;
    if (n > 0)
        RB_LAUNCH(k_hg_write, dim3(hg_blocks), dim3(64 * HG_WAVES), 0, s, n, cell_start, occ,
                  level_used, boxes, g, offsets, cursor, max_pairs, ys, rec, rec_n);
    if (ev) hipEventRecord(ev[3], s);
    launch_pairs_group(n, counts, offsets, total, max_pairs, ys, pairs, num_pairs, overflow, big,
                       big_n, blocks, s);
    if (ev) hipEventRecord(ev[4], s);
    return rb_launch_status();
}

// Sweep and prune of n AABBs along `axis`: keys, 32-bit sort, scatter, count
// per body, scan, write, then each body's pairs ordered by y (as the grid).
hipError_t launch_sap_pairs(const float4 *mn, const float4 *mx, const int *is_large, int n,
                            int axis, uint2 *kv, float4 *smn, float4 *smx, uint32_t *counts,
                            uint32_t *offsets, uint32_t *cursor, uint32_t *big, uint32_t *lg,
                            uint32_t *total, uint32_t *ys, int max_pairs, int2 *pairs,
                            int *num_pairs, int *overflow, const SortWork &sw,
                            uint32_t *scan_status, hipStream_t s, hipEvent_t *ev, uint2 *rec,
                            uint32_t *rec_n) {
    const int blocks = n > 0 ? (n + 255) / 256 : 1;
    const int sweeps = (n + SAP_BLOCK_OWN - 1) / SAP_BLOCK_OWN;
    uint32_t *big_n = big + (n > 0 ? n : 0);
    uint32_t *lg_n = lg + (n > 0 ? n : 0);
    if (ev) hipEventRecord(ev[0], s);
    hipError_t e = launch_fill_u32(lg_n, 0u, 1, s);
    if (e != hipSuccess) return e;
    RB_LAUNCH(k_sap_keys, dim3(blocks), dim3(256), 0, s, mn, is_large, n, axis, kv, counts,
                       cursor, big_n, lg, lg_n);
    if (ev) hipEventRecord(ev[1], s);
    e = launch_radix_sort(kv, n, 32, 8, sw, s);
    if (e != hipSuccess) return e;
    if (ev) hipEventRecord(ev[2], s);
    if (n > 0) {
        RB_LAUNCH(k_sap_scatter, dim3(blocks), dim3(256), 0, s, kv, n, mn, mx, smn, smx);
        RB_LAUNCH(k_sap_count, dim3(sweeps), dim3(256), 0, s, n, axis, smn, smx, lg_n, counts,
                  rec, rec_n);
        RB_LAUNCH(k_sap_large<0>, dim3(blocks), dim3(256), 0, s, n, mn, mx, smn, smx, lg,
                           lg_n, counts, (const uint32_t *)nullptr, cursor, max_pairs, ys);
    }
    e = launch_exclusive_scan(counts, offsets, n, total, scan_status, s, nullptr, overflow);
    if (e != hipSuccess) return e;
    if (n > 0) {
        RB_LAUNCH(k_sap_write, dim3(sweeps), dim3(256), 0, s, n, axis, smn, smx, lg_n, offsets,
                  cursor, max_pairs, ys, rec, rec_n);
        RB_LAUNCH(k_sap_large<1>, dim3(blocks), dim3(256), 0, s, n, mn, mx, smn, smx, lg,
                           lg_n, counts, offsets, cursor, max_pairs, ys);
    }
    if (ev) hipEventRecord(ev[3], s);
    launch_pairs_group(n, counts, offsets, total, max_pairs, ys, pairs, num_pairs, overflow, big,
                       big_n, blocks, s);
    if (ev) hipEventRecord(ev[4], s);
    return rb_launch_status();
}
