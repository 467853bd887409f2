// k_solver.hip -- contact constraints, tile colouring, batched Gauss-Seidel
// solve and integration for gfx950.
//
// Constraint maths follows the reference solver:
//   setConstraint4      dynamics/basic_demo/Stubs/solverSetup.cl:520-610
//   solveContact        solveContact.cl:272-312 (normal rows, lambda >= 0)
//   solveFriction       solveFriction.cl:297-430 (2 tangents at the centre,
//                       |lambda| <= mu * sum lambda_n, angular damping)
//   integrateTransformsKernel2 + copyVelocitiesKernel
//                       opencl/broadphase_benchmark/integrateKernel.cl:102-158,
//                       broadphaseKernel.cl:216-233
// The schedule replaces the reference's 16x16 solver cells with 4 parity
// launches per iteration and the nondeterministic CreateBatches
// (batchingKernels.cl:130-341): constraints are grouped into tiles (one scene
// each, or XZ columns of a single large scene), each tile is coloured in LDS so
// that no dynamic body repeats within a colour, and one workgroup walks its
// tile's colours with barriers between them, keeping the tile's body velocities
// in LDS.  Spatial tiles are run in 4 phases (tile x and z parity) per sweep
// so that tiles sharing bodies never run together; scene tiles are independent
// and run every sweep in one launch.  An optional warm start applies the
// previous step's (or a learned prediction of the) impulses before the sweeps.
#include <float.h>
#include <hip/hip_runtime.h>

#include <type_traits>

#include "dmath.h"
#include "rb_internal.h"

using namespace rb;

namespace {

constexpr int TB = 256;        // threads per tile workgroup (colouring, packing)
constexpr int HASH_SLOTS = 2 * RB_TILE_MAX_BODIES;

__device__ __forceinline__ uint32_t color_prio(uint32_t k) {
    k ^= k >> 16; k *= 0x7feb352dU; k ^= k >> 15; k *= 0x846ca68bU; k ^= k >> 16;
    return k;
}

__device__ __forceinline__ float jac_coeff(float4 a0, float4 a1, float imA, const float4 *IA,
                                           float imB, const float4 *IB) {
    float j0 = imA, j1 = dot3(mt_mul3(a0, IA), a0), j2 = imB, j3 = dot3(mt_mul3(a1, IB), a1);
    return -1.f / (((j0 + j1) + j2) + j3);
}
__device__ __forceinline__ float rel_vel(float4 l0, float4 l1, float4 a0, float4 a1, float4 vA,
                                         float4 wA, float4 vB, float4 wB) {
    return ((dot3(l0, vA) + dot3(a0, wA)) + dot3(l1, vB)) + dot3(a1, wB);
}
// (btPlaneSpace1, both cases by selects: one square root and one division for
// the whole wave, and nothing for the compiler to put into scratch)
__device__ __forceinline__ void plane_space(float4 n, float4 &p, float4 &q) {
    const bool z = fabsf(n.z) > 0.70710678f;
    const float yy = n.y * n.y;
    const float a = z ? yy + n.z * n.z : n.x * n.x + yy;
    const float k = 1.f / sqrtf(a), ak = a * k;
    const float pz = n.y * k, py = z ? -n.z * k : n.x * k;
    p = mk4(z ? 0.f : -n.y * k, py, z ? pz : 0.f, 0.f);
    q = mk4(z ? ak : -n.z * py, z ? -n.x * pz : n.z * p.x, z ? n.x * py : ak, 0.f);
}

// Tile coordinates of a point (clamped, so neighbours stay neighbours).
__device__ __forceinline__ int2 tile_xz(float x, float z, const StepParams &sp) {
    int tx = (int)floorf((x - sp.tile_origin_x) * sp.tile_inv);
    int tz = (int)floorf((z - sp.tile_origin_z) * sp.tile_inv);
    tx = tx < 0 ? 0 : (tx >= sp.tiles_x ? sp.tiles_x - 1 : tx);
    tz = tz < 0 ? 0 : (tz >= sp.tiles_z ? sp.tiles_z - 1 : tz);
    return make_int2(tx, tz);
}

// ---- compaction of the pair slots + ContactToConstraintKernel ----
// One thread per contact, from the list of pairs that have one (a thread per
// pair, of which one in six had a contact, took 226 us against 102 at 553k
// contacts of 3.4M pairs, 37.5 against 16.0 at 60k of 635k).  Bound by its reads and writes, 500 B a contact.
__global__ __launch_bounds__(256) void k_constraints(
    StepParams sp, const uint32_t *__restrict__ contact_pair, const Contact4 *__restrict__ slots,
    Contact4 *__restrict__ contacts, const float4 *__restrict__ pos,
    const float4 *__restrict__ linvel, const float4 *__restrict__ angvel,
    const float *__restrict__ inv_mass, const float4 *__restrict__ invI, const int *__restrict__ scene,
    const float4 *__restrict__ aabb_min, const float4 *__restrict__ aabb_max, ConstraintSoA cs,
    uint2 *__restrict__ tile_kv, int *counters, const int2 *__restrict__ prev_keys,
    const float4 *__restrict__ prev_imp, const float4 *__restrict__ prev_pts,
    const int *__restrict__ prev_count, float *__restrict__ features, int *__restrict__ solve_pos,
    const int2 *__restrict__ pairs) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    // the contact count for the later kernels: the compaction's total, capped
    // at the capacity (no kernel of this launch reads it)
    const uint32_t total = (uint32_t)counters[RB_CNT_CONTACT_TOTAL];
    const uint32_t nc = total < (uint32_t)sp.max_contacts ? total : (uint32_t)sp.max_contacts;
    if (k == 0) {
        counters[RB_CNT_CONTACTS] = (int)nc;
        if (nc < total) atomicOr(counters + RB_CNT_OVERFLOW, (int)MI_RB_OVERFLOW_CONTACTS);
    }
    if (k >= (int)nc) return;
    const int p = (int)contact_pair[k];
    Contact4 src = slots[p];
    contacts[k] = src;
    int a = abs(src.body_a), b = abs(src.body_b);
    float4 pA = pos[a], pB = pos[b];
    float4 vA = linvel[a], wA = angvel[a], vB = linvel[b], wB = angvel[b];
    float imA = inv_mass[a], imB = inv_mass[b];
    float4 IA[3] = {invI[3 * a], invI[3 * a + 1], invI[3 * a + 2]};
    float4 IB[3] = {invI[3 * b], invI[3 * b + 1], invI[3 * b + 2]};
    // static bodies: zero velocity and inverse inertia (setupBodiesKernel)
    if (imA == 0.f) { vA = mk4(0, 0, 0, 0); wA = vA; }
    if (imB == 0.f) { vB = mk4(0, 0, 0, 0); wB = vB; }
    float dt_inv = 1.f / sp.solver_dt;
    float4 n = src.normal;
    float npts = n.w;
    cs.linear[k] = mk4(-n.x, -n.y, -n.z, sp.friction);
    // (the loops over the 4 points are unrolled so that the point arrays and
    // the contact stay in registers)
    float jac[4], bb[4];
#pragma unroll
    for (int ic = 0; ic < 4; ic++) {
        float4 wp = src.pos[ic];
        float4 r0 = sub4(wp, pA), r1 = sub4(wp, pB);
        if ((float)ic >= npts) { jac[ic] = 0.f; bb[ic] = 0.f; continue; }
        float4 lin = neg4(n);
        float4 a0 = neg4(cross3(r0, n));
        float4 a1 = cross3(r1, n);
        jac[ic] = jac_coeff(a0, a1, imA, IA, imB, IB);
        float rv = rel_vel(lin, neg4(lin), a0, a1, vA, wA, vB, wB);
        float e = 0.f;
        float bv = e * rv;
        bv += ((wp.w + sp.drift) * sp.baumgarte) * dt_inv;
        bb[ic] = bv;
    }
    cs.jac_inv[k] = mk4(jac[0], jac[1], jac[2], jac[3]);
    cs.b[k] = mk4(bb[0], bb[1], bb[2], bb[3]);
    cs.lambda[k] = mk4(0, 0, 0, 0);
    float4 fr = mk4(0, 0, 0, 0);
    float4 cen = mk4(0, 0, 0, 0);
    if (npts > 0) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if ((float)i < npts) cen = add4(cen, src.pos[i]);
        cen = mk4(cen.x / npts, cen.y / npts, cen.z / npts, cen.w / npts);
        float4 t0, t1;
        plane_space(n, t0, t1);
        float4 r0 = sub4(cen, pA), r1 = sub4(cen, pB);
        fr.x = jac_coeff(neg4(cross3(r0, t0)), cross3(r1, t0), imA, IA, imB, IB);
        fr.y = jac_coeff(neg4(cross3(r0, t1)), cross3(r1, t1), imA, IA, imB, IB);
    }
    cs.center[k] = cen;
#pragma unroll
    for (int i = 0; i < 4; i++) cs.pos[4 * k + i] = (float)i < npts ? src.pos[i] : mk4(0, 0, 0, 0);
    cs.bodies[k] = make_int2(a, b);
    cs.pair[k] = p;
    solve_pos[k] = -1;  // set by the tile packing when the row is solved
    // ---- warm start: previous step's impulses of the same pair entry (the
    // body pair, or for a compound child or mesh triangle the child pair) ----
    int prev_n = *prev_count;
    float4 prev = mk4(0, 0, 0, 0);
    int has_prev = 0, lo_match = 0;
    {
        const int2 key = pairs[p];
        int lo = 0, hi = prev_n;
        while (lo < hi) {
            int mid = (lo + hi) >> 1;
            int2 kk = prev_keys[mid];
            if (kk.x < key.x || (kk.x == key.x && kk.y < key.y)) lo = mid + 1; else hi = mid;
        }
        if (lo < prev_n && prev_keys[lo].x == key.x && prev_keys[lo].y == key.y) {
            prev = prev_imp[lo];
            has_prev = 1;
            lo_match = lo;
        }
    }
    // per-contact features of the learned warm start (16 floats)
    {
        float4 t0, t1;
        plane_space(n, t0, t1);
        float4 rA = sub4(cen, pA), rB = sub4(cen, pB);
        float4 va = add4(vA, cross3(wA, rA)), vb = add4(vB, cross3(wB, rB));
        float4 vr = sub4(va, vb);
        float dmin = FLT_MAX, jsum = 0.f, bsum = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++)
            if ((float)i < npts) {
                dmin = fminf(dmin, src.pos[i].w);
                jsum += jac[i];
                bsum += bb[i];
            }
        float inv_n = npts > 0 ? 1.f / npts : 0.f;
        float f[16] = {n.x, n.y, n.z, npts > 0 ? 10.f * dmin : 0.f,
                       dot3(vr, n), dot3(vr, t0), dot3(vr, t1), imA,
                       imB, prev.x * RB_MLP_SCALE, prev.y * RB_MLP_SCALE, prev.z * RB_MLP_SCALE,
                       npts * 0.25f, (float)has_prev, -jsum * inv_n, bsum * inv_n};
        float4 *fo = reinterpret_cast<float4 *>(features + 16 * (size_t)k);
        fo[0] = mk4(f[0], f[1], f[2], f[3]);
        fo[1] = mk4(f[4], f[5], f[6], f[7]);
        fo[2] = mk4(f[8], f[9], f[10], f[11]);
        fo[3] = mk4(f[12], f[13], f[14], f[15]);
    }
    if (sp.warm_start != MI_RB_WARM_ZERO && has_prev && npts > 0) {
        // each point takes the normal impulse of the nearest point of the
        // pair's previous manifold (first of equals); the learned start
        // rescales these to its predicted total
        const int pn = (int)prev.w;
        float lv[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if ((float)i >= npts || jac[i] == 0.f) continue;
            float4 q = src.pos[i];
            float dbest = FLT_MAX, lbest = 0.f;
            for (int j = 0; j < pn; j++) {
                float4 pp = prev_pts[4 * (size_t)lo_match + j];
                float dx = q.x - pp.x, dy = q.y - pp.y, dz = q.z - pp.z;
                float d2 = (dx * dx + dy * dy) + dz * dz;
                if (d2 < dbest) { dbest = d2; lbest = pp.w; }
            }
            lv[i] = lbest;
        }
        cs.lambda[k] = mk4(lv[0], lv[1], lv[2], lv[3]);
        fr.z = prev.y;
        fr.w = prev.z;
    }
    cs.fric[k] = fr;
    // Owner tile (the reference bins by body A's cell, SetSortDataKernel,
    // solverSetup2.cl:452-479).  Scene tiles: the scene.  Spatial tiles: the
    // minimum, per axis, of the tiles of the dynamic bodies' AABB centres; a
    // row then only touches bodies in its owner tile and the next tile in +x
    // and +z (AABB centres of touching bodies are at most one cell apart and a
    // tile is at least a cell), so tiles of equal (x, z) parity share no
    // dynamic body and 4 phases per sweep suffice.
    int t;
    if (sp.tile_mode == 1) {
        t = scene[imA != 0.f ? a : b];
    } else {
        float4 ca = mk4((aabb_min[a].x + aabb_max[a].x) * 0.5f, 0.f,
                        (aabb_min[a].z + aabb_max[a].z) * 0.5f, 0.f);
        float4 cb = mk4((aabb_min[b].x + aabb_max[b].x) * 0.5f, 0.f,
                        (aabb_min[b].z + aabb_max[b].z) * 0.5f, 0.f);
        int2 ta = tile_xz(ca.x, ca.z, sp), tb = tile_xz(cb.x, cb.z, sp);
        if (imA == 0.f) ta = tb;
        if (imB == 0.f) tb = ta;
        int tx = ta.x < tb.x ? ta.x : tb.x, tz = ta.y < tb.y ? ta.y : tb.y;
        t = tz * sp.tiles_x + tx;
    }
    tile_kv[k] = make_uint2((uint32_t)t, (uint32_t)k);
}

// tile_first/tile_cnt of every tile (zeroed by the step's first kernel):
// the run boundaries of the sorted tile keys
__global__ void k_tile_bounds2(const uint2 *__restrict__ tile_kv, const int *counters,
                               int *tile_first, int *tile_cnt) {
    int nc = counters[RB_CNT_CONTACTS];
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nc) return;
    uint32_t t = tile_kv[k].x;
    if (k == 0 || tile_kv[k - 1].x != t) tile_first[t] = k;
    if (k == nc - 1 || tile_kv[k + 1].x != t) tile_cnt[t] = k + 1;  // end of the run
}

// ---- per-tile colouring (Luby rounds in LDS) and colour-major order ----
struct TileLDS {
    int key[HASH_SLOTS];                 // body index per hash slot, -1 empty
    unsigned long long mark[HASH_SLOTS]; // (round << 32) | priority
    unsigned long long used[HASH_SLOTS]; // colours already taken by the body's rows
    short la[RB_TILE_MAX_ROWS], lb[RB_TILE_MAX_ROWS];  // local slots (-1 static)
    unsigned char color[RB_TILE_MAX_ROWS];
    int ccount[RB_MAX_LOCAL_COLORS + 1];
    int coff[RB_MAX_LOCAL_COLORS + 1];
    int remaining;
};

// open-addressing body -> LDS slot tables (SLOTS a power of two)
template <int SLOTS>
__device__ __forceinline__ int hash_insert(int *key, int body) {
    uint32_t h = ((uint32_t)body * 2654435761u) & (SLOTS - 1);
    for (int probe = 0; probe < SLOTS; probe++) {
        int old = atomicCAS(&key[h], -1, body);
        if (old == -1 || old == body) return (int)h;
        h = (h + 1) & (SLOTS - 1);
    }
    return -1;
}
template <int SLOTS>
__device__ __forceinline__ int hash_find(const int *key, int body) {
    uint32_t h = ((uint32_t)body * 2654435761u) & (SLOTS - 1);
    for (int probe = 0; probe < SLOTS; probe++) {
        int k = key[h];
        if (k == body) return (int)h;
        if (k == -1) return -1;
        h = (h + 1) & (SLOTS - 1);
    }
    return -1;
}

__global__ __launch_bounds__(TB) void k_tile_color(
    const uint2 *__restrict__ tile_kv, const int *__restrict__ tile_first,
    const int *__restrict__ tile_cnt, const int2 *__restrict__ bodies,
    const float *__restrict__ inv_mass, int *__restrict__ order, int *__restrict__ row_color,
    int *__restrict__ tile_color_off, int *__restrict__ tile_ncolors, int *counters) {
    __shared__ TileLDS L;
    const int t = blockIdx.x;
    const int first = tile_first[t];
    int R = tile_cnt[t] - first;
    if (R > RB_TILE_MAX_ROWS) {
        if (threadIdx.x == 0) atomicOr(counters + RB_CNT_OVERFLOW, (int)MI_RB_OVERFLOW_TILE);
        R = RB_TILE_MAX_ROWS;
    }
    for (int i = threadIdx.x; i < HASH_SLOTS; i += TB) {
        L.key[i] = -1;
        L.mark[i] = 0ull;
        L.used[i] = 0ull;
    }
    for (int i = threadIdx.x; i <= RB_MAX_LOCAL_COLORS; i += TB) L.ccount[i] = 0;
    if (threadIdx.x == 0) L.remaining = 0;
    __syncthreads();
    for (int r = threadIdx.x; r < R; r += TB) {
        int k = (int)tile_kv[first + r].y;
        int2 bd = bodies[k];
        int sa = inv_mass[bd.x] != 0.f ? hash_insert<HASH_SLOTS>(L.key, bd.x) : -1;
        int sb = inv_mass[bd.y] != 0.f ? hash_insert<HASH_SLOTS>(L.key, bd.y) : -1;
        L.la[r] = (short)sa;
        L.lb[r] = (short)sb;
        L.color[r] = 0xff;
    }
    __syncthreads();
    // Jones-Plassmann rounds: a row whose priority is the highest among the
    // uncoloured rows at both its dynamic bodies takes the lowest colour that
    // none of those bodies' coloured rows holds.  The rows taking colours in
    // one round share no body, so each body's colour mask has one writer.
    int ncol = 0;
    for (int round = 0; round < RB_MAX_LOCAL_COLORS; round++) {
        unsigned long long tag = ((unsigned long long)(round + 1) << 32);
        for (int r = threadIdx.x; r < R; r += TB) {
            if (L.color[r] != 0xff) continue;
            unsigned long long v = tag | color_prio(tile_kv[first + r].y);
            if (L.la[r] >= 0) atomicMax(&L.mark[L.la[r]], v);
            if (L.lb[r] >= 0) atomicMax(&L.mark[L.lb[r]], v);
        }
        __syncthreads();
        int left = 0;
        for (int r = threadIdx.x; r < R; r += TB) {
            if (L.color[r] != 0xff) continue;
            unsigned long long v = tag | color_prio(tile_kv[first + r].y);
            const int la = L.la[r], lb = L.lb[r];
            bool win = (la < 0 || L.mark[la] == v) && (lb < 0 || L.mark[lb] == v);
            if (win) {
                const unsigned long long u = (la >= 0 ? L.used[la] : 0ull) |
                                             (lb >= 0 ? L.used[lb] : 0ull);
                int c = RB_MAX_LOCAL_COLORS - 1;
                if (~u) c = __builtin_ctzll(~u);
                else atomicOr(counters + RB_CNT_OVERFLOW, (int)MI_RB_OVERFLOW_COLORS);
                L.color[r] = (unsigned char)c;
                if (la >= 0) L.used[la] |= 1ull << c;
                if (lb >= 0) L.used[lb] |= 1ull << c;
            } else {
                left++;
            }
        }
        if (left) atomicAdd(&L.remaining, left);
        __syncthreads();
        int rem = L.remaining;
        __syncthreads();
        if (threadIdx.x == 0) L.remaining = 0;
        if (rem == 0) break;
        __syncthreads();
    }
    __syncthreads();
    // rows still uncoloured: one colour each after the last (serial, rare)
    if (threadIdx.x == 0) {
        int extra = 0;
        for (int r = 0; r < R; r++)
            if (L.color[r] == 0xff) extra++;
        if (extra) atomicOr(counters + RB_CNT_OVERFLOW, (int)MI_RB_OVERFLOW_COLORS);
    }
    for (int r = threadIdx.x; r < R; r += TB) {
        if (L.color[r] == 0xff) L.color[r] = (unsigned char)(RB_MAX_LOCAL_COLORS - 1);
        atomicAdd(&L.ccount[L.color[r]], 1);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int run = 0;
        for (int c = 0; c < RB_MAX_LOCAL_COLORS; c++) {
            L.coff[c] = run;
            tile_color_off[t * (RB_MAX_LOCAL_COLORS + 1) + c] = run;
            run += L.ccount[c];
            L.ccount[c] = 0;
        }
        tile_color_off[t * (RB_MAX_LOCAL_COLORS + 1) + RB_MAX_LOCAL_COLORS] = run;
        int nc = ncol;
        for (int c = 0; c < RB_MAX_LOCAL_COLORS; c++)
            if (L.coff[c] < run && c + 1 > nc) nc = c + 1;
        tile_ncolors[t] = nc;
        atomicMax(counters + RB_CNT_NCOLORS, nc);
    }
    __syncthreads();
    // colour-major, index order within a colour: rows are in index order here,
    // so a ballot-ranked stable scatter per colour keeps it
    for (int base = 0; base < R; base += TB) {
        int r = base + threadIdx.x;
        int c = r < R ? L.color[r] : -1;
        // stable rank among equal colours within this chunk: serial over waves
        for (int w = 0; w < TB / 64; w++) {
            if ((threadIdx.x >> 6) == w && r < R) {
                uint64_t peers = __ballot(true);
                for (int bit = 0; bit < 6; bit++) {
                    uint64_t bal = __ballot((c >> bit) & 1);
                    peers &= ((c >> bit) & 1) ? bal : ~bal;
                }
                int below = __popcll(peers & lanemask_lt());
                int before = L.ccount[c];
                wave_sync();
                if (below == 0) L.ccount[c] = before + __popcll(peers);
                wave_sync();
                int dst = L.coff[c] + before + below;
                int k = (int)tile_kv[first + r].y;
                order[first + dst] = k;
                row_color[k] = c;
            }
            __syncthreads();
        }
    }
}

// ---- solve ----
// Four lanes (a quad) run one row: lane 0 holds body A's linear velocity,
// lane 1 its angular velocity, lanes 2 and 3 body B's.  Each lane multiplies
// its own quarter of the row's Jacobian, the four dot products are summed in
// lane order across the quad (DPP), every lane forms the same impulse, and
// each lane updates its own velocity: the same operations in the same order
// as one thread working through the row, so the results are identical.  What
// bounds a sweep is the serial chain of a colour (up to four points, each
// reading the velocities the last one wrote) in the one or two waves that
// hold the colour's rows: split over a quad a point issues about 25
// instructions where one thread per row issued 61, and the row's data is
// spread over four lanes' registers (110 of them where a thread per row took
// 212, so twice the workgroups of a phase run at once).  Launches of 65,537
// hulls in contact: normal 9.6 -> 7.1 us, friction 9.9 -> 6.7 us; 4,096 cubes
// on a triangle mesh: 16.3 -> 6.4 and 17.2 -> 6.2 us.
constexpr int SOLVE_SLOTS = 1012;  // LDS velocity cache of one tile (five such tiles in a CU's LDS)
constexpr int SLOT_STATIC = SOLVE_SLOTS;      // static body: the zero slot, no writes
constexpr int SLOT_GLOBAL = SOLVE_SLOTS + 1;  // dynamic body beyond the LDS cache: global memory
enum { ROW_NORMAL = 0, ROW_FRICTION = 1, ROW_WARM = 2 };

struct TileSolveLDS {
    // slot s: linear at 2s + 2, angular at 2s + 3; the first two are zero
    float4 vel[2 * (SOLVE_SLOTS + 1)];
    uint2 red[8];  // store_tile_residual's waves
};

#define QUAD_PERM(p) " quad_perm:" p " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
// ((x0 + x1) + x2) + x3 over the lanes of a quad.  Lanes 0 and 1 first swap
// and add (their sum is the same either way round).  A DPP read must trail the
// write of its source by two instructions; written out, the copies of lanes 2
// and 3 fill one of the two gaps, where the compiler's order needs four waits.
__device__ __forceinline__ float quad_sum(float x) {
    float r, y, z;
    asm("s_nop 1\n\t"
        "v_add_f32_dpp %0, %3, %3" QUAD_PERM("[1,0,3,2]")
        "v_mov_b32_dpp %1, %3" QUAD_PERM("[2,2,2,2]")
        "v_mov_b32_dpp %2, %3" QUAD_PERM("[3,3,3,3]")
        "v_add_f32_dpp %1, %0, %1" QUAD_PERM("[0,0,0,0]")
        "v_add_f32_e32 %0, %1, %2"
        : "=&v"(r), "=&v"(y), "=&v"(z)
        : "v"(x));
    return r;
}
// The quad's four values in every lane, formed before the row's serial chain
// starts (folded into the chain's instructions as DPP operands, each would
// cost the chain a wait instead).
__device__ __forceinline__ void quad_spread(float x, float out[4]) {
    asm("s_nop 1\n\t"
        "v_mov_b32_dpp %0, %4" QUAD_PERM("[0,0,0,0]")
        "v_mov_b32_dpp %1, %4" QUAD_PERM("[1,1,1,1]")
        "v_mov_b32_dpp %2, %4" QUAD_PERM("[2,2,2,2]")
        "v_mov_b32_dpp %3, %4 quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf bound_ctrl:1"
        : "=&v"(out[0]), "=&v"(out[1]), "=&v"(out[2]), "=&v"(out[3])
        : "v"(x));
}

// A lane's part of a row: its LDS velocity slot in the low half, the row's
// colour in the high half.
__device__ __forceinline__ float4 fetch_vel(int slot, int body, int l, const float4 *vel,
                                            const float4 *linvel, const float4 *angvel) {
    const int s = slot < SLOT_STATIC ? slot + 1 : 0;
    float4 v = vel[2 * s + (l & 1)];
    if (slot == SLOT_GLOBAL) v = (l & 1 ? angvel : linvel)[body];
    return v;
}
__device__ __forceinline__ void put_vel(int slot, int body, int l, float4 v, float4 *vel,
                                        float4 *linvel, float4 *angvel) {
    if (slot < SLOT_STATIC) vel[2 * (slot + 1) + (l & 1)] = v;
    else if (slot == SLOT_GLOBAL) (l & 1 ? angvel : linvel)[body] = v;
}

// (a choice between two float4 variables is written by value: as a choice of
// addresses it puts both into scratch)
__device__ __forceinline__ float4 sel4(bool c, float4 a, float4 b) {
    return mk4(c ? a.x : b.x, c ? a.y : b.y, c ? a.z : b.z, c ? a.w : b.w);
}

// What a solve reads besides the packed rows: the constraints and bodies the
// scene tiles form their rows from, and the velocities.
struct SolveView {
    ConstraintSoA cs;
    const int *order;
    const float4 *pos;
    const float *inv_mass;
    const float4 *invI;
    float4 *linvel, *angvel;
};

// A lane's quarter of a normal row: per point its Jacobian and the velocity
// change per impulse (w of the linear lanes' is the friction coefficient over
// the mass, the same for every point).  Lane q of the quad holds point q's
// 1/J M J^T, bias and impulse; the quad reads them by DPP.
struct NormalRow {
    int code;  // slot | colour << 16, -1: no row
    float J[4][3], M[4][3], mw, jac, b, lam;
};
// (the operations the constraint maths forms these terms with; every lane goes
// through the angular ones and the linear lanes drop them, which costs a wave
// nothing)
__device__ __forceinline__ void form_normal(bool side, bool ang, float4 lin0, float im,
                                            const float4 I[3], float4 p, const float4 wp[4],
                                            float4 J[4], float4 M[4]) {
    const float4 n = neg4(lin0), lin = sel4(side, neg4(lin0), lin0), lm = scl4(lin, im);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const float4 a = cross3(sub4(wp[q], p), n), j = sel4(side, a, neg4(a));
        J[q] = sel4(ang, j, lin);
        M[q] = sel4(ang, mt_mul1(I, j), lm);
    }
}
// ... and of a friction row: the tangents t0, t1 at the manifold centre
__device__ __forceinline__ void form_friction(bool side, bool ang, float4 lin0, float im,
                                              const float4 I[3], float4 p, float4 cen,
                                              float4 J[2], float4 M[2]) {
    float4 t[2];
    plane_space(neg4(lin0), t[0], t[1]);
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const float4 lin = sel4(side, t[q], neg4(t[q]));
        const float4 a = cross3(sub4(cen, p), t[q]), j = sel4(side, a, neg4(a));
        J[q] = sel4(ang, j, lin);
        M[q] = sel4(ang, mt_mul1(I, j), scl4(lin, im));
    }
}
// whether a friction row damps the spin about its normal (the manifold centre
// on the line of the bodies, or a static body)
__device__ __forceinline__ bool row_damps(float4 pA, float4 pB, float4 cen, float imA, float imB) {
    const float4 ab = normalize3(sub4(pB, pA)), ac = normalize3(sub4(cen, pA));
    return dot3(ab, ac) > 0.95f || (imA == 0.f || imB == 0.f);
}

__device__ __forceinline__ float lane_of(const float4 *a, int i, int l) {
    return reinterpret_cast<const float *>(a + i)[l];
}
__device__ __forceinline__ int row_code(const PackedRows &pk, int i, int l) {
    return pk.meta[2 * (size_t)i + (l >> 1)].y;
}
__device__ __forceinline__ int row_body(const PackedRows &pk, int i, int l) {
    return pk.meta[2 * (size_t)i + (l >> 1)].x;
}
// Spatial tiles: row i from the packed arrays.
__device__ __forceinline__ void load_normal(int i, int l, const PackedRows &pk, NormalRow &r) {
    r.code = row_code(pk, i, l);
    const float4 *J = pk.nj + 10 * (size_t)i + (l >> 1), *M = pk.nm + 10 * (size_t)i + (l >> 1);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int e = l & 1 ? 2 * (q + 1) : 0;
        const float4 j = J[e], m = M[e];
        r.J[q][0] = j.x; r.J[q][1] = j.y; r.J[q][2] = j.z;
        r.M[q][0] = m.x; r.M[q][1] = m.y; r.M[q][2] = m.z;
        if (q == 0) r.mw = m.w;
    }
    r.jac = lane_of(pk.jac, i, l);
    r.b = lane_of(pk.b, i, l);
    r.lam = lane_of(pk.lam, i, l);
}
// Scene tiles: the row at solve position i from its constraint.
__device__ __forceinline__ void load_normal(int i, int l, const PackedRows &pk,
                                            const SolveView &sv, NormalRow &r) {
    const int2 m = pk.meta[2 * (size_t)i + (l >> 1)];
    const int k = sv.order[i], side = l >> 1;
    const bool ang = l & 1;
    r.code = m.y;
    float4 J[4], M[4], I[3], wp[4];
    const float4 lin0 = sv.cs.linear[k], p = sv.pos[m.x];
    const float im = sv.inv_mass[m.x];
#pragma unroll
    for (int q = 0; q < 3; q++) I[q] = sv.invI[3 * (size_t)m.x + q];
#pragma unroll
    for (int q = 0; q < 4; q++) wp[q] = sv.cs.pos[4 * (size_t)k + q];
    form_normal(side, ang, lin0, im, I, p, wp, J, M);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        r.J[q][0] = J[q].x; r.J[q][1] = J[q].y; r.J[q][2] = J[q].z;
        r.M[q][0] = M[q].x; r.M[q][1] = M[q].y; r.M[q][2] = M[q].z;
    }
    r.mw = M[0].w;
    r.jac = lane_of(sv.cs.jac_inv, k, l);
    r.b = lane_of(sv.cs.b, k, l);
    r.lam = lane_of(sv.cs.lambda, k, l);
}
// solveContact (solveContact.cl:272-312): sequential impulses on the normal
// rows, lambda >= 0.
// RES: compute the sweep residual terms (the largest scaled impulse change
// and the largest impulse); sweeps whose residual nobody reads skip them,
// which leaves every velocity and impulse unchanged.
// (a point beyond the manifold's has jac, b and lambda zero: its impulse
// change is zero and its residual term 0 / 0, which fmaxf drops, so no branch
// is needed to skip it)
template <bool RES>
__device__ __forceinline__ void run_normal(NormalRow &d, int i, int l, const PackedRows &pk,
                                           float4 *vel, float4 *linvel, float4 *angvel,
                                           float &rmax, float &lmax) {
    const int slot = d.code & 0xffff;
    const int body = slot == SLOT_GLOBAL ? row_body(pk, i, l) : 0;
    float4 v = fetch_vel(slot, body, l, vel, linvel, angvel);
    float jv[4], bv[4], lv[4];
    quad_spread(d.jac, jv);
    quad_spread(d.b, bv);
    quad_spread(d.lam, lv);
#pragma unroll
    for (int ic = 0; ic < 4; ic++) {
        float rl = quad_sum((d.J[ic][0] * v.x + d.J[ic][1] * v.y) + d.J[ic][2] * v.z) + bv[ic];
        rl *= jv[ic];
        // (min(max(x, 0), FLT_MAX), NaN to 0, in one instruction)
        const float upd = __builtin_amdgcn_fmed3f(lv[ic] + rl, 0.f, FLT_MAX);
        rl = upd - lv[ic];
        if (l == ic) d.lam = upd;
        v = mk4(v.x + d.M[ic][0] * rl, v.y + d.M[ic][1] * rl, v.z + d.M[ic][2] * rl,
                v.w + d.mw * rl);
        if (RES) {
            rmax = fmaxf(rmax, fabsf(rl) / fabsf(jv[ic]));
            lmax = fmaxf(lmax, fabsf(upd));
        }
    }
    put_vel(slot, body, l, v, vel, linvel, angvel);
}

// A lane's quarter of a friction row: both tangents' Jacobians and velocity
// changes per impulse, the normal (w: the friction coefficient, negated) and
// the cone's limit.  Lanes 0 and 1 of the quad hold the tangents' 1/J M J^T,
// lanes 2 and 3 their impulses.
struct FrictionRow {
    int code;
    float J[2][3], M[2][3];
    float4 n;
    float fr, mx;
};
constexpr int ROW_DAMPS = 1 << 15;  // in a friction row's code: the angular damping applies
static_assert(SLOT_GLOBAL < ROW_DAMPS, "slot, flag and colour share a word");
__device__ __forceinline__ void set_friction(FrictionRow &r, const float4 J[2], const float4 M[2],
                                             float4 lin0, float fr, float4 lam, float friction,
                                             bool damp) {
#pragma unroll
    for (int q = 0; q < 2; q++) {
        r.J[q][0] = J[q].x; r.J[q][1] = J[q].y; r.J[q][2] = J[q].z;
        r.M[q][0] = M[q].x; r.M[q][1] = M[q].y; r.M[q][2] = M[q].z;
    }
    r.n = neg4(lin0);
    r.fr = fr;
    float sum = 0;
    sum += lam.x; sum += lam.y; sum += lam.z; sum += lam.w;
    r.mx = friction * sum;
    if (damp) r.code |= ROW_DAMPS;
}
__device__ __forceinline__ void load_friction(int i, int l, const PackedRows &pk, float friction,
                                              FrictionRow &r) {
    r.code = row_code(pk, i, l);
    const float4 *j = pk.fj + 8 * (size_t)i + l, *m = pk.fm + 8 * (size_t)i + l;
    const float4 J[2] = {j[0], j[4]}, M[2] = {m[0], m[4]};
    set_friction(r, J, M, pk.lin0[i], lane_of(pk.fric, i, l), pk.lam[i], friction, J[0].w != 0.f);
}
__device__ __forceinline__ void load_friction(int i, int l, const PackedRows &pk,
                                              const SolveView &sv, float friction,
                                              FrictionRow &r) {
    const int2 mA = pk.meta[2 * (size_t)i], mB = pk.meta[2 * (size_t)i + 1];
    const int k = sv.order[i], side = l >> 1;
    const bool ang = l & 1;
    const int body = side ? mB.x : mA.x;
    r.code = side ? mB.y : mA.y;
    const float4 lin0 = sv.cs.linear[k], cen = sv.cs.center[k];
    const float4 pA = sv.pos[mA.x], pB = sv.pos[mB.x];
    const float imA = sv.inv_mass[mA.x], imB = sv.inv_mass[mB.x];
    float4 I[3], J[2], M[2];
#pragma unroll
    for (int q = 0; q < 3; q++) I[q] = sv.invI[3 * (size_t)body + q];
    form_friction(side, ang, lin0, side ? imB : imA, I, sel4(side, pB, pA), cen, J, M);
    set_friction(r, J, M, lin0, lane_of(sv.cs.fric, k, l), sv.cs.lambda[k], friction,
                 row_damps(pA, pB, cen, imA, imB));
}
// solveFriction (solveFriction.cl:297-430): two tangents at the manifold
// centre, |lambda| <= mu * sum lambda_n, then the angular damping about n.
template <bool RES>
__device__ __forceinline__ void run_friction(FrictionRow &d, int i, int l, const PackedRows &pk,
                                             float4 *vel, float4 *linvel, float4 *angvel,
                                             float &rmax, float &lmax) {
    float f[4];
    quad_spread(d.fr, f);
    if (f[0] == 0.f) return;
    const int slot = d.code & (ROW_DAMPS - 1);
    const int body = slot == SLOT_GLOBAL ? row_body(pk, i, l) : 0;
    float4 v = fetch_vel(slot, body, l, vel, linvel, angvel);
#pragma unroll
    for (int t = 0; t < 2; t++) {
        float rl = quad_sum((d.J[t][0] * v.x + d.J[t][1] * v.y) + d.J[t][2] * v.z);
        rl *= f[t];
        float upd = f[2 + t] + rl;
        upd = fmaxf(upd, -d.mx);
        upd = fminf(upd, d.mx);
        rl = upd - f[2 + t];
        if (l == 2 + t) d.fr = upd;
        v.x += d.M[t][0] * rl; v.y += d.M[t][1] * rl; v.z += d.M[t][2] * rl;
        if (RES) {
            rmax = fmaxf(rmax, fabsf(rl) / fabsf(f[t]));
            lmax = fmaxf(lmax, fabsf(upd));
        }
    }
    if ((l & 1) && (d.code & ROW_DAMPS)) v = sub4(v, scl4(d.n, dot3(d.n, v) * 0.1f));
    put_vel(slot, body, l, v, vel, linvel, angvel);
}

// Apply the impulses a row already holds (warm start) to its bodies.
__device__ __forceinline__ void run_warm(const NormalRow &d, const FrictionRow &f, int i, int l,
                                         const PackedRows &pk, float4 *vel, float4 *linvel,
                                         float4 *angvel) {
    const int slot = d.code & 0xffff;
    const int body = slot == SLOT_GLOBAL ? row_body(pk, i, l) : 0;
    float4 v = fetch_vel(slot, body, l, vel, linvel, angvel);
    float jv[4], lv[4], fv[4];
    quad_spread(d.jac, jv);
    quad_spread(d.lam, lv);
    quad_spread(f.fr, fv);
#pragma unroll
    for (int ic = 0; ic < 4; ic++) {
        if (jv[ic] == 0.f || lv[ic] == 0.f) continue;
        v = mk4(v.x + d.M[ic][0] * lv[ic], v.y + d.M[ic][1] * lv[ic], v.z + d.M[ic][2] * lv[ic],
                v.w + d.mw * lv[ic]);
    }
    if (fv[0] != 0.f) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const float fl = fv[2 + q];
            if (fl == 0.f) continue;
            v.x += f.M[q][0] * fl; v.y += f.M[q][1] * fl; v.z += f.M[q][2] * fl;
        }
    }
    put_vel(slot, body, l, v, vel, linvel, angvel);
}

// After the solve: the impulses go back from the packed solve arrays to the
// constraints, and into the previous-step impulse cache for the warm start,
// keyed by the constraint's pair entry (unique per manifold; constraints are
// ordered by pair, so without compound child pairs, which are appended after
// the body pairs, the keys come out sorted): the totals (sum of normal
// impulses, friction 0, friction 1, number of points) and each point's
// position with its normal impulse.
__global__ void k_save_prev(const int *counters, ConstraintSoA cs, const int *solve_pos,
                            const float4 *pk_lam, const float4 *pk_fric, int2 *prev_keys,
                            float4 *prev_imp, float4 *prev_pts, int *prev_count,
                            const int2 *pairs) {
    int nc = counters[RB_CNT_CONTACTS];
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k == 0) *prev_count = nc;
    if (k >= nc) return;
    float4 l, f;
    const int pos = solve_pos[k];
    if (pos >= 0) {
        l = pk_lam[pos];
        f = pk_fric[pos];
        cs.lambda[k] = l;
        cs.fric[k] = f;
    } else {  // solved in place, or not at all (tile capacity exceeded): the initial impulses
        l = cs.lambda[k];
        f = cs.fric[k];
    }
    float4 jac = cs.jac_inv[k];
    int np = (jac.x != 0.f) + (jac.y != 0.f) + (jac.z != 0.f) + (jac.w != 0.f);
    prev_keys[k] = pairs[cs.pair[k]];
    prev_imp[k] = mk4(((l.x + l.y) + l.z) + l.w, f.z, f.w, (float)np);
    float lv[4] = {l.x, l.y, l.z, l.w};
    for (int i = 0; i < 4; i++) {
        float4 p = cs.pos[4 * (size_t)k + i];
        prev_pts[4 * (size_t)k + i] = mk4(p.x, p.y, p.z, lv[i]);
    }
}

// Per step, after the colouring: each tile's dynamic bodies as a dense list
// and each row's slots in it, so that a solve does no hashing.  Spatial tiles
// also get their rows in solve order as packed arrays with everything of a
// row that no sweep changes already formed (the Jacobians, the velocity
// changes per impulse): 20 launches read them, contiguously.  (A scene's rows
// are read by one launch, which forms them itself from the constraints: packed
// for it as well, they took this kernel from 130 to 265 us at 4,096 scenes.)
// Four lanes pack a row, each the quarter that the same lane of the solver's
// quad reads.
constexpr int SOLVED_IN_PLACE = -2;  // solve_pos: the solve stores to the constraint itself
struct PackLDS {
    int key[HASH_SLOTS];
    int dense[HASH_SLOTS];
    int count;
};
__global__ __launch_bounds__(TB) void k_tile_pack(
    const int *__restrict__ tile_first, const int *__restrict__ tile_cnt,
    const int *__restrict__ order, const int *__restrict__ row_color, ConstraintSoA cs,
    const float4 *__restrict__ pos, const float *__restrict__ inv_mass,
    const float4 *__restrict__ invI, PackedRows pk, int *__restrict__ solve_pos,
    int *__restrict__ tile_bodies, int *__restrict__ tile_nb,
    const int *__restrict__ tile_ncolors, int4 *__restrict__ tile_hdr, int *counters,
    uint2 *__restrict__ tile_res, int spatial) {
    __shared__ PackLDS L;
    const int t = blockIdx.x, tid = threadIdx.x;
    const int first = tile_first[t];
    // (the residuals of a tile that no sweep visits are zero)
    if (tid < 2) tile_res[tid * (int)gridDim.x + t] = make_uint2(0u, 0u);
    int R = tile_cnt[t] - first;
    if (R > RB_TILE_MAX_ROWS) R = RB_TILE_MAX_ROWS;
    if (R <= 0) {
        if (tid == 0) {
            tile_nb[t] = 0;
            tile_hdr[t] = make_int4(first, 0, 0, 0);
        }
        return;
    }
    for (int i = tid; i < HASH_SLOTS; i += TB) { L.key[i] = -1; L.dense[i] = -1; }
    if (tid == 0) L.count = 0;
    __syncthreads();
    for (int r = tid; r < R; r += TB) {
        int2 bd = cs.bodies[order[first + r]];
        bool fail = false;
        if (inv_mass[bd.x] != 0.f) fail |= hash_insert<HASH_SLOTS>(L.key, bd.x) < 0;
        if (inv_mass[bd.y] != 0.f) fail |= hash_insert<HASH_SLOTS>(L.key, bd.y) < 0;
        if (fail) atomicOr(counters + RB_CNT_OVERFLOW, (int)MI_RB_OVERFLOW_TILE);
    }
    __syncthreads();
    // dense slots: the occupied hash slots numbered in slot order
    for (int i = tid; i < HASH_SLOTS; i += TB)
        if (L.key[i] >= 0) L.dense[i] = atomicAdd(&L.count, 1);
    __syncthreads();
    const int nb = L.count;
    for (int i = tid; i < HASH_SLOTS; i += TB)
        if (L.key[i] >= 0) tile_bodies[2 * (size_t)first + L.dense[i]] = L.key[i];
    if (tid == 0) {
        tile_nb[t] = nb;
        tile_hdr[t] = make_int4(first, R, tile_ncolors[t], nb < SOLVE_SLOTS ? nb : SOLVE_SLOTS);
        atomicAdd(counters + RB_CNT_SOLVE_BODIES, nb);
    }
    const int l = tid & 3, side = l >> 1;
    const bool ang = l & 1;
    for (int r = tid >> 2; r < R; r += TB / 4) {
        const int i = first + r;
        const int k = order[i];
        const int2 bd = cs.bodies[k];
        const int body = side ? bd.y : bd.x;
        const float imA = inv_mass[bd.x], imB = inv_mass[bd.y], im = side ? imB : imA;
        if (!ang) {
            int slot = SLOT_STATIC;
            if (im != 0.f) {
                const int h = hash_find<HASH_SLOTS>(L.key, body);
                slot = h >= 0 && L.dense[h] < SOLVE_SLOTS ? L.dense[h] : SLOT_GLOBAL;
            }
            pk.meta[2 * (size_t)i + side] = make_int2(body, slot | row_color[k] << 16);
        }
        if (!spatial) {
            if (l == 0) solve_pos[k] = SOLVED_IN_PLACE;
            continue;
        }
        const float4 lin0 = cs.linear[k], fr = cs.fric[k];
        const float4 pA = pos[bd.x], pB = pos[bd.y], p = sel4(side, pB, pA);
        float4 I[3], wp[4];
        for (int q = 0; q < 3; q++) I[q] = invI[3 * (size_t)body + q];
        for (int q = 0; q < 4; q++) wp[q] = cs.pos[4 * (size_t)k + q];
        if (l == 0) {
            pk.lin0[i] = lin0;
            pk.lam[i] = cs.lambda[k];
            solve_pos[k] = i;
        } else if (l == 1) {
            pk.jac[i] = cs.jac_inv[k];
        } else if (l == 2) {
            pk.b[i] = cs.b[k];
        } else {
            pk.fric[i] = fr;
        }
        float4 J[4], M[4];
        form_normal(side, ang, lin0, im, I, p, wp, J, M);
        float4 *nj = pk.nj + 10 * (size_t)i + side, *nm = pk.nm + 10 * (size_t)i + side;
        for (int q = 0; q < 4; q++)
            if (ang || q == 0) {
                nj[ang ? 2 * (q + 1) : 0] = J[q];
                nm[ang ? 2 * (q + 1) : 0] = M[q];
            }
        const float4 cen = cs.center[k];
        form_friction(side, ang, lin0, im, I, p, cen, J, M);
        const bool damp = row_damps(pA, pB, cen, imA, imB);
        float4 *fj = pk.fj + 8 * (size_t)i + l, *fm = pk.fm + 8 * (size_t)i + l;
        for (int q = 0; q < 2; q++) {
            J[q].w = damp ? 1.f : 0.f;  // (no sweep reads w)
            fj[4 * q] = J[q];
            fm[4 * q] = M[q];
        }
    }
}

// The sweep residual terms (largest scaled impulse change, largest impulse):
// the maximum over the workgroup's lanes and waves, in LDS, then one store to
// the tile's own place, where k_sweep_done and k_sweep_summary look (the terms
// are >= 0, so their float bits order like the values).  (Gathered by one
// atomic pair per workgroup, a launch of the 841 tiles of a phase of a mesh
// scene took 22.4 us against 6.4 us without; 65,537 hulls 12.6 against 7.1.)
// They are needed after every sweep with a tolerance, otherwise only for the
// last normal and the last friction sweep, the residuals a step reports.
__host__ __device__ __forceinline__ bool sweep_residual_needed(const StepParams &sp, int sweep) {
    return sp.tol > 0.f || sweep == sp.normal_iters - 1 ||
           sweep == sp.normal_iters + sp.friction_iters - 1;
}
// max over a wave, whose quads hold equal values
__device__ __forceinline__ uint2 wave_residual(float rmax, float lmax) {
    unsigned r = __float_as_uint(rmax), m = __float_as_uint(lmax);
#pragma unroll
    for (int o = 32; o >= 4; o >>= 1) {
        r = max(r, (unsigned)__shfl_xor((int)r, o));
        m = max(m, (unsigned)__shfl_xor((int)m, o));
    }
    return make_uint2(r, m);
}
// Every thread of the workgroup calls it; red: one word pair per wave in LDS.
__device__ __forceinline__ void store_tile_residual(uint2 *dst, float rmax, float lmax,
                                                    uint2 *red) {
    const uint2 w = wave_residual(rmax, lmax);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = w;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint2 t = red[0];
        for (unsigned k = 1; k < blockDim.x / 64; k++) {
            t.x = max(t.x, red[k].x);
            t.y = max(t.y, red[k].y);
        }
        *dst = t;
    }
}

// A tile's sweeps take their rows through a row source: load(i, row) and
// store(i, row) of normal and friction rows by solve position, from the packed
// arrays (spatial tiles: a row is read by 20 launches) or straight from the
// constraints (scene tiles: one launch reads it once and keeps it).
struct PackedSource {
    const PackedRows &pk;
    float friction;
    __device__ void load(int i, int l, NormalRow &r) const { load_normal(i, l, pk, r); }
    __device__ void load(int i, int l, FrictionRow &r) const { load_friction(i, l, pk, friction, r); }
    __device__ void store(int i, int l, const NormalRow &r) const {
        reinterpret_cast<float *>(pk.lam + i)[l] = r.lam;
    }
    __device__ void store(int i, int l, const FrictionRow &r) const {
        if (l & 2) reinterpret_cast<float *>(pk.fric + i)[l] = r.fr;
    }
};
struct ConstraintSource {
    const PackedRows &pk;
    const SolveView &sv;
    float friction;
    __device__ void load(int i, int l, NormalRow &r) const { load_normal(i, l, pk, sv, r); }
    __device__ void load(int i, int l, FrictionRow &r) const {
        load_friction(i, l, pk, sv, friction, r);
    }
    __device__ void store(int i, int l, const NormalRow &r) const {
        reinterpret_cast<float *>(sv.cs.lambda + sv.order[i])[l] = r.lam;
    }
    __device__ void store(int i, int l, const FrictionRow &r) const {
        if (l & 2) reinterpret_cast<float *>(sv.cs.fric + sv.order[i])[l] = r.fr;
    }
};
template <bool RES>
__device__ __forceinline__ void run_row(NormalRow &d, int i, int l, const PackedRows &pk,
                                        float4 *vel, float4 *linvel, float4 *angvel, float &rmax,
                                        float &lmax) {
    run_normal<RES>(d, i, l, pk, vel, linvel, angvel, rmax, lmax);
}
template <bool RES>
__device__ __forceinline__ void run_row(FrictionRow &d, int i, int l, const PackedRows &pk,
                                        float4 *vel, float4 *linvel, float4 *angvel, float &rmax,
                                        float &lmax) {
    run_friction<RES>(d, i, l, pk, vel, linvel, angvel, rmax, lmax);
}

// The quad of a thread among the QN quads that share a tile, and its lane.
struct Quad {
    int QN, q, l;
};
// The rows of a tile of at most K * QN rows in the registers of QN quads: row
// r in quad r % QN, set r / QN.  Within a colour rows share no dynamic body,
// so which quad runs a row does not change the result.
template <int K, class Row, class Src>
__device__ __forceinline__ void load_rows(Row (&row)[K], Quad u, const Src &src, int first, int R) {
#pragma unroll
    for (int k = 0; k < K; k++) {
        row[k].code = -1;
        if (k * u.QN + u.q < R) src.load(first + k * u.QN + u.q, u.l, row[k]);
    }
}
template <int K, class Row, class Src>
__device__ __forceinline__ void store_rows(const Row (&row)[K], Quad u, const Src &src, int first,
                                           int R) {
#pragma unroll
    for (int k = 0; k < K; k++)
        if (k * u.QN + u.q < R) src.store(first + k * u.QN + u.q, u.l, row[k]);
}
// One sweep, colour by colour; sync() orders the velocities between colours
// among the tile's threads (after_last: what every thread does between the
// last colour and its sync).
template <int K, bool RES, class Row, class S, class F>
__device__ __forceinline__ void sweep_rows(Row (&row)[K], Quad u, int first, int nc,
                                           const PackedRows &pk, float4 *vel, float4 *linvel,
                                           float4 *angvel, float &rmax, float &lmax, S sync,
                                           F after_last) {
    for (int c = 0; c < nc; c++) {
#pragma unroll
        for (int k = 0; k < K; k++)
            if (row[k].code >> 16 == c)
                run_row<RES>(row[k], first + k * u.QN + u.q, u.l, pk, vel, linvel, angvel, rmax,
                             lmax);
        if (c == nc - 1) after_last();
        sync();
    }
}
// The same for a tile of more rows: they are read on every pass.
template <bool RES, class Row, class Src, class S, class F>
__device__ __forceinline__ void sweep_memory(Quad u, const Src &src, int first, int R, int nc,
                                             const int *coff, const PackedRows &pk, float4 *vel,
                                             float4 *linvel, float4 *angvel, float &rmax,
                                             float &lmax, S sync, F after_last) {
    for (int c = 0; c < nc; c++) {
        const int c1 = min(coff[c + 1], R);
        for (int r = coff[c] + u.q; r < c1; r += u.QN) {
            Row d;
            src.load(first + r, u.l, d);
            run_row<RES>(d, first + r, u.l, pk, vel, linvel, angvel, rmax, lmax);
            src.store(first + r, u.l, d);
        }
        if (c == nc - 1) after_last();
        sync();
    }
}
template <class Src, class S>
__device__ __forceinline__ void sweep_warm(Quad u, const Src &src, int first, int R, int nc,
                                           const int *coff, const PackedRows &pk, float4 *vel,
                                           float4 *linvel, float4 *angvel, S sync) {
    for (int c = 0; c < nc; c++) {
        const int c1 = min(coff[c + 1], R);
        for (int r = coff[c] + u.q; r < c1; r += u.QN) {
            NormalRow d;
            FrictionRow f;
            src.load(first + r, u.l, d);
            src.load(first + r, u.l, f);
            run_warm(d, f, first + r, u.l, pk, vel, linvel, angvel);
        }
        sync();
    }
}

// The tile's dynamic bodies' velocities into LDS slots (slot s: body
// bodies[s]), thread pairs of a slot taking its linear and its angular half
// (nt threads, tid counted among them).  Thread tid keeps the body of slot
// tid / 2 in a register for the store back, which then waits on no index load.
__device__ __forceinline__ int gather_velocities(int tid, int nt, const int *__restrict__ bodies,
                                                 int nb, const float4 *__restrict__ linvel,
                                                 const float4 *__restrict__ angvel, float4 *vel) {
    const float4 *src = tid & 1 ? angvel : linvel;
    const int b0 = tid < 2 * nb ? bodies[tid >> 1] : 0;
    if (tid < 2 * nb) vel[2 + tid] = src[b0];
    for (int s = tid + nt; s < 2 * nb; s += nt) vel[2 + s] = src[bodies[s >> 1]];
    if (tid < 2) vel[tid] = mk4(0.f, 0.f, 0.f, 0.f);
    return b0;
}
__device__ __forceinline__ void store_velocities(int tid, int nt, const int *__restrict__ bodies,
                                                 int nb, int b0, float4 *__restrict__ linvel,
                                                 float4 *__restrict__ angvel, const float4 *vel) {
    float4 *dst = tid & 1 ? angvel : linvel;
    if (tid < 2 * nb) dst[b0] = vel[2 + tid];
    for (int s = tid + nt; s < 2 * nb; s += nt) dst[bodies[s >> 1]] = vel[2 + s];
}

// Spatial tiles: one sweep (MODE: normal, friction, or the warm start's
// impulses) over the tiles of one parity phase, a workgroup of TBK threads per
// tile, the tile's dynamic body velocities in LDS.  A colour of more rows than
// the tile has quads takes a turn for each TBK / 4 of them: 64 quads were
// slower on tall columns than the 256 threads, a row each, before them (8 x 8
// columns of 64 cubes 458 -> 481 us a step, of 128 662 -> 806), 128 quads are
// faster (360 and 592).
template <int TBK, int MODE, bool RES>
__global__ __launch_bounds__(TBK) void k_tile_solve(
    StepParams sp, int phase, const int4 *__restrict__ tile_hdr,
    const int *__restrict__ tile_color_off, const int *__restrict__ tile_bodies, PackedRows pk,
    float4 *linvel, float4 *angvel, uint2 *__restrict__ tile_res, const int *counters) {
    constexpr int K = 2;
    __shared__ TileSolveLDS L;
    // tiles of this phase: (tx & 1, tz & 1) == (phase & 1, phase >> 1)
    const int px = phase & 1, pz = phase >> 1;
    const int nx = (sp.tiles_x - px + 1) / 2;
    const int tx = px + 2 * (int)(blockIdx.x % nx), tz = pz + 2 * (int)(blockIdx.x / nx);
    if (tx >= sp.tiles_x || tz >= sp.tiles_z) return;
    const int t = tz * sp.tiles_x + tx, tid = threadIdx.x;
    // (first, rows, colours, cached bodies) of the tile, written by k_tile_pack
    const int4 hdr = tile_hdr[t];
    if (sp.tol > 0.f && counters[RB_CNT_DONE] != 0) return;  // converged in an earlier sweep
    const int first = hdr.x, R = hdr.y, nc = hdr.z, nb = hdr.w;
    if (R <= 0) return;
    const int *coff = tile_color_off + t * (RB_MAX_LOCAL_COLORS + 1);
    const int *bodies = tile_bodies + 2 * (size_t)first;
    float rmax = 0.f, lmax = 0.f;
    auto sync = []() { __syncthreads(); };
    auto nothing = []() {};
    const Quad u{TBK / 4, tid >> 2, tid & 3};
    const PackedSource src{pk, sp.friction};
    int b0;
    if constexpr (MODE == ROW_WARM) {
        b0 = gather_velocities(tid, TBK, bodies, nb, linvel, angvel, L.vel);
        __syncthreads();
        sweep_warm(u, src, first, R, nc, coff, pk, L.vel, linvel, angvel, sync);
    } else {
        using Row = std::conditional_t<MODE == ROW_NORMAL, NormalRow, FrictionRow>;
        if (R <= K * TBK / 4) {
            // (the rows' loads go out before the velocity gather's)
            Row row[K];
            load_rows(row, u, src, first, R);
            b0 = gather_velocities(tid, TBK, bodies, nb, linvel, angvel, L.vel);
            __syncthreads();
            sweep_rows<K, RES>(row, u, first, nc, pk, L.vel, linvel, angvel, rmax, lmax, sync,
                               nothing);
            store_rows(row, u, src, first, R);
        } else {
            b0 = gather_velocities(tid, TBK, bodies, nb, linvel, angvel, L.vel);
            __syncthreads();
            sweep_memory<RES, Row>(u, src, first, R, nc, coff, pk, L.vel, linvel, angvel, rmax,
                                   lmax, sync, nothing);
        }
    }
    if (RES)
        store_tile_residual(tile_res + (MODE == ROW_FRICTION ? sp.n_tiles : 0) + t, rmax, lmax, L.red);
    store_velocities(tid, TBK, bodies, nb, b0, linvel, angvel, L.vel);
}

// Scene tiles: every sweep of a scene in one workgroup, the warm-start pass
// first; with a tolerance a scene ends each phase as soon as its own residual
// is below it.  A workgroup (a whole CU: 1,024 threads of up to 128 registers)
// solves 2^lg scenes, each with 1024 >> lg threads whose quads hold two rows
// each in registers, lg by the scene's rows (scene_class).  The scenes of a
// workgroup share its hardware barrier (see sync below).  Scenes are sorted by
// rows, so those that share a workgroup take about as long.  What bounds a
// scene is its colours times its sweeps in sequence; what bounds the launch at
// thousands of scenes is how many of those chains the chip runs at once, which
// the registers limit (124 words a row).  4,096 scenes of 8 to 512 bodies, 10 +
// 10 sweeps: 994 -> 479 us against 256 threads per scene, a thread per row and
// the rows of scenes above 256 read on every pass; 256 scenes to a tolerance:
// 2.4x.  A launch per class in sequence took 612 us, and on 256 scenes, where
// each is as long as its longest scene, twice this one's time.
constexpr int SCENE_TB = 1024, SCENE_CLASSES = 5;
constexpr int SCENE_SLOTS = SCENE_TB + (1 << (SCENE_CLASSES - 1));
// Threads of a scene: at most two rows a quad while that leaves a whole wave,
// and no fewer than leave every CU a workgroup (max_class).
__device__ __forceinline__ int scene_class(int R, int max_class) {
    int lg = 0;
    while (lg < max_class && 2 * (SCENE_TB >> (lg + 1)) / 4 >= R) lg++;
    return lg;
}
__global__ __launch_bounds__(SCENE_TB) void k_scene_solve(
    StepParams sp, int warm, const int4 *__restrict__ tile_hdr,
    const int *__restrict__ tile_color_off, const int *__restrict__ tile_bodies, PackedRows pk,
    SolveView sv, uint2 *__restrict__ tile_res, int4 *__restrict__ tile_stats,
    const uint2 *__restrict__ tile_order, const int *__restrict__ counters) {
    __shared__ float4 s_vel[2 * SCENE_SLOTS];
    __shared__ uint2 s_red[2][SCENE_TB / 64];  // per sweep parity: the waves' residual maxima
    // this workgroup's scenes: the classes in turn, largest scenes first, so
    // that the workgroups dispatched last are the short ones
    int b = blockIdx.x, base = 0, lg = 0, n = 0;
    for (; lg < SCENE_CLASSES; lg++) {
        n = counters[RB_CNT_SCENES + lg];
        const int wgs = (n + (1 << lg) - 1) >> lg;
        if (b < wgs) break;
        b -= wgs;
        base += n;
    }
    if (lg == SCENE_CLASSES) return;
    const int nt = SCENE_TB >> lg;
    const int g = __builtin_amdgcn_readfirstlane((int)threadIdx.x / nt), tid = threadIdx.x - g * nt;
    if ((b << lg) + g >= n) return;
    const int t = (int)tile_order[base + (b << lg) + g].y;
    const int4 hdr = tile_hdr[t];
    const int first = hdr.x, R = hdr.y, nc = hdr.z, nb = hdr.w;
    const bool tol = sp.tol > 0.f;
    if (R <= 0) {
        if (tol && tid == 0) tile_stats[t] = make_int4(-1, -1, 0, 0);
        return;
    }
    const int *coff = tile_color_off + t * (RB_MAX_LOCAL_COLORS + 1);
    const int *bodies = tile_bodies + 2 * (size_t)first;
    // (a scene of a shared workgroup has at most nt / 2 rows, hence nt bodies)
    float4 *vel = s_vel + 2 * g * (nt + 1);
    float4 *linvel = sv.linvel, *angvel = sv.angvel;
    const ConstraintSource src{pk, sv, sp.friction};
    const Quad u{nt / 4, tid >> 2, tid & 3};
    const int wave0 = g * (nt / 64), waves = nt / 64;
    // Orders the scene's velocities between its colours.  (One wave: its LDS
    // operations are in order.)  The scenes of a workgroup come here different
    // numbers of times and leave at different times, which HIP leaves undefined
    // for __syncthreads().  What this needs is the hardware's own barrier: it
    // counts the waves that arrive, at whatever s_barrier, and waits only on
    // those that have not ended (CDNA ISA, S_BARRIER): a wave passes its k-th
    // when every running wave has arrived k times, its own scene's among them,
    // and the waves of a scene arrive and leave together.  A whole wave comes
    // here or none of it does: every branch on the way depends on values that
    // the scene's lanes share.
    auto sync = [&]() {
        if (waves == 1) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        } else {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        }
    };
    const int b0 = gather_velocities(tid, nt, bodies, nb, linvel, angvel, vel);
    sync();
    if (warm) sweep_warm(u, src, first, R, nc, coff, pk, vel, linvel, angvel, sync);

    int used[2] = {0, 0};
    float rfin[2] = {0.f, 0.f};
    int parity = 0;
    // the sweeps of one phase; sweep(res, rmax, lmax, after_last) runs one.
    // The residual is needed after every sweep with a tolerance, else of the
    // last one.
    auto run_phase = [&](int phase, int nsw, auto sweep) {
        for (int it = 0; it < nsw; it++) {
            float rmax = 0.f, lmax = 0.f;
            if (!tol && it < nsw - 1) {
                sweep(std::false_type{}, rmax, lmax, []() {});
                continue;
            }
            // each wave's maxima reach the scene's threads over the last
            // colour's sync; the buffer of the other parity is free again by
            // the syncs of this sweep
            uint2 *red = s_red[parity];
            parity ^= 1;
            sweep(std::true_type{}, rmax, lmax, [&]() {
                const uint2 w = wave_residual(rmax, lmax);
                if ((tid & 63) == 0) red[wave0 + (tid >> 6)] = w;
            });
            unsigned r = 0u, m = 0u;
            for (int w = 0; w < waves; w++) {
                r = max(r, red[wave0 + w].x);
                m = max(m, red[wave0 + w].y);
            }
            if (tol) {
                const float rm = __uint_as_float(r), lm = __uint_as_float(m);
                const float res = rm / (lm > 1.f ? lm : 1.f);
                used[phase] = it + 1;
                rfin[phase] = res;
                if (__builtin_amdgcn_readfirstlane((int)(res < sp.tol))) break;
            } else if (tid == 0) {
                tile_res[phase * sp.n_tiles + t] = make_uint2(r, m);
            }
        }
    };
    auto solve_held = [&](auto row0, auto sets, int phase, int nsw) {
        constexpr int K = decltype(sets)::value;
        decltype(row0) row[K];
        load_rows(row, u, src, first, R);
        run_phase(phase, nsw, [&](auto res, float &rmax, float &lmax, auto last) {
            sweep_rows<K, decltype(res)::value>(row, u, first, nc, pk, vel, linvel, angvel, rmax,
                                                lmax, sync, last);
        });
        store_rows(row, u, src, first, R);
    };
    auto solve_rows = [&](auto row0, int phase, int nsw) {
        if (R <= 2 * u.QN) {
            solve_held(row0, std::integral_constant<int, 2>{}, phase, nsw);
        } else if (R <= 3 * u.QN) {
            // (a few of the third set's registers spill, which is still faster
            // than reading the rows again)
            solve_held(row0, std::integral_constant<int, 3>{}, phase, nsw);
        } else {
            run_phase(phase, nsw, [&](auto res, float &rmax, float &lmax, auto last) {
                sweep_memory<decltype(res)::value, decltype(row0)>(
                    u, src, first, R, nc, coff, pk, vel, linvel, angvel, rmax, lmax, sync, last);
            });
        }
    };
    if (sp.normal_iters > 0) {
        solve_rows(NormalRow{}, 0, sp.normal_iters);
        // the friction rows read the stored normal impulses
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        sync();
    }
    if (sp.friction_iters > 0) solve_rows(FrictionRow{}, 1, sp.friction_iters);
    if (tol && tid == 0)
        tile_stats[t] = make_int4(used[0], used[1], (int)__float_as_uint(rfin[0]),
                                  (int)__float_as_uint(rfin[1]));
    store_velocities(tid, nt, bodies, nb, b0, linvel, angvel, vel);
}

// Scene tiles with a tolerance: sweeps used and final residuals over the
// tiles that had rows (maximum, and sums for the mean).
__global__ __launch_bounds__(256) void k_tile_summary(int n_tiles, const int4 *tile_stats,
                                                      int *counters) {
    __shared__ int smax[2], ssum[2], scnt;
    __shared__ unsigned int sres[2];
    if (threadIdx.x == 0) {
        smax[0] = smax[1] = 0; ssum[0] = ssum[1] = 0; scnt = 0; sres[0] = sres[1] = 0u;
    }
    __syncthreads();
    int mx0 = 0, mx1 = 0, sm0 = 0, sm1 = 0, cnt = 0;
    unsigned int r0 = 0u, r1 = 0u;
    for (int t = threadIdx.x; t < n_tiles; t += blockDim.x) {
        int4 st = tile_stats[t];
        if (st.x < 0) continue;
        mx0 = max(mx0, st.x); mx1 = max(mx1, st.y);
        sm0 += st.x; sm1 += st.y; cnt++;
        r0 = max(r0, (unsigned int)st.z); r1 = max(r1, (unsigned int)st.w);
    }
    atomicMax(&smax[0], mx0); atomicMax(&smax[1], mx1);
    atomicAdd(&ssum[0], sm0); atomicAdd(&ssum[1], sm1); atomicAdd(&scnt, cnt);
    atomicMax(&sres[0], r0); atomicMax(&sres[1], r1);
    __syncthreads();
    if (threadIdx.x == 0) {
        counters[RB_CNT_ITERS_N] = smax[0];
        counters[RB_CNT_ITERS_F] = smax[1];
        counters[RB_CNT_SUM_ITERS_N] = ssum[0];
        counters[RB_CNT_SUM_ITERS_F] = ssum[1];
        counters[RB_CNT_TILES_SOLVED] = scnt;
        counters[RB_CNT_RES_N] = (int)sres[0];
        counters[RB_CNT_RES_F] = (int)sres[1];
    }
}

// The largest residual over the tiles' places of one phase kind, by a
// workgroup of 256: every thread gets r = max scaled change / max(1, max impulse).
__device__ __forceinline__ float max_residual(const uint2 *__restrict__ res, int n_tiles) {
    __shared__ uint2 red[4];
    unsigned r = 0u, m = 0u;
    for (int t = threadIdx.x; t < n_tiles; t += 256) {
        const uint2 v = res[t];
        r = max(r, v.x);
        m = max(m, v.y);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        r = max(r, (unsigned)__shfl_xor((int)r, o));
        m = max(m, (unsigned)__shfl_xor((int)m, o));
    }
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = make_uint2(r, m);
    __syncthreads();
    r = max(max(red[0].x, red[1].x), max(red[2].x, red[3].x));
    m = max(max(red[0].y, red[1].y), max(red[2].y, red[3].y));
    const float lm = __uint_as_float(m);
    return __uint_as_float(r) / (lm > 1.f ? lm : 1.f);
}
// After a sweep (spatial tiles): decide convergence for the remaining sweeps.
__global__ __launch_bounds__(256) void k_sweep_done(const uint2 *__restrict__ tile_res, int n_tiles,
                                                    int is_friction, float tol, int *counters) {
    if (counters[RB_CNT_DONE] != 0) return;
    const float r = max_residual(tile_res + (is_friction ? n_tiles : 0), n_tiles);
    if (threadIdx.x != 0) return;
    int slot = is_friction ? RB_CNT_ITERS_F : RB_CNT_ITERS_N;
    counters[slot] += 1;
    ((float *)counters)[is_friction ? RB_CNT_RES_F : RB_CNT_RES_N] = r;
    if (tol > 0.f && r < tol) counters[RB_CNT_DONE] = 1;
}
__global__ void k_clear_done(int *counters) { counters[RB_CNT_DONE] = 0; }

// fixed sweep counts: iterations used and the last sweep's residual per phase
__global__ __launch_bounds__(256) void k_sweep_summary(const uint2 *__restrict__ tile_res,
                                                       int n_tiles, int nn, int nf, int *counters) {
    const float rn = max_residual(tile_res, n_tiles);
    const float rf = max_residual(tile_res + n_tiles, n_tiles);
    if (threadIdx.x != 0) return;
    counters[RB_CNT_ITERS_N] = nn;
    counters[RB_CNT_ITERS_F] = nf;
    float *f = (float *)counters;
    if (nn > 0) f[RB_CNT_RES_N] = rn;
    if (nf > 0) f[RB_CNT_RES_F] = rf;
}

// ---- integration ----
__global__ __launch_bounds__(256) void k_integrate(int n, float4 *__restrict__ pos,
                                                   float4 *__restrict__ quat,
                                                   const float4 *__restrict__ linvel,
                                                   float4 *__restrict__ angvel,
                                                   const float *__restrict__ inv_mass, float dt,
                                                   float damping, float max_ang) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 w = angvel[i];
    w.x *= damping; w.y *= damping; w.z *= damping;
    angvel[i] = w;
    float l2 = (w.x * w.x + w.y * w.y) + w.z * w.z;
    float ang = sqrtf(l2);
    if (ang * dt > max_ang) ang = max_ang / dt;
    float s;
    if (ang < 0.001f)
        s = 0.5f * dt - (((dt * dt * dt) * 0.020833333333f) * ang) * ang;
    else
        s = sinf((0.5f * ang) * dt) / ang;
    float ax = w.x * s, ay = w.y * s, az = w.z * s;
    float dw = cosf((ang * dt) * 0.5f);
    float4 q = quat[i];
    float rx = ((dw * q.x + ax * q.w) + ay * q.z) - az * q.y;
    float ry = ((dw * q.y + ay * q.w) + az * q.x) - ax * q.z;
    float rz = ((dw * q.z + az * q.w) + ax * q.y) - ay * q.x;
    float rw = ((dw * q.w - ax * q.x) - ay * q.y) - az * q.z;
    float len = sqrtf(((rx * rx + ry * ry) + rz * rz) + rw * rw);
    if (len > 0.f) {
        float inv = 1.f / len;
        q = mk4(rx * inv, ry * inv, rz * inv, rw * inv);
    } else {
        q = mk4(0.f, 0.f, 0.f, 1.f);
    }
    quat[i] = q;
    float4 v = linvel[i];
    float4 p = pos[i];
    p.x = p.x + v.x * dt;
    p.y = p.y + v.y * dt;
    p.z = p.z + v.z * dt;
    pos[i] = p;
    (void)inv_mass;
}

}  // namespace

// ---------------------------------------------------------------- launchers
hipError_t launch_constraints(const DeviceWorld &d, const StepParams &p, hipStream_t s) {
    int grid = (p.max_contacts + 255) / 256;
    RB_LAUNCH(k_constraints, dim3(grid), dim3(256), 0, s, p, d.contact_pair, d.contact_slots,
                       d.contacts, d.pos, d.linvel,
                       d.angvel, d.inv_mass, d.inv_inertia_world, d.scene, d.aabb_min, d.aabb_max,
                       d.cs, d.tile_kv, d.counters, d.prev_keys, d.prev_imp, d.prev_pts, d.prev_count,
                       d.features, d.solve_pos, d.pairs);
    return rb_launch_status();
}

hipError_t launch_tile_bounds(const DeviceWorld &d, const StepParams &p, hipStream_t s) {
    RB_LAUNCH(k_tile_bounds2, dim3((p.max_contacts + 255) / 256), dim3(256), 0, s,
                       d.tile_kv, d.counters, d.tile_first, d.tile_cnt);
    return rb_launch_status();
}

hipError_t launch_tiles(const DeviceWorld &d, const StepParams &p, hipStream_t s) {
    RB_LAUNCH(k_tile_color, dim3(p.n_tiles), dim3(TB), 0, s, d.tile_kv, d.tile_first,
                       d.tile_cnt, d.cs.bodies, d.inv_mass, d.solve_order, d.row_color,
                       d.tile_color_off, d.tile_ncolors, d.counters);
    RB_LAUNCH(k_tile_pack, dim3(p.n_tiles), dim3(TB), 0, s, d.tile_first, d.tile_cnt,
                       d.solve_order, d.row_color, d.cs, d.pos, d.inv_mass, d.inv_inertia_world,
                       d.pk, d.solve_pos, d.tile_bodies, d.tile_nb, d.tile_ncolors, d.tile_hdr,
                       d.counters, d.tile_res, p.tile_mode == 0 ? 1 : 0);
    return rb_launch_status();
}

namespace {
__global__ void k_tile_order_keys(int n_tiles, int max_class, const int4 *__restrict__ tile_hdr,
                                  uint2 *__restrict__ kv, int *counters) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    int lg = -1;
    if (t < n_tiles) {
        const int R = tile_hdr[t].y;
        const uint32_t r = (uint32_t)(R < 0 ? 0 : (R > 0xffff ? 0xffff : R));
        kv[t] = make_uint2(0xffffu - r, (uint32_t)t);
        lg = scene_class(R, max_class);
    }
    for (int c = 0; c < SCENE_CLASSES; c++) {
        const uint64_t m = __ballot(lg == c);
        if (m && (threadIdx.x & 63) == 0)
            atomicAdd(counters + RB_CNT_SCENES + c, (int)__popcll(m));
    }
}
}  // namespace

// log2 of the most scenes that share a workgroup: only as many as leave every
// CU a workgroup.  Steps in us with up to 1, 2 and 4 scenes a workgroup, 256
// CUs: scenes of 8 to 64 bodies, 10 + 10 sweeps, 257 of them 325, 336, 360; 300
// 344, 333, 359; 500 379, 359, 385; 1,100 532, 484, 481; scenes of 8 to 128
// bodies to a tolerance, 300 1,361, 1,479, 1,621; 500 1,636, 1,680, 1,838;
// 1,000 2,381, 1,901, 2,045; 1,500 3,351, 2,377, 2,016.  (From about 300 to 511
// scenes two would share at a gain of 3 to 6% with fixed sweeps, and at a loss
// of 3 to 9% to a tolerance, where a lone scene's chain is what counts.)
static int most_shared(const StepParams &p) {
    int lg = 0;
    while (lg < SCENE_CLASSES - 1 && p.n_tiles >> (lg + 1) >= rb_num_cus()) lg++;
    return lg;
}
bool solve_block_matters(const StepParams &p) { return p.tile_mode == 1 && most_shared(p) > 0; }

hipError_t launch_tile_order(const DeviceWorld &d, const StepParams &p, hipStream_t s,
                             const SortWork &sw) {
    if (p.tile_mode != 1) return hipSuccess;
    // (a tuned block of 512 threads gives every scene twice the threads)
    int max_class = most_shared(p);
    if (p.solve_block == 512 && max_class > 0) max_class--;
    RB_LAUNCH(k_tile_order_keys, dim3((p.n_tiles + 255) / 256), dim3(256), 0, s, p.n_tiles,
              max_class, d.tile_hdr, d.tile_order, d.counters);
    hipError_t e = rb_launch_status();
    if (e != hipSuccess) return e;
    // (the order is a schedule only: every scene is solved by itself, so
    // results do not depend on it)
    return launch_radix_sort(d.tile_order, p.n_tiles, 16, 8, sw, s);
}

hipError_t launch_solve(const DeviceWorld &d, const StepParams &p, hipStream_t s,
                        hipEvent_t *kev, int *n_launches, hipEvent_t *span) {
    const int S = p.normal_iters + p.friction_iters;
    const int warm = p.warm_start != MI_RB_WARM_ZERO;
    int nl = 0;
    if (span) hipEventRecord(span[0], s);
    auto mark = [&](int end) {
        if (kev) hipEventRecord(kev[2 * nl + end], s);
        if (end) nl++;
    };
    // (the step's first kernel has cleared the converged flag)
#define RB_SOLVE_ARGS \
    d.tile_hdr, d.tile_color_off, d.tile_bodies, d.pk, d.linvel, d.angvel, d.tile_res
    if (p.tile_mode == 1) {
        // independent scenes: every sweep of a scene in one workgroup; with a
        // tolerance each scene stops on its own residual
        mark(0);
        const SolveView sv{d.cs, d.solve_order, d.pos, d.inv_mass, d.inv_inertia_world, d.linvel,
                           d.angvel};
        // (a workgroup per scene at most: those beyond the classes' end at once)
        RB_LAUNCH(k_scene_solve, dim3(p.n_tiles), dim3(SCENE_TB), 0, s, p, warm, d.tile_hdr,
                  d.tile_color_off, d.tile_bodies, d.pk, sv, d.tile_res, d.tile_stats,
                  d.tile_order, d.counters);
        mark(1);
        if (p.tol > 0.f)
            RB_LAUNCH(k_tile_summary, dim3(1), dim3(256), 0, s, p.n_tiles, d.tile_stats,
                               d.counters);
        else
            RB_LAUNCH(k_sweep_summary, dim3(1), dim3(256), 0, s, d.tile_res, p.n_tiles,
                      p.normal_iters, p.friction_iters, d.counters);
    } else {
        for (int sw = warm ? -1 : 0; sw < S; sw++) {
            const bool fr = sw >= p.normal_iters, res = sw >= 0 && sweep_residual_needed(p, sw);
            for (int ph = 0; ph < 4; ph++) {
                int nx = (p.tiles_x - (ph & 1) + 1) / 2, nz = (p.tiles_z - (ph >> 1) + 1) / 2;
                if (nx <= 0 || nz <= 0) continue;
                mark(0);
                auto solve = [&](auto threads) {
                    constexpr int T = decltype(threads)::value;
                    auto kern = sw < 0 ? k_tile_solve<T, ROW_WARM, false>
                                : !fr  ? (res ? k_tile_solve<T, ROW_NORMAL, true>
                                              : k_tile_solve<T, ROW_NORMAL, false>)
                                       : (res ? k_tile_solve<T, ROW_FRICTION, true>
                                              : k_tile_solve<T, ROW_FRICTION, false>);
                    RB_LAUNCH(kern, dim3(nx * nz), dim3(T), 0, s, p, ph, RB_SOLVE_ARGS, d.counters);
                };
                if (p.tile_threads == 512) solve(std::integral_constant<int, 512>{});
                else solve(std::integral_constant<int, 256>{});
                mark(1);
            }
            if (sw >= 0 && p.tol > 0.f) {
                RB_LAUNCH(k_sweep_done, dim3(1), dim3(256), 0, s, d.tile_res, p.n_tiles, fr, p.tol,
                          d.counters);
                if (sw == p.normal_iters - 1)
                    RB_LAUNCH(k_clear_done, dim3(1), dim3(1), 0, s, d.counters);
            }
        }
        if (p.tol <= 0.f)
            RB_LAUNCH(k_sweep_summary, dim3(1), dim3(256), 0, s, d.tile_res, p.n_tiles,
                      p.normal_iters, p.friction_iters, d.counters);
    }
#undef RB_SOLVE_ARGS
    if (span) hipEventRecord(span[1], s);
    if (n_launches) *n_launches = nl;
    const bool staged = p.n_proxies > 0;
    RB_LAUNCH(k_save_prev, dim3((p.max_contacts + 255) / 256), dim3(256), 0, s,
                       d.counters, d.cs, d.solve_pos, d.pk.lam, d.pk.fric,
                       staged ? d.stage_keys : d.prev_keys, staged ? d.stage_imp : d.prev_imp,
                       staged ? d.stage_pts : d.prev_pts, d.prev_count, d.pairs);
    return rb_launch_status();
}

namespace {
// (key part, row) of every cache entry: y first, then x of the order so far
__global__ void k_cache_key_y(const int *counters, const int2 *keys, uint2 *kv) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < counters[RB_CNT_CONTACTS]) kv[k] = make_uint2((uint32_t)keys[k].y, (uint32_t)k);
}
__global__ void k_cache_key_x(const int *counters, const int2 *keys, uint2 *kv) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < counters[RB_CNT_CONTACTS]) kv[k].x = (uint32_t)keys[kv[k].y].x;
}
__global__ void k_cache_gather(const int *counters, const uint2 *kv, const int2 *keys,
                               const float4 *imp, const float4 *pts, int2 *out_keys,
                               float4 *out_imp, float4 *out_pts) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= counters[RB_CNT_CONTACTS]) return;
    const int src = (int)kv[k].y;
    out_keys[k] = keys[src];
    out_imp[k] = imp[src];
    for (int i = 0; i < 4; i++) out_pts[4 * (size_t)k + i] = pts[4 * (size_t)src + i];
}
}  // namespace

hipError_t launch_cache_order(const DeviceWorld &d, const StepParams &p, hipStream_t s,
                              const SortWork &sw) {
    if (p.n_proxies <= 0) return hipSuccess;
    // pair entries name bodies and compound/triangle proxies below n + proxies
    const uint32_t top = (uint32_t)(p.n_bodies + p.n_proxies);
    int bits = 1;
    while (bits < 32 && (top >> bits) != 0) bits++;
    const int grid = (p.max_contacts + 255) / 256;
    int *nc = d.counters + RB_CNT_CONTACTS;
    RB_LAUNCH(k_cache_key_y, dim3(grid), dim3(256), 0, s, d.counters, d.stage_keys,
                       d.tile_kv);
    hipError_t e = launch_radix_sort(d.tile_kv, p.max_contacts, bits, 8, sw, s, nc);
    if (e != hipSuccess) return e;
    RB_LAUNCH(k_cache_key_x, dim3(grid), dim3(256), 0, s, d.counters, d.stage_keys,
                       d.tile_kv);
    e = launch_radix_sort(d.tile_kv, p.max_contacts, bits, 8, sw, s, nc);
    if (e != hipSuccess) return e;
    RB_LAUNCH(k_cache_gather, dim3(grid), dim3(256), 0, s, d.counters, d.tile_kv,
                       d.stage_keys, d.stage_imp, d.stage_pts, d.prev_keys, d.prev_imp,
                       d.prev_pts);
    return rb_launch_status();
}

// Body transforms into a renderer's vertex buffer (copyTransformsToVBOKernel,
// opencl/broadphase_benchmark/broadphaseKernel.cl:236-247): float4 (x, y, z,
// 1) of body i at base + i, its quaternion at base + n + i.
__global__ __launch_bounds__(256) void k_copy_transforms(int n, const float4 *__restrict__ pos,
                                                         const float4 *__restrict__ quat,
                                                         float4 *__restrict__ dst) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 p = pos[i];
    dst[i] = make_float4(p.x, p.y, p.z, 1.f);
    dst[n + i] = quat[i];
}

hipError_t launch_copy_transforms(const DeviceWorld &d, int n, float4 *dst, hipStream_t s) {
    if (n == 0) return hipSuccess;
    RB_LAUNCH(k_copy_transforms, dim3((n + 255) / 256), dim3(256), 0, s, n, d.pos, d.quat,
                       dst);
    return rb_launch_status();
}

hipError_t launch_integrate(const DeviceWorld &d, const StepParams &p, hipStream_t s) {
    if (p.n_bodies == 0) return hipSuccess;
    RB_LAUNCH(k_integrate, dim3((p.n_bodies + 255) / 256), dim3(256), 0, s, p.n_bodies,
                       d.pos, d.quat, d.linvel, d.angvel, d.inv_mass, p.dt, p.damping, p.max_ang);
    return rb_launch_status();
}
