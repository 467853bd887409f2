// k_mlp.hip -- learned warm start of the contact solver: an MLP 16-64-64-3
// that maps per-contact features to the contact's initial normal and two
// friction impulses.  No reference counterpart: the reference solver zeroes
// lambda every step (dynamics/basic_demo/Stubs/solverSetup.cl:529-531).
//
// Forward: BF16 MFMA (v_mfma_f32_16x16x16_bf16) with FP32 accumulation.  A
// wavefront takes 32 contacts at a time, two independent tiles of 16, and
// computes the layers transposed, H^T = W . X^T, so that the 16x16 accumulator
// of one layer (lane l holds rows 4*(l/16)+j, column l%16) is exactly the B
// operand layout of the next layer: activations never leave registers and the
// 5,312 weights stay resident in 48 VGPRs per lane for the whole grid-stride
// loop.
//
// Backward: the activations, inputs and weights are BF16 values already; the
// deltas are FP32 and stay so: each is split into three BF16 terms that add up
// to its 24 bits, so three BF16 MFMAs form exactly the products that one FP32
// MFMA would, at 5 times its rate, and add them in FP32.  A wave owns 32
// contacts of a tile from the forward pass to its weight gradients (one K = 32
// product over the contacts); it transposes what those need through its own
// part of LDS, with no barrier.  Each workgroup writes its partial gradients;
// one reduction kernel sums them in a fixed order (deterministic) and applies
// Adam to FP32 master weights, rounding the working copy to BF16.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "rb_internal.h"

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int NW1 = RB_MLP_H * RB_MLP_IN;   // 1024
constexpr int NW2 = RB_MLP_H * RB_MLP_H;    // 4096
constexpr int NW3 = RB_MLP_OUT * RB_MLP_H;  // 192
constexpr int NW = RB_MLP_NW;
constexpr int NB = RB_MLP_NB;
constexpr int PSTRIDE = NW + NB + 1;        // partial gradients + loss per workgroup
constexpr int MT = 128;                     // contacts per backward workgroup tile (32 a wave)
constexpr int GRAD_BLOCKS = 256;

__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
// two values rounded to bf16 (one instruction), the first in the low half
__device__ __forceinline__ uint32_t cvt2(float a, float b) {
    const bf16x2 v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ float lo_f(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float hi_f(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }
__device__ __forceinline__ bf16x8 vec8(uint2 a, uint2 b) {
    return __builtin_bit_cast(bf16x8, make_uint4(a.x, a.y, b.x, b.y));
}
__device__ __forceinline__ f32x4 mfma16(uint2 a, uint2 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(bf16x4, a),
                                                     __builtin_bit_cast(bf16x4, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 zero4() { f32x4 z = {0.f, 0.f, 0.f, 0.f}; return z; }
__device__ __forceinline__ uint2 load4(const uint16_t *p) {
    return *reinterpret_cast<const uint2 *>(p);
}

// Weights of one wavefront in MFMA A-operand layout: lane l (q = l / 16) holds
// row l % 16 of each 16-row block and the 4 consecutive inputs 16 * kb + 4 * q
// .. + 3.  Layer 3's rows repeat the 3 outputs, so that every q gets its
// contact's outputs.
struct MlpRegs {
    uint2 w1[4], w2[4][4], w3[4];
    f32x4 b1[4], b2[4], b3;
};

__device__ __forceinline__ void mlp_load(MlpRegs &m, const uint16_t *W, const float *B, int lane) {
    const int r = lane & 15, q = lane >> 4, o = r & 3;
#pragma unroll
    for (int mb = 0; mb < 4; mb++) m.w1[mb] = load4(W + (16 * mb + r) * RB_MLP_IN + 4 * q);
#pragma unroll
    for (int mb = 0; mb < 4; mb++)
#pragma unroll
        for (int kb = 0; kb < 4; kb++)
            m.w2[mb][kb] = load4(W + NW1 + (16 * mb + r) * RB_MLP_H + 16 * kb + 4 * q);
#pragma unroll
    for (int kb = 0; kb < 4; kb++) {
        const uint2 v =
            load4(W + NW1 + NW2 + (o < RB_MLP_OUT ? o : 0) * RB_MLP_H + 16 * kb + 4 * q);
        m.w3[kb] = o < RB_MLP_OUT ? v : make_uint2(0u, 0u);
    }
#pragma unroll
    for (int mb = 0; mb < 4; mb++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            m.b1[mb][j] = B[16 * mb + 4 * q + j];
            m.b2[mb][j] = B[RB_MLP_H + 16 * mb + 4 * q + j];
        }
#pragma unroll
    for (int j = 0; j < 4; j++) m.b3[j] = j < RB_MLP_OUT ? B[2 * RB_MLP_H + j] : 0.f;
}

// Forward pass of T tiles of 16 contacts.  x: this lane's features
// 4*(l/16)..+3 of contact l%16.  a1/a2: post-ReLU activations, lane l holding
// hidden units 16*mb + 4*(l/16) + j of contact l%16.  y: every lane holds
// outputs j = 0..2 of contact l%16.
template <int T>
__device__ __forceinline__ void mlp_tiles(const MlpRegs &m, const float4 x[T], f32x4 a1[T][4],
                                          f32x4 a2[T][4], f32x4 y[T]) {
    uint2 h[T][4];
    // bias, ReLU, and the bf16 values the next layer multiplies (the bias is
    // added to the sum: started from it, three times as many sums lay on the
    // other side of a bf16 rounding than in 64 bits)
    auto activate = [&](f32x4 a[4], const f32x4 b[4], uint2 ht[4]) {
#pragma unroll
        for (int mb = 0; mb < 4; mb++) {
#pragma unroll
            for (int j = 0; j < 4; j++) a[mb][j] = fmaxf(a[mb][j] + b[mb][j], 0.f);
            ht[mb] = make_uint2(cvt2(a[mb][0], a[mb][1]), cvt2(a[mb][2], a[mb][3]));
        }
    };
#pragma unroll
    for (int t = 0; t < T; t++) {
        const uint2 xb = make_uint2(cvt2(x[t].x, x[t].y), cvt2(x[t].z, x[t].w));
#pragma unroll
        for (int mb = 0; mb < 4; mb++) a1[t][mb] = mfma16(m.w1[mb], xb, zero4());
    }
#pragma unroll
    for (int t = 0; t < T; t++) activate(a1[t], m.b1, h[t]);
#pragma unroll
    for (int kb = 0; kb < 4; kb++)
#pragma unroll
        for (int mb = 0; mb < 4; mb++)
#pragma unroll
            for (int t = 0; t < T; t++)
                a2[t][mb] = mfma16(m.w2[mb][kb], h[t][kb], kb == 0 ? zero4() : a2[t][mb]);
#pragma unroll
    for (int t = 0; t < T; t++) activate(a2[t], m.b2, h[t]);
#pragma unroll
    for (int kb = 0; kb < 4; kb++)
#pragma unroll
        for (int t = 0; t < T; t++) y[t] = mfma16(m.w3[kb], h[t][kb], kb == 0 ? zero4() : y[t]);
#pragma unroll
    for (int t = 0; t < T; t++) y[t] += m.b3;
}

// Impulses from a prediction (network units are RB_MLP_SCALE x impulse):
// the predicted normal impulse, clamped at zero, is shared over the points in
// proportion to the impulses the constraint setup matched from the previous
// step (evenly over the points with a row when there are none).  Friction:
// a manifold with matched previous impulses keeps the previous step's
// friction impulses the setup gave it, others take the predicted ones; either
// is clamped to the cone of the predicted normal impulse.
__device__ __forceinline__ void apply_prediction(int k, float y0, float y1, float y2,
                                                 float friction, ConstraintSoA cs) {
    const float4 jac = cs.jac_inv[k], lp = cs.lambda[k];
    const float cnt = (float)((jac.x != 0.f) + (jac.y != 0.f) + (jac.z != 0.f) + (jac.w != 0.f));
    const float sum = ((lp.x + lp.y) + lp.z) + lp.w;
    float ln = y0 / RB_MLP_SCALE;
    ln = ln > 0.f ? ln : 0.f;
    const float jv[4] = {jac.x, jac.y, jac.z, jac.w}, pv[4] = {lp.x, lp.y, lp.z, lp.w};
    float lv[4];
    for (int i = 0; i < 4; i++) {
        if (jv[i] == 0.f) lv[i] = 0.f;
        else if (sum > 0.f) lv[i] = ln * (pv[i] / sum);
        else lv[i] = cnt > 0.f ? ln / cnt : 0.f;
    }
    cs.lambda[k] = make_float4(lv[0], lv[1], lv[2], lv[3]);
    float4 fr = cs.fric[k];
    float lim = friction * ln;
    float f0 = sum > 0.f ? fr.z : y1 / RB_MLP_SCALE, f1 = sum > 0.f ? fr.w : y2 / RB_MLP_SCALE;
    f0 = fminf(fmaxf(f0, -lim), lim);
    f1 = fminf(fmaxf(f1, -lim), lim);
    if (fr.x == 0.f) { f0 = 0.f; f1 = 0.f; }
    fr.z = f0;
    fr.w = f1;
    cs.fric[k] = fr;
}

// Forward over n contacts (n read from *n_dev when given).  APPLY: also set
// the constraints' initial impulses from the prediction.  The next 32 contacts'
// features load while these run.  Bound by its vector instructions (bias, ReLU
// and rounding of 2 x 128 sums a lane, 48 MFMA beside them).  582,217 contacts:
// 36.2 -> 19.9 us, of 8.7 us of memory traffic.
template <bool APPLY>
__global__ __launch_bounds__(256, 3) void k_mlp_forward(const float *__restrict__ x, int n,
                                                     const int *n_dev,
                                                     const uint16_t *__restrict__ W,
                                                     const float *__restrict__ B,
                                                     float *__restrict__ y, float friction,
                                                     ConstraintSoA cs) {
    if (n_dev) n = min(n, *n_dev);
    if (n <= 0) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, q = lane >> 4;
    const unsigned un = (unsigned)n, waves = gridDim.x * (blockDim.x >> 6);
    unsigned i = blockIdx.x * (blockDim.x >> 6) + wave;
    auto fetch = [&](unsigned c) {
        return c < un ? reinterpret_cast<const float4 *>(x)[4 * (size_t)c + q]
                     : make_float4(0.f, 0.f, 0.f, 0.f);
    };
    float4 xv[2] = {fetch(32 * i + r), fetch(32 * i + 16 + r)};
    MlpRegs m;
    mlp_load(m, W, B, lane);
    for (; 32 * i < un; i += waves) {
        const float4 xc[2] = {xv[0], xv[1]};
        xv[0] = fetch(32 * (i + waves) + r);
        xv[1] = fetch(32 * (i + waves) + 16 + r);
        f32x4 a1[2][4], a2[2][4], yv[2];
        mlp_tiles<2>(m, xc, a1, a2, yv);
        // lanes q = 0 and 1 store the two tiles
        const unsigned c = 32 * i + 16 * q + r;
        if (q < 2 && c < un) {
            const float y0 = q ? yv[1][0] : yv[0][0], y1 = q ? yv[1][1] : yv[0][1],
                        y2 = q ? yv[1][2] : yv[0][2];
            y[3 * (size_t)c] = y0;
            y[3 * (size_t)c + 1] = y1;
            y[3 * (size_t)c + 2] = y2;
            if (APPLY) apply_prediction((int)c, y0, y1, y2, friction, cs);
        }
    }
}

__device__ __forceinline__ uint32_t mix32(uint32_t k) {
    k ^= k >> 16; k *= 0x7feb352dU; k ^= k >> 15; k *= 0x846ca68bU; k ^= k >> 16;
    return k;
}

// One wave's transposes: per unit its bf16 values over the wave's 32 contacts
// (position 2 * r + t is contact 16 * t + r), rows of 80 B: 16-byte reads stay
// aligned and the four q of a write fall on different banks.
constexpr int TROW = 20;  // words
struct alignas(16) GradWave {
    uint32_t x[RB_MLP_IN][TROW];
    uint32_t a1[RB_MLP_H][TROW], a2[RB_MLP_H][TROW];
    uint32_t d[3][RB_MLP_H][TROW];  // a delta's three terms: of layer 2, then of layer 1
    uint32_t dy[3][RB_MLP_OUT][TROW];
};
constexpr int GRAD_ACC = 96;  // accumulator words per lane: 64 of W2, 16 of W1, 16 of W3
struct alignas(16) GradLDS {
    float w3[RB_MLP_OUT][RB_MLP_H];
    union {
        GradWave w[4];
        float acc[4][GRAD_ACC][64];
        struct {
            float b[4][2][RB_MLP_H][17];
            float b3[4][RB_MLP_OUT][17], loss[4][17];
        } s;
    };
};

// A pair of FP32 values as three pairs of bf16 whose sums are the values.
__device__ __forceinline__ void split3(float a, float b, uint32_t s[3]) {
    s[0] = cvt2(a, b);
    const float ra = a - lo_f(s[0]), rb = b - hi_f(s[0]);
    s[1] = cvt2(ra, rb);
    s[2] = cvt2(ra - lo_f(s[1]), rb - hi_f(s[1]));
}

// Gradients of loss = mean_s sum_o (y_o - t_o)^2 / 3 over a batch of n rows.
// Row i is sample i (sample_seed < 0) or a hashed draw from n_samples.
// Writes PSTRIDE partial sums per workgroup (weights, biases, sum of e^2).
// One wave a SIMD (its 440 registers hold all weights and accumulators).  A
// wave's 32 contacts take about 1,400 vector instructions, most of them to
// split and transpose, beside 168 MFMA (2,700 cycles), one after the other:
// what bounds it.  Batch of 65,536: 54.8 -> 24.0 us a launch (with FP32 MFMA
// and operands read down LDS columns, 16 lanes to a bank); error of the
// gradients against 64 bits, rms of 8 batches of 20,000: 3.3e-7 -> 2.0e-7.
__global__ __launch_bounds__(256, 1) void k_mlp_grad(const float *__restrict__ x,
                                                     const float *__restrict__ tgt, int n,
                                                     int n_samples, int sample_seed,
                                                     const uint16_t *__restrict__ W,
                                                     const float *__restrict__ B,
                                                     float *__restrict__ part) {
    __shared__ GradLDS L;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, tid = threadIdx.x;
    const int r = lane & 15, q = lane >> 4;
    // a tile's rows (16 * t + r of the wave's 32): features 4 * q .. + 3, targets
    const int ntiles = (n + MT - 1) / MT;
    float4 xn[2];
    float tn[2][RB_MLP_OUT];
    auto fetch = [&](int tile) {
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int row = tile * MT + 32 * wave + 16 * t + r;
            const bool valid = tile < ntiles && row < n;
            int s = row;
            if (sample_seed >= 0)
                s = (int)(mix32((uint32_t)row * 0x9e3779b9u ^ mix32((uint32_t)sample_seed)) %
                          (uint32_t)n_samples);
            xn[t] = valid ? reinterpret_cast<const float4 *>(x)[4 * (size_t)s + q]
                          : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int o = 0; o < RB_MLP_OUT; o++) tn[t][o] = valid ? tgt[3 * (size_t)s + o] : 0.f;
        }
    };
    fetch(blockIdx.x);
    MlpRegs m;
    mlp_load(m, W, B, lane);
    // W2^T as an A operand: row 16 * mb + r (hidden 1), K = hidden 2
    bf16x8 w2t[4][2];
#pragma unroll
    for (int mb = 0; mb < 4; mb++)
#pragma unroll
        for (int p = 0; p < 2; p++) {
            uint32_t u[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int k = 32 * p + 4 * q + (i & 1) * 2 + (i >> 1) * 16;
                const uint16_t *w = W + NW1 + k * RB_MLP_H + 16 * mb + r;
                u[i] = (uint32_t)w[0] | (uint32_t)w[RB_MLP_H] << 16;
            }
            w2t[mb][p] = __builtin_bit_cast(bf16x8, make_uint4(u[0], u[1], u[2], u[3]));
        }
    for (int i = tid; i < NW3; i += blockDim.x) (&L.w3[0][0])[i] = bf2f(W[NW1 + NW2 + i]);
    f32x4 gw2[4][4], gw1[4], gw3[4];
    f32x4 gb1[4], gb2[4];
    float gb3[RB_MLP_OUT] = {0.f, 0.f, 0.f}, lsum = 0.f;
#pragma unroll
    for (int mb = 0; mb < 4; mb++) {
        gw1[mb] = gw3[mb] = gb1[mb] = gb2[mb] = zero4();
#pragma unroll
        for (int nb = 0; nb < 4; nb++) gw2[mb][nb] = zero4();
    }
    const float dscale = 3.f * (float)n;
    __syncthreads();
    GradWave &G = L.w[wave];
    // (a wave's LDS operations are in order; the fences keep the compiler's)
    auto order = []() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };
    auto operand = [&](const uint32_t *row) {
        return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(row + 4 * q));
    };
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        // ---- forward of the wave's 32 rows; the next tile's rows load
        // while this one is worked on ----
        float4 xv[2];
        float tv[2][RB_MLP_OUT];
        bool valid[2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            valid[t] = tile * MT + 32 * wave + 16 * t + r < n;
            xv[t] = xn[t];
#pragma unroll
            for (int o = 0; o < RB_MLP_OUT; o++) tv[t][o] = tn[t][o];
        }
        fetch(tile + gridDim.x);
        f32x4 a1[2][4], a2[2][4], yv[2];
        mlp_tiles<2>(m, xv, a1, a2, yv);
        // ---- the transposes of the inputs and activations ----
        order();
        G.x[4 * q][r] = cvt2(xv[0].x, xv[1].x);
        G.x[4 * q + 1][r] = cvt2(xv[0].y, xv[1].y);
        G.x[4 * q + 2][r] = cvt2(xv[0].z, xv[1].z);
        G.x[4 * q + 3][r] = cvt2(xv[0].w, xv[1].w);
#pragma unroll
        for (int mb = 0; mb < 4; mb++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                G.a1[16 * mb + 4 * q + j][r] = cvt2(a1[0][mb][j], a1[1][mb][j]);
                G.a2[16 * mb + 4 * q + j][r] = cvt2(a2[0][mb][j], a2[1][mb][j]);
            }
        // ---- deltas at the outputs ----
        float dy[2][RB_MLP_OUT];
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int o = 0; o < RB_MLP_OUT; o++) {
                const float e = valid[t] ? yv[t][o] - tv[t][o] : 0.f;
                if (q == 0) lsum += e * e;
                dy[t][o] = 2.f * e / dscale;
                gb3[o] += dy[t][o];
            }
#pragma unroll
        for (int o = 0; o < RB_MLP_OUT; o++) {
            uint32_t s3[3];
            split3(dy[0][o], dy[1][o], s3);
            if (q == 0) {
                G.dy[0][o][r] = s3[0];
                G.dy[1][o][r] = s3[1];
                G.dy[2][o][r] = s3[2];
            }
        }
        // ---- layer 2's deltas: into LDS for the gradients, and as the B
        // operand (pairs of units of one contact) of layer 1's ----
        uint2 db[2][3][4];
#pragma unroll
        for (int mb = 0; mb < 4; mb++) {
            uint32_t s3[4][3];
            const int u = 16 * mb + 4 * q;
            const f32x4 w0 = *reinterpret_cast<const f32x4 *>(&L.w3[0][u]),
                        w1 = *reinterpret_cast<const f32x4 *>(&L.w3[1][u]),
                        w2 = *reinterpret_cast<const f32x4 *>(&L.w3[2][u]);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float d[2];
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const float v = (dy[t][0] * w0[j] + dy[t][1] * w1[j]) + dy[t][2] * w2[j];
                    d[t] = a2[t][mb][j] > 0.f ? v : 0.f;
                }
                gb2[mb][j] += d[0] + d[1];
                split3(d[0], d[1], s3[j]);
#pragma unroll
                for (int k = 0; k < 3; k++) G.d[k][u + j][r] = s3[j][k];
            }
#pragma unroll
            for (int k = 0; k < 3; k++) {
                db[0][k][mb] = make_uint2(__builtin_amdgcn_perm(s3[1][k], s3[0][k], 0x05040100u),
                                          __builtin_amdgcn_perm(s3[3][k], s3[2][k], 0x05040100u));
                db[1][k][mb] = make_uint2(__builtin_amdgcn_perm(s3[1][k], s3[0][k], 0x07060302u),
                                          __builtin_amdgcn_perm(s3[3][k], s3[2][k], 0x07060302u));
            }
        }
        order();
        // ---- dW2 (64 x 64) and dW3 (64 x 3, transposed) over the 32 rows ----
        {
            bf16x8 bv[4];
#pragma unroll
            for (int nb = 0; nb < 4; nb++) bv[nb] = operand(G.a1[16 * nb + r]);
#pragma unroll
            for (int k = 2; k >= 0; k--)
#pragma unroll
                for (int mb = 0; mb < 4; mb++) {
                    const bf16x8 av = operand(G.d[k][16 * mb + r]);
#pragma unroll
                    for (int nb = 0; nb < 4; nb++) gw2[mb][nb] = mfma32(av, bv[nb], gw2[mb][nb]);
                }
#pragma unroll
            for (int mb = 0; mb < 4; mb++) bv[mb] = operand(G.a2[16 * mb + r]);
#pragma unroll
            for (int k = 2; k >= 0; k--) {
                const bf16x8 yk = operand(G.dy[k][r < RB_MLP_OUT ? r : 0]);
                const bf16x8 zk = r < RB_MLP_OUT ? yk : vec8(make_uint2(0u, 0u), make_uint2(0u, 0u));
#pragma unroll
                for (int mb = 0; mb < 4; mb++) gw3[mb] = mfma32(bv[mb], zk, gw3[mb]);
            }
        }
        // ---- layer 1's deltas, masked by its ReLU ----
        f32x4 d1[2][4];
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int mb = 0; mb < 4; mb++) d1[t][mb] = zero4();
#pragma unroll
        for (int k = 2; k >= 0; k--)
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int mb = 0; mb < 4; mb++)
#pragma unroll
                    for (int t = 0; t < 2; t++)
                        d1[t][mb] = mfma32(w2t[mb][p], vec8(db[t][k][2 * p], db[t][k][2 * p + 1]),
                                           d1[t][mb]);
        order();
#pragma unroll
        for (int mb = 0; mb < 4; mb++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float u = a1[0][mb][j] > 0.f ? d1[0][mb][j] : 0.f;
                const float v = a1[1][mb][j] > 0.f ? d1[1][mb][j] : 0.f;
                gb1[mb][j] += u + v;
                uint32_t s3[3];
                split3(u, v, s3);
#pragma unroll
                for (int k = 0; k < 3; k++) G.d[k][16 * mb + 4 * q + j][r] = s3[k];
            }
        order();
        // ---- dW1 (64 x 16) ----
        const bf16x8 xo = operand(G.x[r]);
#pragma unroll
        for (int k = 2; k >= 0; k--)
#pragma unroll
            for (int mb = 0; mb < 4; mb++)
                gw1[mb] = mfma32(operand(G.d[k][16 * mb + r]), xo, gw1[mb]);
    }
    // ---- the workgroup's sums: weights, then biases and loss ----
    float *P = part + (size_t)blockIdx.x * PSTRIDE;
    __syncthreads();
#pragma unroll
    for (int mb = 0; mb < 4; mb++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
#pragma unroll
            for (int nb = 0; nb < 4; nb++) L.acc[wave][(4 * mb + nb) * 4 + j][lane] = gw2[mb][nb][j];
            L.acc[wave][64 + 4 * mb + j][lane] = gw1[mb][j];
            L.acc[wave][80 + 4 * mb + j][lane] = gw3[mb][j];
        }
    __syncthreads();
    for (int k = wave; k < GRAD_ACC; k += 4) {
        const float v = ((L.acc[0][k][lane] + L.acc[1][k][lane]) + L.acc[2][k][lane]) + L.acc[3][k][lane];
        if (k < 64) {
            const int mb = k >> 4, nb = (k >> 2) & 3, j = k & 3;
            P[NW1 + (16 * mb + 4 * q + j) * RB_MLP_H + 16 * nb + r] = v;
        } else if (k < 80) {
            P[(16 * ((k - 64) >> 2) + 4 * q + (k & 3)) * RB_MLP_IN + r] = v;
        } else if (r < RB_MLP_OUT) {  // (dW3 transposed: row = hidden unit, column = output)
            P[NW1 + NW2 + r * RB_MLP_H + 16 * ((k - 80) >> 2) + 4 * q + (k & 3)] = v;
        }
    }
    __syncthreads();
#pragma unroll
    for (int mb = 0; mb < 4; mb++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            L.s.b[wave][0][16 * mb + 4 * q + j][r] = gb1[mb][j];
            L.s.b[wave][1][16 * mb + 4 * q + j][r] = gb2[mb][j];
        }
    if (q == 0) {
        for (int o = 0; o < RB_MLP_OUT; o++) L.s.b3[wave][o][r] = gb3[o];
        L.s.loss[wave][r] = lsum;
    }
    __syncthreads();
    if (tid <= NB) {
        float v = 0.f;
        for (int w = 0; w < 4; w++) {
            const float *row = tid < 2 * RB_MLP_H ? L.s.b[w][tid >> 6][tid & 63]
                               : tid < NB         ? L.s.b3[w][tid - 2 * RB_MLP_H]
                                                  : L.s.loss[w];
            float u = 0.f;
            for (int i = 0; i < 16; i++) u += row[i];
            v += u;
        }
        P[NW + tid] = v;
    }
}

struct AdamArgs {
    float lr_t;      // lr * sqrt(1 - beta2^t) / (1 - beta1^t)
    float beta1, beta2, eps;
    int step;        // index into the loss history
};

// Sum the workgroup partials (fixed order) and, with master != null, take one
// Adam step.  grad/loss outputs are optional.  A workgroup sums 64 parameters,
// each wave every 16th partial with its loads in flight together, then the 16
// sums in order (256 partials: 61.2 -> 4.9 us against a thread per parameter).
constexpr int RED_WAVES = 16;
__global__ __launch_bounds__(64 * RED_WAVES) void k_mlp_reduce_adam(
    const float *__restrict__ part, int nblk, int n, float *grad, float *loss, float *master,
    float *mom, float *vel, uint16_t *W, float *B, AdamArgs a) {
    __shared__ float s[RED_WAVES][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int p = blockIdx.x * 64 + lane;
    float v[GRAD_BLOCKS / RED_WAVES];
#pragma unroll
    for (int i = 0; i < GRAD_BLOCKS / RED_WAVES; i++) {
        const int b = wave + RED_WAVES * i;
        v[i] = b < nblk && p < PSTRIDE ? part[(size_t)b * PSTRIDE + p] : 0.f;
    }
    float u = 0.f;
#pragma unroll
    for (int i = 0; i < GRAD_BLOCKS / RED_WAVES; i++) u += v[i];
    s[wave][lane] = u;
    __syncthreads();
    if (wave != 0 || p >= PSTRIDE) return;
    float g = 0.f;
#pragma unroll
    for (int w = 0; w < RED_WAVES; w++) g += s[w][lane];
    if (p == NW + NB) {
        if (loss) loss[a.step] = g / (3.f * (float)n);
        return;
    }
    if (grad) grad[p] = g;
    if (!master) return;
    float mm = a.beta1 * mom[p] + (1.f - a.beta1) * g;
    float vv = a.beta2 * vel[p] + (1.f - a.beta2) * g * g;
    mom[p] = mm;
    vel[p] = vv;
    float th = master[p] - a.lr_t * mm / (sqrtf(vv) + a.eps);
    master[p] = th;
    if (p < NW) W[p] = f2bf(th);
    else B[p - NW] = th;
}

// Training pairs of the last step: features and the solved impulses in
// network units (sum of normal lambdas, friction 0, friction 1).
__global__ __launch_bounds__(256) void k_mlp_targets(const int *counters, ConstraintSoA cs,
                                                     const float *__restrict__ features,
                                                     int capacity, float *__restrict__ x_out,
                                                     float *__restrict__ t_out) {
    int n = counters[RB_CNT_CONTACTS];
    if (n > capacity) n = capacity;
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const float4 *fi = reinterpret_cast<const float4 *>(features) + 4 * (size_t)k;
    float4 *fo = reinterpret_cast<float4 *>(x_out) + 4 * (size_t)k;
    fo[0] = fi[0]; fo[1] = fi[1]; fo[2] = fi[2]; fo[3] = fi[3];
    float4 l = cs.lambda[k], f = cs.fric[k];
    t_out[3 * (size_t)k] = (((l.x + l.y) + l.z) + l.w) * RB_MLP_SCALE;
    t_out[3 * (size_t)k + 1] = f.z * RB_MLP_SCALE;
    t_out[3 * (size_t)k + 2] = f.w * RB_MLP_SCALE;
}

int forward_grid(int n) {
    int waves = (n + 31) / 32;
    int blocks = (waves + 3) / 4;
    int cap = rb_num_cus() * 3;  // what the chip holds at once: the weights are loaded once a wave
    return blocks < 1 ? 1 : (blocks > cap ? cap : blocks);
}

}  // namespace

hipError_t launch_mlp_warm(const DeviceWorld &d, const StepParams &p, hipStream_t s) {
    RB_LAUNCH(k_mlp_forward<true>, dim3(forward_grid(p.max_contacts)), dim3(256), 0, s,
                       d.features, p.max_contacts, d.counters + RB_CNT_CONTACTS, d.mlp_w, d.mlp_b,
                       d.mlp_out, p.friction, d.cs);
    return rb_launch_status();
}

hipError_t launch_mlp_targets(const DeviceWorld &d, int capacity, float *x_out, float *t_out,
                              hipStream_t s) {
    RB_LAUNCH(k_mlp_targets, dim3((capacity + 255) / 256), dim3(256), 0, s, d.counters,
                       d.cs, d.features, capacity, x_out, t_out);
    return rb_launch_status();
}

// ---- C ABI: a network handle (weights, Adam state, scratch) ----
struct MlpHandle {
    int device = 0;
    hipStream_t stream = nullptr;
    uint16_t *w = nullptr;   // bf16 working weights
    float *b = nullptr;      // fp32 biases
    float *master = nullptr; // fp32 master copy of weights and biases (NW + NB)
    float *mom = nullptr, *vel = nullptr;
    float *part = nullptr;   // GRAD_BLOCKS x PSTRIDE
    float *loss = nullptr;   // per-step loss history
    int loss_cap = 0;
    int adam_t = 0;
};

static mi_rb_status mlp_upload(MlpHandle *h, const uint16_t *w_bf16, const float *bias) {
    std::vector<float> master(NW + NB);
    for (int i = 0; i < NW; i++) {
        uint32_t u = (uint32_t)w_bf16[i] << 16;
        std::memcpy(&master[i], &u, 4);
    }
    for (int i = 0; i < NB; i++) master[NW + i] = bias[i];
    RB_CHECK(hipMemcpyAsync(h->w, w_bf16, 2 * (size_t)NW, hipMemcpyHostToDevice, h->stream));
    RB_CHECK(hipMemcpyAsync(h->b, bias, 4 * (size_t)NB, hipMemcpyHostToDevice, h->stream));
    RB_CHECK(hipMemcpyAsync(h->master, master.data(), 4 * (size_t)(NW + NB), hipMemcpyHostToDevice,
                            h->stream));
    RB_CHECK(hipMemsetAsync(h->mom, 0, 4 * (size_t)(NW + NB), h->stream));
    RB_CHECK(hipMemsetAsync(h->vel, 0, 4 * (size_t)(NW + NB), h->stream));
    RB_CHECK(hipStreamSynchronize(h->stream));
    h->adam_t = 0;
    return MI_RB_OK;
}

extern "C" mi_rb_status mi_rb_mlp_create(uint64_t seed, void **out) {
    if (!out) return MI_RB_INVALID_ARG;
    *out = nullptr;
    MlpHandle *h = new MlpHandle();
    hipGetDevice(&h->device);
    mi_rb_status st = MI_RB_OK;
    auto fail = [&](hipError_t e) {
        if (e != hipSuccess && st == MI_RB_OK) st = rb_device_error(e, "mlp alloc", __FILE__, __LINE__);
    };
    fail(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
    fail(hipMalloc(&h->w, 2 * (size_t)NW));
    fail(hipMalloc(&h->b, 4 * (size_t)NB));
    fail(hipMalloc(&h->master, 4 * (size_t)(NW + NB)));
    fail(hipMalloc(&h->mom, 4 * (size_t)(NW + NB)));
    fail(hipMalloc(&h->vel, 4 * (size_t)(NW + NB)));
    fail(hipMalloc(&h->part, 4 * (size_t)GRAD_BLOCKS * PSTRIDE));
    if (st != MI_RB_OK) {
        mi_rb_mlp_destroy(h);
        return st;
    }
    // He-uniform initial weights from a seeded 64-bit LCG, zero biases
    std::vector<uint16_t> w(NW);
    std::vector<float> bias(NB, 0.f);
    uint64_t x = seed * 6364136223846793005ull + 1442695040888963407ull;
    auto uni = [&]() {
        x = x * 6364136223846793005ull + 1442695040888963407ull;
        return (float)((x >> 40) * (1.0 / 16777216.0)) * 2.f - 1.f;
    };
    auto host_bf = [](float f) {
        uint32_t u;
        std::memcpy(&u, &f, 4);
        return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
    };
    for (int i = 0; i < NW; i++) {
        int fan_in = i < NW1 ? RB_MLP_IN : RB_MLP_H;
        float lim = std::sqrt(6.f / (float)fan_in);
        if (i >= NW1 + NW2) lim = std::sqrt(3.f / (float)fan_in);
        w[i] = host_bf(uni() * lim);
    }
    st = mlp_upload(h, w.data(), bias.data());
    if (st != MI_RB_OK) {
        mi_rb_mlp_destroy(h);
        return st;
    }
    *out = h;
    return MI_RB_OK;
}

extern "C" void mi_rb_mlp_destroy(void *handle) {
    MlpHandle *h = static_cast<MlpHandle *>(handle);
    if (!h) return;
    if (h->stream) hipStreamSynchronize(h->stream);
    hipFree(h->w); hipFree(h->b); hipFree(h->master); hipFree(h->mom); hipFree(h->vel);
    hipFree(h->part); hipFree(h->loss);
    if (h->stream) hipStreamDestroy(h->stream);
    delete h;
}

extern "C" mi_rb_status mi_rb_mlp_set_weights(void *handle, const uint16_t *w_bf16,
                                              const float *bias) {
    MlpHandle *h = static_cast<MlpHandle *>(handle);
    if (!h || !w_bf16 || !bias) return MI_RB_INVALID_ARG;
    return mlp_upload(h, w_bf16, bias);
}

extern "C" mi_rb_status mi_rb_mlp_get_weights(void *handle, uint16_t *w_bf16, float *bias) {
    MlpHandle *h = static_cast<MlpHandle *>(handle);
    if (!h || !w_bf16 || !bias) return MI_RB_INVALID_ARG;
    RB_CHECK(hipMemcpyAsync(w_bf16, h->w, 2 * (size_t)NW, hipMemcpyDeviceToHost, h->stream));
    RB_CHECK(hipMemcpyAsync(bias, h->b, 4 * (size_t)NB, hipMemcpyDeviceToHost, h->stream));
    RB_CHECK(hipStreamSynchronize(h->stream));
    return MI_RB_OK;
}

extern "C" mi_rb_status mi_rb_mlp_forward(void *handle, const float *x_dev, int n, float *y_dev) {
    MlpHandle *h = static_cast<MlpHandle *>(handle);
    if (!h || n < 0 || (n > 0 && (!x_dev || !y_dev))) return MI_RB_INVALID_ARG;
    if (n == 0) return MI_RB_OK;
    ConstraintSoA none{};
    RB_LAUNCH(k_mlp_forward<false>, dim3(forward_grid(n)), dim3(256), 0, h->stream, x_dev,
                       n, (const int *)nullptr, h->w, h->b, y_dev, 0.f, none);
    RB_CHECK(rb_launch_status());
    RB_CHECK(hipStreamSynchronize(h->stream));
    return MI_RB_OK;
}

static int grad_blocks(int n) {
    int tiles = (n + MT - 1) / MT;
    return tiles < GRAD_BLOCKS ? (tiles < 1 ? 1 : tiles) : GRAD_BLOCKS;
}

extern "C" mi_rb_status mi_rb_mlp_gradients(void *handle, const float *x_dev, const float *t_dev,
                                            int n, float *grad_dev, float *loss) {
    MlpHandle *h = static_cast<MlpHandle *>(handle);
    if (!h || n <= 0 || !x_dev || !t_dev || !grad_dev) return MI_RB_INVALID_ARG;
    if (h->loss_cap < 1) {
        hipFree(h->loss);
        h->loss = nullptr;
        RB_CHECK(hipMalloc(&h->loss, sizeof(float)));
        h->loss_cap = 1;
    }
    int nb = grad_blocks(n);
    RB_LAUNCH(k_mlp_grad, dim3(nb), dim3(256), 0, h->stream, x_dev, t_dev, n, n, -1, h->w,
                       h->b, h->part);
    AdamArgs a{0.f, 0.f, 0.f, 0.f, 0};
    RB_LAUNCH(k_mlp_reduce_adam, dim3((PSTRIDE + 63) / 64), dim3(64 * RED_WAVES), 0, h->stream,
                       h->part, nb, n, grad_dev, h->loss, (float *)nullptr, (float *)nullptr,
                       (float *)nullptr, (uint16_t *)nullptr, (float *)nullptr, a);
    RB_CHECK(rb_launch_status());
    float l = 0.f;
    RB_CHECK(hipMemcpyAsync(&l, h->loss, sizeof(float), hipMemcpyDeviceToHost, h->stream));
    RB_CHECK(hipStreamSynchronize(h->stream));
    if (loss) *loss = l;
    return MI_RB_OK;
}

extern "C" mi_rb_status mi_rb_mlp_train(void *handle, const float *x_dev, const float *t_dev,
                                        int n_samples, int batch, int steps, float lr, int seed,
                                        float *loss_history) {
    MlpHandle *h = static_cast<MlpHandle *>(handle);
    if (!h || n_samples <= 0 || batch <= 0 || steps < 0 || !x_dev || !t_dev || !(lr > 0.f))
        return MI_RB_INVALID_ARG;
    // seed < 0: every step takes rows 0..batch-1 in order (full-batch steps)
    if (seed < 0 && batch > n_samples) return MI_RB_INVALID_ARG;
    if (steps == 0) return MI_RB_OK;
    if (h->loss_cap < steps) {
        hipFree(h->loss);
        h->loss = nullptr;
        RB_CHECK(hipMalloc(&h->loss, sizeof(float) * (size_t)steps));
        h->loss_cap = steps;
    }
    const float b1 = 0.9f, b2 = 0.999f;
    int nb = grad_blocks(batch);
    for (int i = 0; i < steps; i++) {
        h->adam_t++;
        double c1 = 1.0 - std::pow((double)b1, h->adam_t), c2 = 1.0 - std::pow((double)b2, h->adam_t);
        AdamArgs a{(float)(lr * std::sqrt(c2) / c1), b1, b2, 1e-8f, i};
        int draw_seed =
            seed < 0 ? -1 : (int)(((uint32_t)seed * 0x9e3779b9u + (uint32_t)h->adam_t) & 0x7fffffffu);
        RB_LAUNCH(k_mlp_grad, dim3(nb), dim3(256), 0, h->stream, x_dev, t_dev, batch,
                           n_samples, draw_seed, h->w, h->b, h->part);
        RB_LAUNCH(k_mlp_reduce_adam, dim3((PSTRIDE + 63) / 64), dim3(64 * RED_WAVES), 0, h->stream,
                           h->part, nb, batch, (float *)nullptr, h->loss, h->master, h->mom, h->vel,
                           h->w, h->b, a);
    }
    RB_CHECK(rb_launch_status());
    if (loss_history)
        RB_CHECK(hipMemcpyAsync(loss_history, h->loss, sizeof(float) * (size_t)steps,
                                hipMemcpyDeviceToHost, h->stream));
    RB_CHECK(hipStreamSynchronize(h->stream));
    return MI_RB_OK;
}
