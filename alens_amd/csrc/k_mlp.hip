// k_mlp.hip -- learned warm start for the BBPGD solve (gfx950, BF16 MFMA with FP32 accumulation).
//
// Per constraint, 12 inputs (gap delta0, normal n, contact arm positions s_I / (L_I/2),
// s_J / (L_J/2), relative contact-point velocity of U_nc times dt, rod lengths L_I, L_J, previous-step
// gamma) are standardised and fed to 12 -> 64 -> 64 -> 64 -> 1 (SiLU hidden, softplus output);
// gamma0 = gscale * output.  Parameters live in one FP32 master array (layout kP*); the MFMA operands
// are the BF16 roundings of the master values.
//
// MFMA, inference, 16 inputs or samples: v_mfma_f32_16x16x16_bf16 (builtin ..._16x16x16bf16_1k).  Lane l holds
// A[l % 16][4 (l / 16) + i], B[4 (l / 16) + i][l % 16] and D[4 (l / 16) + i][l % 16], i = 0..3.
// Constraints run along N, so a layer's output tile (features along rows 4 (l / 16) + i, constraint
// l % 16) is already laid out as the next layer's B operand and stays in registers from layer to layer.
// MFMA, layers of 64 inputs in training: gfx950's v_mfma_f32_16x16x32_bf16 (lane l holds A[l % 16][k] and
// B[k][l % 16] for its eight k of 32, D as above).  Which k a lane's place holds is free as long as both operands
// agree, so a lane's four values of two result tiles are its eight of the next operand.
#include <algorithm>

#include "alens_dev.hpp"
#include "alens_internal.hpp"

namespace alens {

#define LAUNCH_CHECK()                                                                           \
    do {                                                                                         \
        hipError_t e_ = hipGetLastError();                                                       \
        if (e_ != hipSuccess) return HipErr{e_, "kernel launch", __FILE__, __LINE__};             \
    } while (0)

static inline unsigned nblk(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// round to nearest even
__device__ inline short f2bf(float f) { return __builtin_bit_cast(short, (__bf16)f); }

__device__ inline f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}
__device__ inline f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ inline __bf16 f2bf16(float f) { return (__bf16)f; }

__device__ inline float softplus(float o) { return o > 20.0f ? o : log1pf(__expf(o)); }
__device__ inline float sigmoidf(float o) { return 1.0f / (1.0f + __expf(-o)); }

// ------------------------------------------------------------------------------------------------
// raw features, 16 floats per constraint (12 used, 4 zero)
// ------------------------------------------------------------------------------------------------
__global__ void k_features(uint32_t m, uint32_t gs, const int32_t *__restrict__ cI, const int32_t *__restrict__ cJ,
                           const double *__restrict__ delta0, const double *__restrict__ geo,
                           const double *__restrict__ posI, const double *__restrict__ posJ,
                           const double *__restrict__ dir, const double *__restrict__ length,
                           const double *__restrict__ unc, const double2 *__restrict__ xprev, double dt,
                           float *__restrict__ X, const uint32_t *__restrict__ md) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= dcount(m, md)) return;
    const int32_t i = cI[k], j = cJ[k];
    const double n[3] = {geo[k], geo[(size_t)gs + k], geo[2 * (size_t)gs + k]};  // component-major, stride gs
    const double *pi = posI + 3 * (size_t)k, *pj = posJ + 3 * (size_t)k;
    const double *ti = dir + 3 * (size_t)i, *tj = dir + 3 * (size_t)j;
    const double Li = length[i], Lj = length[j];
    const double si = pi[0] * ti[0] + pi[1] * ti[1] + pi[2] * ti[2];
    const double sj = pj[0] * tj[0] + pj[1] * tj[1] + pj[2] * tj[2];
    const double *ui = unc + 6 * (size_t)i, *uj = unc + 6 * (size_t)j;
    double vr[3];
    // v + w x p at each contact point, I minus J
    vr[0] = (ui[0] + (ui[4] * pi[2] - ui[5] * pi[1])) - (uj[0] + (uj[4] * pj[2] - uj[5] * pj[1]));
    vr[1] = (ui[1] + (ui[5] * pi[0] - ui[3] * pi[2])) - (uj[1] + (uj[5] * pj[0] - uj[3] * pj[2]));
    vr[2] = (ui[2] + (ui[3] * pi[1] - ui[4] * pi[0])) - (uj[2] + (uj[3] * pj[1] - uj[4] * pj[0]));
    float *x = X + 16 * (size_t)k;
    x[0] = (float)delta0[k];
    x[1] = (float)n[0];
    x[2] = (float)n[1];
    x[3] = (float)n[2];
    x[4] = (float)(Li > 0.0 ? si / (0.5 * Li) : 0.0);
    x[5] = (float)(Lj > 0.0 ? sj / (0.5 * Lj) : 0.0);
    x[6] = (float)(vr[0] * dt);
    x[7] = (float)(vr[1] * dt);
    x[8] = (float)(vr[2] * dt);
    x[9] = (float)Li;
    x[10] = (float)Lj;
    x[11] = (float)(xprev ? xprev[k].x : 0.0);
    x[12] = 0.0f;
    x[13] = 0.0f;
    x[14] = 0.0f;
    x[15] = 0.0f;
}

HipErr launch_features(hipStream_t st, uint32_t m, uint32_t gs, const int32_t *cI, const int32_t *cJ, const double *delta0,
                       const double *geo, const double *posI, const double *posJ, const double *dir,
                       const double *length, const double *unc, const double2 *xprev, double dt, float *X,
                       const uint32_t *md) {
    if (m == 0) return hip_ok();
    k_features<<<nblk(m, 256), 256, 0, st>>>(m, gs, cI, cJ, delta0, geo, posI, posJ, dir, length, unc, xprev, dt, X,
                                             md);
    LAUNCH_CHECK();
    return hip_ok();
}

// ------------------------------------------------------------------------------------------------
// fused inference: 16 constraints per tile, one wave per tile, all layers in registers
// ------------------------------------------------------------------------------------------------
__device__ inline float silu(float z) { return z / (1.0f + __expf(-z)); }

// Bound by the vector units (48 exponentials and reciprocals per constraint and lane group).  A wave keeps the
// weights in registers and so takes many tiles: two blocks per CU, which share a tile's latency, fetch them 2,048
// times at most.  250,000 constraints: 44 us; with a wave per tile, up to 16,384, the 38 KB of weights of each set
// the pace: 98 us.
constexpr int kInferBlocks = 512;
template <typename OutT>
__global__ __launch_bounds__(256, 2) void k_mlp_infer(uint32_t m, const float *__restrict__ X,
                                                      const float *__restrict__ P, const float *__restrict__ norm,
                                                      OutT *__restrict__ out, int out_stride,
                                                      const uint32_t *__restrict__ md) {
    m = dcount(m, md);
    const int lane = threadIdx.x & 63;
    const int r16 = lane & 15, q = lane >> 4;
    const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
    const int64_t ntiles = ((int64_t)m + 15) / 16;
    if (wave >= ntiles) return;
    const float gscale = norm[2 * kMlpIn];
    // features 4 q .. 4 q + 3 of constraint r16 of a tile (past the end: of the last constraint)
    auto load = [&](int64_t t) {
        const int64_t c = t * 16 + r16;
        return *reinterpret_cast<const float4 *>(X + 16 * (size_t)(c < (int64_t)m ? c : (int64_t)m - 1) + 4 * q);
    };
    float4 x = load(wave);
    // A operands (weights, row = output unit, k = input unit) and biases for this lane
    bf16x4 a1[4], a2[4][4], a3[4][4];
    float b1v[4][4], b2v[4][4], b3v[4][4], w4v[4][4], mean[4], istd[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        mean[i] = q < 3 ? norm[4 * q + i] : 0.0f;
        istd[i] = q < 3 ? norm[kMlpIn + 4 * q + i] : 0.0f;
    }
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int oo = 16 * mt + 4 * q + i;
            a1[mt][i] = f2bf(P[kPW1 + (16 * mt + r16) * 16 + 4 * q + i]);
            b1v[mt][i] = P[kPB1 + oo];
            b2v[mt][i] = P[kPB2 + oo];
            b3v[mt][i] = P[kPB3 + oo];
            w4v[mt][i] = P[kPW4 + oo];
        }
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                a2[mt][kt][i] = f2bf(P[kPW2 + (16 * mt + r16) * 64 + 16 * kt + 4 * q + i]);
                a3[mt][kt][i] = f2bf(P[kPW3 + (16 * mt + r16) * 64 + 16 * kt + 4 * q + i]);
            }
    }
    const float b4 = P[kPB4];
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    for (int64_t t = wave; t < ntiles; t += nwaves) {
        const int64_t c = t * 16 + r16;
        const float xi[4] = {x.x, x.y, x.z, x.w};
        if (t + nwaves < ntiles) x = load(t + nwaves);
        bf16x4 bx;
#pragma unroll
        for (int i = 0; i < 4; ++i) bx[i] = f2bf(q < 3 ? (xi[i] - mean[i]) * istd[i] : 0.0f);
        bf16x4 h[4], h2[4];
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            const f32x4 z = mfma16(a1[mt], bx, zero);
#pragma unroll
            for (int i = 0; i < 4; ++i) h[mt][i] = f2bf(silu(z[i] + b1v[mt][i]));
        }
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            f32x4 z = zero;
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) z = mfma16(a2[mt][kt], h[kt], z);
#pragma unroll
            for (int i = 0; i < 4; ++i) h2[mt][i] = f2bf(silu(z[i] + b2v[mt][i]));
        }
        float part = 0.0f;
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            f32x4 z = zero;
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) z = mfma16(a3[mt][kt], h2[kt], z);
#pragma unroll
            for (int i = 0; i < 4; ++i) part += w4v[mt][i] * silu(z[i] + b3v[mt][i]);
        }
        part += __shfl_xor(part, 16, 64);
        part += __shfl_xor(part, 32, 64);
        if (c < (int64_t)m && q == 0) out[(size_t)c * out_stride] = (OutT)(gscale * softplus(part + b4));
    }
}

template <typename OutT>
static HipErr launch_infer(hipStream_t st, uint32_t m, const float *X, const float *P, const float *norm, OutT *out,
                           int stride, const uint32_t *md) {
    if (m == 0) return hip_ok();
    const int64_t blocks = std::min<int64_t>(kInferBlocks, ((int64_t)m + 63) / 64);
    k_mlp_infer<OutT><<<(unsigned)blocks, 256, 0, st>>>(m, X, P, norm, out, stride, md);
    LAUNCH_CHECK();
    return hip_ok();
}

HipErr launch_mlp_infer_f32(hipStream_t st, uint32_t m, const float *X, const float *P, const float *norm,
                            float *out) {
    return launch_infer<float>(st, m, X, P, norm, out, 1, nullptr);
}

// writes gamma0 into the x component of the solver state (double2 stride 2)
HipErr launch_mlp_infer_xg(hipStream_t st, uint32_t m, const float *X, const float *P, const float *norm,
                           double2 *xg, const uint32_t *md) {
    return launch_infer<double>(st, m, X, P, norm, reinterpret_cast<double *>(xg), 2, md);
}

// ------------------------------------------------------------------------------------------------
// training: loss and gradient of a batch in one pass
//
// One wave takes 16 samples through forward and backward pass in registers; nothing of a sample goes to memory.
// Every layer's result is wanted in two forms: samples along lanes (the next layer's operand) and units along
// lanes (the operands of the weight gradients, which contract over samples).  The operands of an MFMA have the
// same lane layout, so mfma(a, b) and mfma(b, a) are each other's transpose: the second form costs the same
// products again, on matrix cores that are otherwise idle, and no transposition.  Weight gradients stay in
// accumulators over all the wave's tiles; a block adds its four waves' in LDS and writes one partial gradient,
// k_mlp_update adds the blocks' in order (the result does not depend on scheduling).
//
// A batch of 4,096 is bound by latency: loading the operands, the chain of six layers, two launches.  Layer by
// layer through memory (35 launches, FP32 activations) it took 180 us, in this form 19 us and 4.6 us for the sum
// over the blocks with the Adam step.
// ------------------------------------------------------------------------------------------------
// Sigmoid-weighted unit and its slope.  The quotients 1 / e and z / e share one reciprocal, refined by Newton's
// iteration; a residual step of its own then corrects each.  Far below zero, where the reciprocal leaves the normal
// range, both are 0 (e is capped there, or its residuals would be undefined).
__device__ inline void silu2(float z, float &h, float &g) {
    const float e = fminf(1.0f + __expf(-z), 0x1p125f);
    float r = __builtin_amdgcn_rcpf(e);
    r = fmaf(fmaf(-e, r, 1.0f), r, r);
    r = z < -86.5f ? 0.0f : r;
    float s = fmaf(fmaf(-e, r, 1.0f), r, r);
    s = fmaf(fmaf(-e, s, 1.0f), r, s);
    h = z * r;
    h = fmaf(fmaf(-e, h, z), r, h);
    h = fmaf(fmaf(-e, h, z), r, h);
    g = s * (1.0f + z * (1.0f - s));
}
__device__ inline bf16x8 join(bf16x4 a, bf16x4 b) {
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    return __builtin_bit_cast(bf16x8, s16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]});
}
// The unit in row r of result tile mt.  A lane's rows 4 q .. 4 q + 3 of tiles 2 p and 2 p + 1 are units
// 32 p + 8 q .. 32 p + 8 q + 7: its eight values of the next operand, in their order.
__device__ inline int unit(int mt, int r) { return 32 * (mt >> 1) + 8 * (r >> 2) + 4 * (mt & 1) + (r & 3); }
// A lane's operand of inputs 32 p .. 32 p + 31 for 64 x 64 weights W, result tile mt (T: of W transposed).
__device__ inline bf16x8 weights(const float *W, int mt, int p, bool T) {
    const int lane = threadIdx.x & 63, o = unit(mt, lane & 15), k = 32 * p + 8 * (lane >> 4);
    bf16x8 v;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (__bf16)(T ? W[(k + i) * 64 + o] : W[o * 64 + k + i]);
    return v;
}

constexpr int kGradWaves = 4, kGradLoss = kMlpParams;  // a partial gradient's last element: the loss
static_assert(kMlpGradStride >= kMlpParams + 1, "a partial gradient and its loss");

__global__ __launch_bounds__(64 * kGradWaves) void k_mlp_grad(int B, const int32_t *__restrict__ idx,
                                                              const float *__restrict__ X, const float *__restrict__ t,
                                                              const float *__restrict__ P, const float *__restrict__ norm,
                                                              float *__restrict__ part) {
    // in the loop: the layers' weights in operand form, biases and output weights; then the waves' sums
    __shared__ __align__(16) float sum[kGradWaves * kMlpGradStride];
    const int lane = threadIdx.x & 63, r16 = lane & 15, q = lane >> 4, wv = threadIdx.x >> 6;
    // W2, W3 by output unit, then both by input unit
    bf16x8 *ops = reinterpret_cast<bf16x8 *>(sum);  // [matrix][mt][kp][lane]
    float *vec = sum + 4 * 4 * 2 * 64 * 4;          // b1, b2, b3, w4
#pragma unroll
    for (int z = 0; z < 8; ++z) {
        const int f = z * 4 + wv, mx = f >> 3, mt = (f >> 1) & 3, kp = f & 1;
        ops[f * 64 + lane] = weights(P + ((mx & 1) ? kPW3 : kPW2), mt, kp, mx >= 2);
    }
    vec[threadIdx.x] = P[(wv == 0 ? kPB1 : wv == 1 ? kPB2 : wv == 2 ? kPB3 : kPW4) + lane];
    bf16x4 a1[4];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) a1[mt][i] = f2bf(P[kPW1 + unit(mt, r16) * 16 + 4 * q + i]);
    __syncthreads();
    const float b4 = P[kPB4];
    float mean[4], istd[4];  // of features 4 q + i
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        mean[i] = q < 3 ? norm[4 * q + i] : 0.0f;
        istd[i] = q < 3 ? norm[kMlpIn + 4 * q + i] : 0.0f;
    }
    const float meanT = r16 < kMlpIn ? norm[r16] : 0.0f, istdT = r16 < kMlpIn ? norm[kMlpIn + r16] : 0.0f;

    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 d1[4], d2[4][4], d3[4][4];  // weight gradients: rows unit(mt, 4 q + i), columns unit(nt, r16)
    float db1[4], db2[4], db3[4], dw4[4], db4 = 0.0f, loss = 0.0f;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
        d1[mt] = zero;
        db1[mt] = db2[mt] = db3[mt] = dw4[mt] = 0.0f;
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) d2[mt][nt] = d3[mt][nt] = zero;
    }
    const int tiles = B / 16;
    for (int tile = blockIdx.x * kGradWaves + wv; tile < tiles; tile += gridDim.x * kGradWaves) {
        // (the lane index is formed anew for each tile, or the operands would be kept in registers across tiles)
        int ln = lane;
        asm volatile("" : "+v"(ln));
        auto op = [&](int mx, int mt, int kp) { return ops[(mx * 8 + mt * 2 + kp) * 64 + ln]; };
        auto along = [&](int v, int mt) { return *reinterpret_cast<const float4 *>(vec + v * 64 + unit(mt, 4 * (ln >> 4))); };
        auto vecT = [&](int v, int mt) { return vec[v * 64 + unit(mt, ln & 15)]; };
        // inputs; a sample's 16 floats are one line of memory
        const size_t s1 = (size_t)(idx ? idx[16 * tile + r16] : 16 * tile + r16);
        const float4 x = *reinterpret_cast<const float4 *>(X + 16 * s1 + 4 * q);
        const float tgt = t[s1];
        bf16x4 bx, xT;
        {
            const float xi[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const size_t s2 = (size_t)(idx ? idx[16 * tile + 4 * q + i] : 16 * tile + 4 * q + i);
                bx[i] = f2bf(q < 3 ? (xi[i] - mean[i]) * istd[i] : 0.0f);
                xT[i] = f2bf(r16 < kMlpIn ? (X[16 * s2 + r16] - meanT) * istdT : 0.0f);
            }
        }
        // forward: h (samples along lanes), hT (units along lanes) and the slopes the way back needs
        bf16x4 h1[4], h1T[4], h2[4], h2T[4];
        float g1T[4][4], g2[4][4], g2T[4][4], g3[4][4], g3T[4][4], h3T[4][4];
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            const f32x4 z = mfma16(a1[mt], bx, zero), zT = mfma16(bx, a1[mt], zero);
            const float bT = vecT(0, mt);
            const float4 b = along(0, mt);
            const float bi[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float h, g;
                silu2(z[i] + bi[i], h, g);
                h1[mt][i] = f2bf(h);
                silu2(zT[i] + bT, h, g1T[mt][i]);
                h1T[mt][i] = f2bf(h);
            }
        }
        bf16x8 o0 = join(h1[0], h1[1]), o1 = join(h1[2], h1[3]);
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            const bf16x8 w0 = op(0, mt, 0), w1 = op(0, mt, 1);
            const f32x4 z = mfma32(w1, o1, mfma32(w0, o0, zero));
            const f32x4 zT = mfma32(o1, w1, mfma32(o0, w0, zero));
            const float bT = vecT(1, mt);
            const float4 b = along(1, mt);
            const float bi[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float h;
                silu2(z[i] + bi[i], h, g2[mt][i]);
                h2[mt][i] = f2bf(h);
                silu2(zT[i] + bT, h, g2T[mt][i]);
                h2T[mt][i] = f2bf(h);
            }
        }
        o0 = join(h2[0], h2[1]);
        o1 = join(h2[2], h2[3]);
        float wh[4][4];
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            const bf16x8 w0 = op(1, mt, 0), w1 = op(1, mt, 1);
            const f32x4 z = mfma32(w1, o1, mfma32(w0, o0, zero));
            const f32x4 zT = mfma32(o1, w1, mfma32(o0, w0, zero));
            const float bT = vecT(2, mt);
            const float4 b = along(2, mt);
            const float bi[4] = {b.x, b.y, b.z, b.w};
            const float4 w = along(3, mt);
            const float wi[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float h;
                silu2(z[i] + bi[i], h, g3[mt][i]);
                wh[mt][i] = wi[i] * h;
                silu2(zT[i] + bT, h3T[mt][i], g3T[mt][i]);
            }
        }
        // head: loss (y - t)^2 / B and dO = 2 (y - t) / B sigmoid(o) of sample r16
        // (o: the units' products added to the bias one by one, handed from lane to lane)
        float o = b4;
#pragma unroll
        for (int z = 0; z < 8; ++z) {
            float s = o;
#pragma unroll
            for (int i = 0; i < 8; ++i) s += wh[2 * (z >> 2) + (i >> 2)][i & 3];
            o = __shfl(s, 16 * (z & 3) + r16, 64);
        }
        const float d = softplus(o) - tgt;
        const float dO = 2.0f * d / (float)B * sigmoidf(o);
        if (q == 0) {
            loss += d * d / (float)B;
            db4 += dO;
        }
        float dOT[4];  // of samples 4 q + i
#pragma unroll
        for (int i = 0; i < 4; ++i) dOT[i] = __shfl(dO, 4 * q + i, 64);
        // backward
        bf16x4 e[4], eT[4];
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            const float wT = vecT(3, mt);
            const float4 w = along(3, mt);
            const float wi[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                e[mt][i] = f2bf(wi[i] * dO * g3[mt][i]);
                const float dz = wT * dOT[i] * g3T[mt][i];
                eT[mt][i] = f2bf(dz);
                db3[mt] += dz;
                dw4[mt] += h3T[mt][i] * dOT[i];
            }
        }
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) d3[mt][nt] = mfma16(eT[mt], h2T[nt], d3[mt][nt]);
        o0 = join(e[0], e[1]);
        o1 = join(e[2], e[3]);
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            const bf16x8 w0 = op(3, mt, 0), w1 = op(3, mt, 1);
            const f32x4 z = mfma32(w1, o1, mfma32(w0, o0, zero));
            const f32x4 zT = mfma32(o1, w1, mfma32(o0, w0, zero));
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                e[mt][i] = f2bf(z[i] * g2[mt][i]);
                const float dz = zT[i] * g2T[mt][i];
                eT[mt][i] = f2bf(dz);
                db2[mt] += dz;
            }
        }
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) d2[mt][nt] = mfma16(eT[mt], h1T[nt], d2[mt][nt]);
        o0 = join(e[0], e[1]);
        o1 = join(e[2], e[3]);
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            const f32x4 zT = mfma32(o1, op(2, mt, 1), mfma32(o0, op(2, mt, 0), zero));
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float dz = zT[i] * g1T[mt][i];
                eT[mt][i] = f2bf(dz);
                db1[mt] += dz;
            }
            d1[mt] = mfma16(eT[mt], xT, d1[mt]);
        }
    }
    // the wave's sums into its part of LDS, the block's to memory
    __syncthreads();
    float *w = sum + wv * kMlpGradStride;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = unit(mt, 4 * q + i);
            w[kPW1 + row * 16 + r16] = d1[mt][i];
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) {
                w[kPW2 + row * 64 + unit(nt, r16)] = d2[mt][nt][i];
                w[kPW3 + row * 64 + unit(nt, r16)] = d3[mt][nt][i];
            }
        }
        auto over_q = [](float v) {
            v += __shfl_xor(v, 16, 64);
            return v + __shfl_xor(v, 32, 64);
        };
        const float v1 = over_q(db1[mt]), v2 = over_q(db2[mt]), v3 = over_q(db3[mt]), v4 = over_q(dw4[mt]);
        if (q == 0) {
            const int u = unit(mt, r16);
            w[kPB1 + u] = v1;
            w[kPB2 + u] = v2;
            w[kPB3 + u] = v3;
            w[kPW4 + u] = v4;
        }
    }
#pragma unroll
    for (int h = 32; h >= 1; h >>= 1) {
        db4 += __shfl_xor(db4, h, 64);
        loss += __shfl_xor(loss, h, 64);
    }
    if (lane == 0) {
        w[kPB4] = db4;
        w[kGradLoss] = loss;
    }
    __syncthreads();
    float *dst = part + (size_t)blockIdx.x * kMlpGradStride;
    for (int k = threadIdx.x; k <= kGradLoss; k += 64 * kGradWaves)
        dst[k] = ((sum[k] + sum[kMlpGradStride + k]) + sum[2 * kMlpGradStride + k]) + sum[3 * kMlpGradStride + k];
}

// Adam (Kingma & Ba 2015); W1 columns >= 12 stay zero
__device__ inline void adam(int i, float gi, float *P, float *m1, float *m2, const AdamStep &s) {
    if (i < kPB1 && (i % 16) >= kMlpIn) {
        P[i] = 0.0f;
        return;
    }
    const float a = s.b1 * m1[i] + (1.0f - s.b1) * gi;
    const float b = s.b2 * m2[i] + (1.0f - s.b2) * gi * gi;
    m1[i] = a;
    m2[i] = b;
    P[i] -= s.lr * (a / s.c1) / (sqrtf(b / s.c2) + s.eps);
}

// The gradient: blocks' partials added in a fixed order (64 elements a block, four lanes each take every fourth
// partial); with P the Adam step that follows, else the gradient itself to grad.
__global__ __launch_bounds__(256) void k_mlp_update(int np, const float *__restrict__ part, float *__restrict__ grad,
                                                    float *__restrict__ loss, float *__restrict__ P,
                                                    float *__restrict__ m1, float *__restrict__ m2, AdamStep s) {
    __shared__ float sh[4][64];
    const int e = threadIdx.x & 63, g = threadIdx.x >> 6, k = blockIdx.x * 64 + e;
    float v = 0.0f;
    if (k <= kGradLoss)
#pragma unroll 8
        for (int b = g; b < np; b += 4) v += part[(size_t)b * kMlpGradStride + k];
    sh[g][e] = v;
    __syncthreads();
    if (g != 0 || k > kGradLoss) return;
    v = ((sh[0][e] + sh[1][e]) + sh[2][e]) + sh[3][e];
    if (k == kGradLoss)
        *loss = v;
    else if (P)
        adam(k, v, P, m1, m2, s);
    else
        grad[k] = v;
}

__global__ void k_adam(float *__restrict__ P, const float *__restrict__ g, float *__restrict__ m1, float *__restrict__ m2,
                       AdamStep s) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kMlpParams) adam(i, g[i], P, m1, m2, s);
}

static AdamStep adam_of(float lr, int step) {
    const float b1 = 0.9f, b2 = 0.999f;
    return AdamStep{lr, b1, b2, 1e-8f, 1.0f - powf(b1, (float)step), 1.0f - powf(b2, (float)step)};
}

// one wave per SIMD at most: a wave's operands and accumulators take most of a SIMD's registers
static int grad_blocks(int B) { return std::max(1, std::min(kMlpGradBlocks, (B / 16 + kGradWaves - 1) / kGradWaves)); }

HipErr mlp_gradient(hipStream_t st, int B, const float *X, const float *t, const float *P, const float *norm, float *part,
                    float *grad, float *loss) {
    const int nb = grad_blocks(B);
    k_mlp_grad<<<nb, 64 * kGradWaves, 0, st>>>(B, nullptr, X, t, P, norm, part);
    LAUNCH_CHECK();
    k_mlp_update<<<nblk(kGradLoss + 1, 64), 256, 0, st>>>(nb, part, grad, loss, nullptr, nullptr, nullptr, AdamStep{});
    LAUNCH_CHECK();
    return hip_ok();
}

HipErr mlp_train_batch(hipStream_t st, int B, const int32_t *idx, const float *X, const float *t, float *P,
                       const float *norm, float *part, float *m1, float *m2, float lr, int step, float *loss) {
    const int nb = grad_blocks(B);
    k_mlp_grad<<<nb, 64 * kGradWaves, 0, st>>>(B, idx, X, t, P, norm, part);
    LAUNCH_CHECK();
    k_mlp_update<<<nblk(kGradLoss + 1, 64), 256, 0, st>>>(nb, part, nullptr, loss, P, m1, m2, adam_of(lr, step));
    LAUNCH_CHECK();
    return hip_ok();
}

HipErr mlp_adam_step(hipStream_t st, float *P, const float *grad, float *m1, float *m2, float lr, int step) {
    k_adam<<<nblk(kMlpParams, 256), 256, 0, st>>>(P, grad, m1, m2, adam_of(lr, step));
    LAUNCH_CHECK();
    return hip_ok();
}

}  // namespace alens
