// Training and evaluation of the far-field model of mlp.h: forward, backward and Adam,
// hand-written on BF16 MFMA (v_mfma_f32_16x16x16_bf16) with FP32 accumulation.
//
// Loss: L = (1/N) sum_s sum_o (y_so - t_so)^2 over the N samples of a batch.
// k_mlp_grad  16 waves per 64 samples: forward (activations in LDS, pre-activations in registers),
//             backward through the layers (dH = W^T dZ on MFMA with the transposed
//             weights as A), weight gradients dW = dZ^T H on MFMA with the samples as the K
//             dimension, bias gradients by lane reductions; writes its partial gradient
// k_mlp_reduce  sums the partial gradients of the workgroups in a fixed order (deterministic)
// k_adam      the same sums, and an Adam step on the FP32 master parameters
// k_mlp_eval  inference, four waves per workgroup sharing the BF16 weights
#include <math.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "bl_internal.h"
#include "mlp.h"

namespace bl {
namespace {

constexpr int NP1 = MLP_NPARAM + 1;  // parameters + the loss sum

// A workgroup's weights and activations in LDS, rows padded by 4 so that the 8-byte fragments of 16
// rows fall in different banks; what a contraction over the samples reads is kept by unit as well.
constexpr int LH = MLP_H + 4, LX = 16 + 4;
struct GradLds {
    short w1[MLP_H * LX];              // [64][16], inputs 8..15 zero
    short w2[MLP_H * LH], w3[MLP_H * LH];
    short w4[16 * LH];                 // [16][64], outputs 2..15 zero
    short w2t[MLP_H * LH], w3t[MLP_H * LH];  // W2^T, W3^T: rows = input units
    short w4t[MLP_H * LX];             // W4^T [64][16], columns 2..15 zero
    float b1[MLP_H], b2[MLP_H], b3[MLP_H], b4[4];
    short x[64 * LX], xt[16 * LH];     // inputs by sample, by input
    short h[3][64 * LH], ht[3][MLP_H * LH];  // H1, H2, H3 by sample, by unit
    short dz[64 * LH], dzt[MLP_H * LH];      // dZ of the layer being differentiated
    float dzf[64 * LH];                // dZ in FP32 by sample (bias gradients)
    short dz4[64 * LX], dz4t[16 * LH];
    float dz4f[64][2], sq[64];         // dZ4 and the squared errors
};

// sum over the 16 lanes of each lane group (same lane/16)
__device__ __forceinline__ float group16_sum(float v) {
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Four consecutive values of sample s from unit o in both orders.
__device__ __forceinline__ void put4(short *by_sample, int ld, short *by_unit, int s, int o, bf16x4 v) {
    *reinterpret_cast<bf16x4 *>(by_sample + s * ld + o) = v;
#pragma unroll
    for (int i = 0; i < 4; ++i) by_unit[(o + i) * LH + s] = v[i];
}

// One 16 x 16 tile of Z^T = W H^T + b over 64 units, as mlp_hidden.
__device__ __forceinline__ f32x4 layer_tile(const short *W, const float *b, const short *h, int ob, int sb, int lane) {
    bf16x4 w[4], x[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
        w[kb] = frag_a(W, LH, ob * 16, kb * 16, lane);
        x[kb] = frag_a(h, LH, sb * 16, kb * 16, lane);
    }
    f32x4 acc;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = b[ob * 16 + 4 * (lane >> 4) + i];
    acc = mfma32(cat8(w[0], w[1]), cat8(x[0], x[1]), acc);
    return mfma32(cat8(w[2], w[3]), cat8(x[2], x[3]), acc);
}

// One tile of dH^T = W^T dZ^T.
__device__ __forceinline__ f32x4 back_tile(const short *Wt, const short *dz, int ob, int sb, int lane) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
        acc = mfma16(frag_a(Wt, LH, ob * 16, kb * 16, lane), frag_a(dz, LH, sb * 16, kb * 16, lane), acc);
    return acc;
}

// One tile of dW = sum over the 64 samples of dZ[s][o] * H[s][in], samples in order: rows o <
// orows and columns in < icols are written to out (row stride ldo).
__device__ __forceinline__ void wgrad_tile(const short *dzt, const short *ht, int ob, int ib, float *out, int ldo,
                                           int orows, int icols, int lane) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int sb = 0; sb < 4; ++sb)
        acc = mfma16(frag_a(dzt, LH, ob * 16, sb * 16, lane), frag_a(ht, LH, ib * 16, sb * 16, lane), acc);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int o = ob * 16 + 4 * (lane >> 4) + i, in = ib * 16 + (lane & 15);
        if (o < orows && in < icols) out[o * ldo + in] = acc[i];
    }
}

// Partial gradient of the samples idx[base + wg*64 + 0..63] (those below count).  A wave has one 16 x 16
// tile of each layer (16 units of 16 samples) and keeps its pre-activations in registers; the
// activations go through LDS, a barrier a layer.  With one wave for all 16 tiles a batch of 4,096 samples
// left every latency exposed: 69 us, now 11.  Every sum is formed in the same
// order as by one wave.
constexpr int GRAD_T = 1024;
__global__ __launch_bounds__(GRAD_T) void k_mlp_grad(const float *__restrict__ P, const float *__restrict__ X,
                                                     const float *__restrict__ T, const int *__restrict__ idx, int base,
                                                     int count, float inv_n, float *__restrict__ part) {
    extern __shared__ __align__(16) unsigned char smem[];
    GradLds &S = *reinterpret_cast<GradLds *>(smem);
    const int tid = threadIdx.x, lane = tid & 63, ob = tid >> 8, sb = (tid >> 6) & 3;
    const int s0 = blockIdx.x * 64;
    auto sample = [&](int s) { return s0 + s < count ? (idx ? idx[base + s0 + s] : base + s0 + s) : -1; };
    {
        const int s = tid >> 4, f = tid & 15;  // 64 samples x 16 inputs
        const int g = sample(s);
        const short v = g >= 0 && f < MLP_IN ? f2bf(X[(size_t)g * MLP_IN + f]) : (short)0;
        S.x[s * LX + f] = v;
        S.xt[f * LH + s] = v;
    }
#pragma unroll
    for (int k = tid; k < MLP_H * MLP_H; k += GRAD_T) {
        const int o = k >> 6, i = k & 63;
        const short v2 = f2bf(P[MLP_W2 + k]), v3 = f2bf(P[MLP_W3 + k]);
        S.w2[o * LH + i] = v2;
        S.w2t[i * LH + o] = v2;
        S.w3[o * LH + i] = v3;
        S.w3t[i * LH + o] = v3;
    }
    {
        const int o = tid >> 4, i = tid & 15;  // 64 x 16
        S.w1[o * LX + i] = i < MLP_IN ? f2bf(P[MLP_W1 + o * MLP_IN + i]) : (short)0;
        S.w4t[o * LX + i] = i < MLP_OUT ? f2bf(P[MLP_W4 + i * MLP_H + o]) : (short)0;
        const int o4 = tid >> 6, i4 = tid & 63;  // 16 x 64
        S.w4[o4 * LH + i4] = o4 < MLP_OUT ? f2bf(P[MLP_W4 + tid]) : (short)0;
    }
    if (tid < MLP_H) {
        S.b1[tid] = P[MLP_B1 + tid];
        S.b2[tid] = P[MLP_B2 + tid];
        S.b3[tid] = P[MLP_B3 + tid];
    }
    if (tid < 4) S.b4[tid] = tid < MLP_OUT ? P[MLP_B4 + tid] : 0.0f;
    __syncthreads();

    // forward: this wave's sample and units in the MFMA result layout
    const int s = sb * 16 + (lane & 15), o = ob * 16 + 4 * (lane >> 4);
    f32x4 Z[3];
    auto activate = [&](int l) {
        f32x4 h;
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i] = gelu(Z[l][i]);
        put4(S.h[l], LH, S.ht[l], s, o, pack4(h));
    };
#pragma unroll
    for (int i = 0; i < 4; ++i) Z[0][i] = S.b1[o + i];
    Z[0] = mfma16(frag_a(S.w1, LX, ob * 16, 0, lane), frag_a(S.x, LX, sb * 16, 0, lane), Z[0]);
    activate(0);
    __syncthreads();
    Z[1] = layer_tile(S.w2, S.b2, S.h[0], ob, sb, lane);
    activate(1);
    __syncthreads();
    Z[2] = layer_tile(S.w3, S.b3, S.h[1], ob, sb, lane);
    activate(2);
    __syncthreads();

    // outputs, loss and dZ4 = 2 (y - t) / N: a wave per 16 samples, lanes 0..15 hold their outputs
    if (ob == 0) {
        bf16x4 w[4], h[4];
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
            w[kb] = frag_a(S.w4, LH, 0, kb * 16, lane);
            h[kb] = frag_a(S.h[2], LH, sb * 16, kb * 16, lane);
        }
        f32x4 y;
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = lane < 16 ? S.b4[i] : 0.0f;
        y = mfma32(cat8(w[0], w[1]), cat8(h[0], h[1]), y);
        y = mfma32(cat8(w[2], w[3]), cat8(h[2], h[3]), y);
        f32x4 d = {0.f, 0.f, 0.f, 0.f};
        float sq = 0.f;
        const int g = sample(s);
        if (lane < 16 && g >= 0) {
            const float e0 = y[0] - T[2 * (size_t)g], e1 = y[1] - T[2 * (size_t)g + 1];
            sq = e0 * e0 + e1 * e1;
            d[0] = 2.f * e0 * inv_n;
            d[1] = 2.f * e1 * inv_n;
        }
        put4(S.dz4, LX, S.dz4t, s, 4 * (lane >> 4), pack4(d));
        if (lane < 16) {
            S.dz4f[s][0] = d[0];
            S.dz4f[s][1] = d[1];
            S.sq[s] = sq;
        }
    }
    __syncthreads();

    float *G = part + (size_t)blockIdx.x * NP1;
    // dZ = dH * gelu'(Z) of a layer, in all three forms
    auto differentiate = [&](f32x4 dH, int l) {
        f32x4 d;
#pragma unroll
        for (int i = 0; i < 4; ++i) d[i] = dH[i] * gelu_grad(Z[l][i]);
        put4(S.dz, LH, S.dzt, s, o, pack4(d));
        *reinterpret_cast<f32x4 *>(S.dzf + s * LH + o) = d;
    };
    // db[u] = sum over the samples of dZ[s][u]: 16 threads a unit, four samples each, then their sum
    auto bgrad = [&](float *out) {
        const int u = tid >> 4, l = tid & 15;
        float v = 0.f;
#pragma unroll
        for (int q = 0; q < 4; ++q) v += S.dzf[(q * 16 + l) * LH + u];
        v = group16_sum(v);
        if (l == 0) out[u] = v;
    };
    // layer 4
    differentiate(mfma16(frag_a(S.w4t, LX, ob * 16, 0, lane), frag_a(S.dz4, LX, sb * 16, 0, lane),
                         f32x4{0.f, 0.f, 0.f, 0.f}),
                  2);
    if (ob == 0) wgrad_tile(S.dz4t, S.ht[2], 0, sb, G + MLP_W4, MLP_H, MLP_OUT, MLP_H, lane);
    if (ob == 1 && sb < 3) {  // the biases of the outputs, and the loss
        float v = 0.f;
        const int l = lane & 15;
#pragma unroll
        for (int q = 0; q < 4; ++q) v += sb < 2 ? S.dz4f[q * 16 + l][sb] : S.sq[q * 16 + l];
        v = group16_sum(v);
        if (lane == 0) G[sb < 2 ? MLP_B4 + sb : MLP_NPARAM] = v;
    }
    __syncthreads();
    // layers 3, 2 and 1: the gradients of a layer, and dH of the one before
#pragma unroll
    for (int l = 2; l > 0; --l) {
        wgrad_tile(S.dzt, S.ht[l - 1], ob, sb, G + (l == 2 ? MLP_W3 : MLP_W2), MLP_H, MLP_H, MLP_H, lane);
        bgrad(G + (l == 2 ? MLP_B3 : MLP_B2));
        const f32x4 dH = back_tile(l == 2 ? S.w3t : S.w2t, S.dz, ob, sb, lane);
        __syncthreads();  // dZ has been read
        differentiate(dH, l - 1);
        __syncthreads();
    }
    if (sb == 0) wgrad_tile(S.dzt, S.xt, ob, 0, G + MLP_W1, MLP_IN, MLP_H, MLP_IN, lane);
    bgrad(G + MLP_B1);
}

// The gradient of parameter p: the sum over workgroups of part[w][p], in workgroup order (16 loads in
// flight).
__device__ __forceinline__ float grad_of(const float *__restrict__ part, int nwg, int p) {
    float s = 0.f;
    int w = 0;
    for (; w + 16 <= nwg; w += 16) {
        float v[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) v[k] = part[(size_t)(w + k) * NP1 + p];
#pragma unroll
        for (int k = 0; k < 16; ++k) s += v[k];
    }
    for (; w < nwg; ++w) s += part[(size_t)w * NP1 + p];
    return s;
}

__global__ __launch_bounds__(64) void k_mlp_reduce(const float *__restrict__ part, int nwg, float *__restrict__ grad) {
    const int p = blockIdx.x * 64 + threadIdx.x;
    if (p < NP1) grad[p] = grad_of(part, nwg, p);
}

// Adam on the gradient that the workgroups' partials add up to; acc += the loss.
__global__ __launch_bounds__(64) void k_adam(const float *__restrict__ part, int nwg, float *__restrict__ P,
                                             float *__restrict__ m, float *__restrict__ v, float lr, float b1, float b2,
                                             float eps, float bc1, float bc2, float *__restrict__ acc) {
    const int p = blockIdx.x * 64 + threadIdx.x;
    if (p >= NP1) return;
    const float m0 = p < MLP_NPARAM ? m[p] : 0.f, v0 = p < MLP_NPARAM ? v[p] : 0.f, P0 = p < MLP_NPARAM ? P[p] : 0.f;
    const float gp = grad_of(part, nwg, p);
    if (p == MLP_NPARAM) {
        *acc += gp;
        return;
    }
    const float mp = b1 * m0 + (1.f - b1) * gp;
    const float vp = b2 * v0 + (1.f - b2) * gp * gp;
    m[p] = mp;
    v[p] = vp;
    P[p] = P0 - lr * (mp / bc1) / (sqrtf(vp / bc2) + eps);
}

__global__ __launch_bounds__(256) void k_mlp_eval(const float *__restrict__ P, const float *__restrict__ X, int n,
                                                  float *__restrict__ Y) {
    __shared__ MlpLds L;
    mlp_load(L, P, threadIdx.x, 256);
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int s0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 64;
    auto feat = [&](int s, int f) { return s0 + s < n ? X[(size_t)(s0 + s) * MLP_IN + f] : 0.0f; };
    f32x4 out[4];
    mlp_forward(L, feat, out, lane);
    if (lane < 16) {
#pragma unroll
        for (int sb = 0; sb < 4; ++sb) {
            const int s = s0 + sb * 16 + lane;
            if (s < n) {
                Y[2 * (size_t)s] = out[sb][0];
                Y[2 * (size_t)s + 1] = out[sb][1];
            }
        }
    }
}

struct Mem {
    std::vector<void *> p;
    hipStream_t s = nullptr;
    ~Mem() {
        if (s) (void)hipStreamSynchronize(s);
        for (void *q : p) (void)hipFree(q);
        if (s) (void)hipStreamDestroy(s);
    }
    template <class T> int alloc(T **out, size_t count) {
        void *q = nullptr;
        if (hipMalloc(&q, sizeof(T) * std::max<size_t>(count, 1)) != hipSuccess) return BL_E_NOMEM;
        p.push_back(q);
        *out = static_cast<T *>(q);
        return BL_OK;
    }
};

// The partial gradients of count samples, one a workgroup of 64.
int grad_launch(const float *P, const float *X, const float *T, const int *idx, int base, int count, float *part,
                hipStream_t s) {
    static bool attr = false;
    if (!attr) {
        BL_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k_mlp_grad),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(GradLds)));
        attr = true;
    }
    hipLaunchKernelGGL(k_mlp_grad, dim3((count + 63) / 64), dim3(GRAD_T), sizeof(GradLds), s, P, X, T, idx, base,
                       count, 1.0f / (float)count, part);
    BL_HIP(hipGetLastError());
    return BL_OK;
}

}  // namespace

int far_model_grad_host(const float *params, int32_t n, const float *feat, const float *targ, float *loss,
                        float *grad) {
    Mem M;
    BL_HIP(hipStreamCreateWithFlags(&M.s, hipStreamNonBlocking));
    float *dP, *dX, *dT, *dpart, *dg;
    const int nwg = (n + 63) / 64;
    if (M.alloc(&dP, MLP_NPARAM) || M.alloc(&dX, (size_t)n * MLP_IN) || M.alloc(&dT, (size_t)n * 2) ||
        M.alloc(&dpart, (size_t)nwg * NP1) || M.alloc(&dg, NP1))
        return BL_E_NOMEM;
    BL_HIP(hipMemcpyAsync(dP, params, 4 * MLP_NPARAM, hipMemcpyHostToDevice, M.s));
    BL_HIP(hipMemcpyAsync(dX, feat, 4 * (size_t)n * MLP_IN, hipMemcpyHostToDevice, M.s));
    BL_HIP(hipMemcpyAsync(dT, targ, 8 * (size_t)n, hipMemcpyHostToDevice, M.s));
    int rc = grad_launch(dP, dX, dT, nullptr, 0, n, dpart, M.s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_mlp_reduce, dim3((NP1 + 63) / 64), dim3(64), 0, M.s, dpart, nwg, dg);
    BL_HIP(hipGetLastError());
    std::vector<float> g(NP1);
    BL_HIP(hipMemcpyAsync(g.data(), dg, 4 * NP1, hipMemcpyDeviceToHost, M.s));
    BL_HIP(hipStreamSynchronize(M.s));
    if (grad) memcpy(grad, g.data(), 4 * MLP_NPARAM);
    if (loss) *loss = g[MLP_NPARAM] / (float)n;
    return BL_OK;
}

int far_model_eval_host(const float *params, int32_t n, const float *feat, float *out) {
    Mem M;
    BL_HIP(hipStreamCreateWithFlags(&M.s, hipStreamNonBlocking));
    float *dP, *dX, *dY;
    if (M.alloc(&dP, MLP_NPARAM) || M.alloc(&dX, (size_t)n * MLP_IN) || M.alloc(&dY, (size_t)n * 2))
        return BL_E_NOMEM;
    BL_HIP(hipMemcpyAsync(dP, params, 4 * MLP_NPARAM, hipMemcpyHostToDevice, M.s));
    BL_HIP(hipMemcpyAsync(dX, feat, 4 * (size_t)n * MLP_IN, hipMemcpyHostToDevice, M.s));
    hipLaunchKernelGGL(k_mlp_eval, dim3((n + 255) / 256), dim3(256), 0, M.s, dP, dX, n, dY);
    BL_HIP(hipGetLastError());
    BL_HIP(hipMemcpyAsync(out, dY, 8 * (size_t)n, hipMemcpyDeviceToHost, M.s));
    BL_HIP(hipStreamSynchronize(M.s));
    return BL_OK;
}

// Deterministic Adam training: epochs over a permutation of the samples drawn from `seed`
// (xorshift64*, Fisher-Yates), batches of `batch` samples, learning rate lr (beta1 0.9,
// beta2 0.999, eps 1e-8).  losses[e] = mean loss over the batches of epoch e.
int far_model_train_host(float *params, int32_t n, const float *feat, const float *targ, int32_t epochs,
                         int32_t batch, float lr, uint64_t seed, float *losses) {
    Mem M;
    BL_HIP(hipStreamCreateWithFlags(&M.s, hipStreamNonBlocking));
    float *dP, *dX, *dT, *dpart, *dm, *dv, *dacc;
    int *didx;
    const int nwg = (batch + 63) / 64;
    if (M.alloc(&dP, MLP_NPARAM) || M.alloc(&dX, (size_t)n * MLP_IN) || M.alloc(&dT, (size_t)n * 2) ||
        M.alloc(&dpart, (size_t)nwg * NP1) || M.alloc(&dm, MLP_NPARAM) ||
        M.alloc(&dv, MLP_NPARAM) || M.alloc(&dacc, std::max(epochs, 1)) || M.alloc(&didx, n))
        return BL_E_NOMEM;
    BL_HIP(hipMemcpyAsync(dP, params, 4 * MLP_NPARAM, hipMemcpyHostToDevice, M.s));
    BL_HIP(hipMemcpyAsync(dX, feat, 4 * (size_t)n * MLP_IN, hipMemcpyHostToDevice, M.s));
    BL_HIP(hipMemcpyAsync(dT, targ, 8 * (size_t)n, hipMemcpyHostToDevice, M.s));
    BL_HIP(hipMemsetAsync(dm, 0, 4 * MLP_NPARAM, M.s));
    BL_HIP(hipMemsetAsync(dv, 0, 4 * MLP_NPARAM, M.s));
    BL_HIP(hipMemsetAsync(dacc, 0, 4 * (size_t)std::max(epochs, 1), M.s));
    std::vector<int> perm(n);
    uint64_t st = seed ? seed : 0x9E3779B97F4A7C15ull;
    auto rnd = [&]() {
        st ^= st >> 12;
        st ^= st << 25;
        st ^= st >> 27;
        return st * 2685821657736338717ull;
    };
    const float b1 = 0.9f, b2 = 0.999f;
    double p1 = 1.0, p2 = 1.0;
    std::vector<int> nbatches(std::max(epochs, 1), 0);
    for (int e = 0; e < epochs; ++e) {
        for (int i = 0; i < n; ++i) perm[i] = i;
        for (int i = n - 1; i > 0; --i) std::swap(perm[i], perm[(int)(rnd() % (uint64_t)(i + 1))]);
        // the upload is ordered on the stream before this epoch's kernels; wait before the
        // next epoch rewrites perm
        BL_HIP(hipMemcpyAsync(didx, perm.data(), 4 * (size_t)n, hipMemcpyHostToDevice, M.s));
        for (int off = 0; off < n; off += batch) {
            const int cnt = std::min(batch, n - off);
            int rc = grad_launch(dP, dX, dT, didx, off, cnt, dpart, M.s);
            if (rc) return rc;
            p1 *= b1;
            p2 *= b2;
            hipLaunchKernelGGL(k_adam, dim3((NP1 + 63) / 64), dim3(64), 0, M.s, dpart, (cnt + 63) / 64, dP, dm, dv, lr,
                               b1, b2, 1e-8f, (float)(1.0 - p1), (float)(1.0 - p2), dacc + e);
            ++nbatches[e];
        }
        BL_HIP(hipGetLastError());
        BL_HIP(hipStreamSynchronize(M.s));
    }
    std::vector<float> acc(std::max(epochs, 1));
    BL_HIP(hipMemcpyAsync(acc.data(), dacc, 4 * acc.size(), hipMemcpyDeviceToHost, M.s));
    BL_HIP(hipMemcpyAsync(params, dP, 4 * MLP_NPARAM, hipMemcpyDeviceToHost, M.s));
    BL_HIP(hipStreamSynchronize(M.s));
    // acc[e] is the sum over batches of the summed squared errors: mean per sample
    if (losses)
        for (int e = 0; e < epochs; ++e) losses[e] = acc[e] / (float)n;
    return BL_OK;
}

}  // namespace bl
