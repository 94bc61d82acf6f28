// Device arithmetic shared by the minibatch kernels (single graph and batched).
//
// Reference semantics (sample/algorithms.cpp:758-768): a neighbour j of i contributes the
// attraction A(d) with d = x_j - x_i; any other j with |d|^2 > 0 contributes -d/|d|^2.
// The dense loops add -d/|d|^2 for every j (the self pair gives 0); correct_pair() then
// removes, for each neighbour, the product the dense loop added and adds A(d).
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>

#include "bl_internal.h"

namespace bl {

// |d|^2 floors: the self pair and coincident vertices give 0 * (1/floor) = 0, as the
// reference's `dist > 0` test skips them.  The FP64 floor is below the last bit of |d|^2 for
// |d| > 1e-22 (1e-30 moved the terms of a layout of extent 1e-7 by 1e-14).
constexpr float kTiny = 1e-30f;
constexpr double kTiny64 = 0x1p-200;

// v + the value of the lane CTRL names (a DPP move; lanes without a source lane, or outside
// ROW_MASK, add +0.0).
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_add(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROW_MASK, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROW_MASK, 0xF, false);
    return v + __hiloint2double(hi, lo);
}

// Sum over the 64 lanes of the wave (all active), the same value in every lane: an inclusive
// scan by DPP moves (row_shr 1, 2, 4, 8 within rows of 16 lanes, then row_bcast:15 into rows
// 1 and 3 and row_bcast:31 into rows 2 and 3) leaves the total in lane 63, which is
// broadcast.  DPP moves cost a few cycles where the LDS permutes of a shuffle butterfly
// cost a round trip through the LDS unit each.
__device__ __forceinline__ double wave_sum(double v) {
    v = dpp_add<0x111, 0xF>(v);
    v = dpp_add<0x112, 0xF>(v);
    v = dpp_add<0x114, 0xF>(v);
    v = dpp_add<0x118, 0xF>(v);
    v = dpp_add<0x142, 0xA>(v);
    v = dpp_add<0x143, 0xC>(v);
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                            __builtin_amdgcn_readlane(__double2loint(v), 63));
}

// Attraction of one neighbour pair, in the reference's FP64 operation order:
// f += d * (W * |d|) (:759), f += d * W (:985), f += d * log2(1 + W|d|) (:912).
__device__ __forceinline__ void attract64(int law, double W, double dx, double dy, double &fx, double &fy) {
    double s;
    if (law == LAW_FA) {
        s = W;
    } else {
        const double mag = sqrt(dx * dx + dy * dy);
        s = (law == LAW_FR) ? W * mag : log2(1.0 + W * mag);
    }
    fx += dx * s;
    fy += dy * s;
}

// 1/x for x > 0: the hardware estimate (relative error about 2^-25) and one Newton step (about
// 2^-50).
__device__ __forceinline__ double recip(const double x) {
    const double s = __builtin_amdgcn_rcp(x);
    return fma(s, fma(-x, s, 1.0), s);
}

// 1/|d|^2 for a pair with FP64 difference (dx, dy).  REFINE: FP64 throughout.  Otherwise |d|^2 and
// the reciprocal in FP32 (relative error ~1e-7).
template <bool REFINE>
__device__ __forceinline__ double inv_r2(const double dx, const double dy) {
    if constexpr (REFINE) {
        return recip(fma(dy, dy, fma(dx, dx, kTiny64)));
    } else {
        const float fx = (float)dx, fy = (float)dy;
        const float r2 = fmaf(fy, fy, fmaf(fx, fx, kTiny));
        return (double)__builtin_amdgcn_rcpf(r2);
    }
}

// One dense repulsion pair: -d/|d|^2 accumulated in FP64.
template <bool REFINE>
__device__ __forceinline__ void pair_rep(const double qx, const double qy, const double px, const double py,
                                         double &ax, double &ay) {
    const double dx = qx - px, dy = qy - py;
    const double inv = inv_r2<REFINE>(dx, dy);
    ax = fma(-dx, inv, ax);
    ay = fma(-dy, inv, ay);
}

// 1/r[k] of N (a power of two) values from one reciprocal, that of their product: the product's
// inverse times the other half's product is a half's inverse, down to single values.
template <int N>
__device__ __forceinline__ void recip_all(double *r) {
    if constexpr (N == 1) {
        r[0] = recip(r[0]);
    } else {
        double h[N / 2];
#pragma unroll
        for (int k = 0; k < N / 2; ++k) h[k] = r[2 * k] * r[2 * k + 1];
        recip_all<N / 2>(h);
#pragma unroll
        for (int k = 0; k < N / 2; ++k) {
            const double a = r[2 * k];
            r[2 * k] = h[k] * r[2 * k + 1];
            r[2 * k + 1] = h[k] * a;
        }
    }
}

// N dense repulsion pairs added in order.  What bounds the dense sum is its FP64 operations (a
// reciprocal takes about four of them): 6 a pair (difference, |d|^2, the two sums) and the
// reciprocal.  One of its own costs a pair 6 more (REFINE's former seed in FP32: two conversions, the FP32
// reciprocal, the Newton step); shared by a group of N, 3 products and 6/N.  Measured: the all-pairs step's pair kernel on
// the 250k random geometric graph 25.6 -> 20.6 us, on the R-MAT graph at -batch 1024 189 -> 162 us.
// A product past the FP64 range (|d| beyond 1e19 in all of 8 pairs) makes the sum NaN (see
// dense_sum).
template <bool REFINE, int N>
__device__ __forceinline__ void pair_rep_group(const double *qx, const double *qy, const double px, const double py,
                                               double &ax, double &ay) {
    if constexpr (REFINE) {
        double dx[N], dy[N], r[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
            dx[k] = qx[k] - px;
            dy[k] = qy[k] - py;
            r[k] = fma(dy[k], dy[k], fma(dx[k], dx[k], kTiny64));
        }
        recip_all<N>(r);
#pragma unroll
        for (int k = 0; k < N; ++k) {
            ax = fma(-dx[k], r[k], ax);
            ay = fma(-dy[k], r[k], ay);
        }
    } else {
#pragma unroll
        for (int k = 0; k < N; ++k) pair_rep<false>(qx[k], qy[k], px, py, ax, ay);
    }
}

// The positions [j, j1) past the last whole group of N, added in order.  REFINE: one more group, filled
// up with pairs of distance 0 and |d|^2 = 1 (a serial chain of reciprocals took 5 us of a batch step).
template <bool REFINE, int N, class Src>
__device__ __forceinline__ void dense_tail(Src src, const int j, const int j1, const double px, const double py,
                                           double &ax, double &ay) {
    if constexpr (REFINE) {
        double dx[N], dy[N], r[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const int q = min(j + k, j1 - 1);
            const double qx = src[2 * q], qy = src[2 * q + 1];
            const bool in = j + k < j1;
            dx[k] = in ? qx - px : 0.0;
            dy[k] = in ? qy - py : 0.0;
            r[k] = in ? fma(dy[k], dy[k], fma(dx[k], dx[k], kTiny64)) : 1.0;
        }
        recip_all<N>(r);
#pragma unroll
        for (int k = 0; k < N; ++k) {
            ax = fma(-dx[k], r[k], ax);
            ay = fma(-dy[k], r[k], ay);
        }
    } else {
        for (int k = j; k < j1; ++k) pair_rep<false>(src[2 * k], src[2 * k + 1], px, py, ax, ay);
    }
}

// The dense repulsion of position (px, py) against positions [j0, j1) of src (x, y interleaved),
// U positions loaded at a time, in (ax, ay).  A sum that is not finite is formed again pair by
// pair: a group's product may have left the FP64 range where no single |d|^2 does.
// PAD: the positions past the last whole group by dense_tail (for short ranges; otherwise one by one, in less code).
template <bool REFINE, int U, bool PAD = false, class Src>
__device__ __forceinline__ void dense_sum(Src src, const int j0, const int j1, const double px, const double py,
                                          double &ax, double &ay) {
    constexpr int N = 8;  // pairs that share a reciprocal
    static_assert(U % N == 0, "whole groups");
    ax = ay = 0.0;
    int j = j0;
    for (; j + U <= j1; j += U) {
        double qx[U], qy[U];
#pragma unroll
        for (int k = 0; k < U; ++k) {
            qx[k] = src[2 * (j + k)];
            qy[k] = src[2 * (j + k) + 1];
        }
#pragma unroll
        for (int k = 0; k < U; k += N) pair_rep_group<REFINE, N>(qx + k, qy + k, px, py, ax, ay);
    }
    if constexpr (PAD) {
        if (j < j1) dense_tail<REFINE, N>(src, j, j1, px, py, ax, ay);
        j = j1;
    }
    for (; j < j1; ++j) pair_rep<REFINE>(src[2 * j], src[2 * j + 1], px, py, ax, ay);
    if (REFINE && !(isfinite(ax) && isfinite(ay))) {
        ax = ay = 0.0;
        for (j = j0; j < j1; ++j) pair_rep<REFINE>(src[2 * j], src[2 * j + 1], px, py, ax, ay);
    }
}

// The dense repulsion of (px, py) against positions j0, j0 + D, ... below n, added to (ax, ay): groups of 8
// as dense_sum, the last one filled up as dense_tail.
template <bool REFINE, int D>
__device__ __forceinline__ void strided_sum(const double2 *__restrict__ src, const int j0, const int n, const double px,
                                            const double py, double &ax, double &ay) {
    constexpr int N = 8;
    double sx = 0.0, sy = 0.0;
    int j = j0;
    for (; j + (N - 1) * D < n; j += N * D) {
        double qx[N], qy[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const double2 q = src[j + k * D];
            qx[k] = q.x, qy[k] = q.y;
        }
        pair_rep_group<REFINE, N>(qx, qy, px, py, sx, sy);
    }
    if constexpr (REFINE) {
        if (j < n) {
            double dx[N], dy[N], r[N];
#pragma unroll
            for (int k = 0; k < N; ++k) {
                const bool in = j + k * D < n;
                const double2 q = src[in ? j + k * D : j];
                dx[k] = in ? q.x - px : 0.0;
                dy[k] = in ? q.y - py : 0.0;
                r[k] = in ? fma(dy[k], dy[k], fma(dx[k], dx[k], kTiny64)) : 1.0;
            }
            recip_all<N>(r);
#pragma unroll
            for (int k = 0; k < N; ++k) {
                sx = fma(-dx[k], r[k], sx);
                sy = fma(-dy[k], r[k], sy);
            }
        }
        if (!(isfinite(sx) && isfinite(sy))) {
            sx = sy = 0.0;
            for (j = j0; j < n; j += D) pair_rep<true>(src[j].x, src[j].y, px, py, sx, sy);
        }
    } else {
        for (; j < n; j += D) pair_rep<false>(src[j].x, src[j].y, px, py, sx, sy);
    }
    ax += sx;
    ay += sy;
}

// Neighbour correction for one (i, j) pair: removes the dense loop's product (dx * inv; with REFINE
// to its last bits, of the order of the dense sum's own rounding) and adds the attraction.
template <bool REFINE>
__device__ __forceinline__ void correct_pair(int law, double W, double dx, double dy, double &cx, double &cy) {
    const double inv = inv_r2<REFINE>(dx, dy);
    cx += dx * inv;
    cy += dy * inv;
    attract64(law, W, dx, dy, cx, cy);
}

// x_i += (F/|F|) * STEP, algorithms.cpp:775-779 / Coordinate.h:57-65.
__device__ __forceinline__ double2 moved(double2 p, double fx, double fy, double step) {
    const double mag = sqrt(fx * fx + fy * fy);
    p.x = p.x + (fx / mag) * step;
    p.y = p.y + (fy / mag) * step;
    return p;
}

}  // namespace bl
