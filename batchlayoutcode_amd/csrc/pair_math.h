// Device arithmetic shared by the minibatch kernels (single graph and batched).
//
// Reference semantics (sample/algorithms.cpp:758-768): a neighbour j of i contributes the
// attraction A(d) with d = x_j - x_i; any other j with |d|^2 > 0 contributes -d/|d|^2.
// The dense loops add -d/|d|^2 for every j (the self pair gives 0); correct_pair() then
// removes, for each neighbour, the product the dense loop added and adds A(d).  Neighbours almost
// on top of a vertex, whose product would drown its force, are left out instead (apart_share).
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

// A group's differences to (px, py) and |d|^2: positions at(j), at(j + D), ... below end; those past it stand
// for a pair of distance 0 and |d|^2 = 1.
template <int N, class At>
__device__ __forceinline__ void load_group(At at, const int j, const int D, const int end, const double px,
                                           const double py, double *dx, double *dy, double *r) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const bool in = j + k * D < end;
        const double2 q = at(in ? j + k * D : j);
        dx[k] = in ? q.x - px : 0.0;
        dy[k] = in ? q.y - py : 0.0;
        r[k] = in ? fma(dy[k], dy[k], fma(dx[k], dx[k], kTiny64)) : 1.0;
    }
}

// Adds the terms of a group.  CAREFUL: a product of |d|^2 may have left the FP64 range; where a pair's factor
// is not finite, it has one of its own.
template <int N, bool CAREFUL, class At>
__device__ __forceinline__ void add_group(At at, const int j, const int D, const int end, const double px,
                                          const double py, double &ax, double &ay) {
    double dx[N], dy[N], r[N], own[N];
    load_group<N>(at, j, D, end, px, py, dx, dy, r);
#pragma unroll
    for (int k = 0; k < N; ++k) own[k] = r[k];
    recip_all<N>(r);
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const double f = CAREFUL && !isfinite(r[k]) ? recip(own[k]) : r[k];
        ax = fma(-dx[k], f, ax);
        ay = fma(-dy[k], f, ay);
    }
}

// x, y interleaved as positions.
template <class Src>
__device__ __forceinline__ auto interleaved(Src src) {
    return [=](int j) { return make_double2(src[2 * j], src[2 * j + 1]); };
}

constexpr int GROUP = 8;  // pairs that share a reciprocal

// The dense repulsion of position (px, py) against positions [j0, j1) of src (x, y interleaved),
// U positions loaded at a time, in (ax, ay).  A sum that is not finite is formed again with care: a
// group's product may have left the FP64 range where no single |d|^2 does.
// PAD: the positions past the last U in one more group filled up (for short ranges; a serial chain of
// reciprocals took 5 us of a batch step); otherwise one by one, in less code.
template <bool REFINE, int U, bool PAD = false, class Src>
__device__ __forceinline__ void dense_sum(Src src, const int j0, const int j1, const double px, const double py,
                                          double &ax, double &ay) {
    constexpr int N = GROUP;
    static_assert(U % N == 0 && (!PAD || U == N), "whole groups");
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
    if constexpr (PAD && REFINE) {
        if (j < j1) add_group<N, false>(interleaved(src), j, 1, j1, px, py, ax, ay);
    } else {
        for (; j < j1; ++j) pair_rep<REFINE>(src[2 * j], src[2 * j + 1], px, py, ax, ay);
    }
    if (REFINE && !(isfinite(ax) && isfinite(ay))) {
        ax = ay = 0.0;
        const int grouped = PAD ? j1 : j0 + (j1 - j0) / U * U;
        for (j = j0; j < grouped; j += N) add_group<N, true>(interleaved(src), j, 1, j1, px, py, ax, ay);
        for (; j < j1; ++j) pair_rep<REFINE>(src[2 * j], src[2 * j + 1], px, py, ax, ay);
    }
}

// The dense repulsion of (px, py) against positions j0, j0 + D, ... below n, added to (ax, ay): groups of 8
// as dense_sum, the last one filled up.
template <bool REFINE, int D>
__device__ __forceinline__ void strided_sum(const double2 *__restrict__ src, const int j0, const int n, const double px,
                                            const double py, double &ax, double &ay) {
    constexpr int N = GROUP;
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
        const auto at = [=](int q) { return src[q]; };
        if (j < n) add_group<N, false>(at, j, D, n, px, py, sx, sy);
        if (!(isfinite(sx) && isfinite(sy))) {
            sx = sy = 0.0;
            for (j = j0; j < n; j += N * D) add_group<N, true>(at, j, D, n, px, py, sx, sy);
        }
    } else {
        for (; j < n; j += D) pair_rep<false>(src[j].x, src[j].y, px, py, sx, sy);
    }
    ax += sx;
    ay += sy;
}

// The factor 1/|d|^2 that a dense sum gave the pair at place m of the group at(first), at(first + D), ...
// below end, bit for bit: the products of recip_all, which are the same from every place of the group.
template <class At>
__device__ __forceinline__ double group_factor(At at, const int first, const int m, const int D, const int end,
                                               const double px, const double py) {
    double r[GROUP];
    static_assert(GROUP == 8, "three levels of products");
#pragma unroll
    for (int k = 0; k < GROUP; ++k) {
        const int j = first + (m ^ k) * D;
        const double2 q = at(j < end ? j : first);
        const double dx = q.x - px, dy = q.y - py;
        r[k] = j < end ? fma(dy, dy, fma(dx, dx, kTiny64)) : 1.0;
    }
    const double two = r[2] * r[3], four = (r[4] * r[5]) * (r[6] * r[7]);
    const double f = recip(((r[0] * r[1]) * two) * four) * four * two * r[1];
    return isfinite(f) ? f : recip(r[0]);
}

// The factor to remove a linked pair (dx, dy) with: bit for bit the dense sum's where the pair is close (group:
// whether it was in one).  Further away than 2^-8 one of its own, which differs by about 2^-52: less than the
// roundings of the dense sum's additions after the pair.  (Eight loads for every neighbour made the step of the
// 250k random geometric graph 4% longer: the correction's workgroups hold up the last of the others.)
constexpr double kNear2 = 0x1p-16;
template <bool REFINE, class At>
__device__ __forceinline__ double linked_factor(At at, const bool group, const int first, const int m, const int D,
                                                const int end, const double px, const double py, const double dx,
                                                const double dy) {
    if (REFINE && group && fma(dy, dy, dx * dx) < kNear2) return group_factor(at, first, m, D, end, px, py);
    return inv_r2<REFINE>(dx, dy);
}

// A linked pair closer than 2^-40 (coincident ones aside, whose terms are 0): its repulsion, which the
// reference never forms, would take the force's low digits with it when it is added and removed again.
constexpr double kApart2 = 0x1p-80;
template <bool REFINE>
__device__ __forceinline__ bool too_close(const double dx, const double dy) {
    return REFINE && fma(dy, dy, dx * dx) < kApart2 && (dx != 0.0 || dy != 0.0);
}

// Neighbour correction for one (i, j) pair: removes the dense loop's product, formed from the same factor
// `inv`, and adds the attraction.
__device__ __forceinline__ void correct_pair(int law, double W, double dx, double dy, double inv, double &cx, double &cy) {
    cx += dx * inv;
    cy += dy * inv;
    attract64(law, W, dx, dy, cx, cy);
}

// A thread's share t, t + D, ... of the whole force on position (px, py) of a vertex whose neighbours are
// entries [e0, e1) of ci (ascending), one of them too close: such neighbours are not added at all.  Rare,
// so a pair at a time.
template <class At, class Weight>
__device__ __forceinline__ double2 apart_share(At at, const int n, const int t, const int D, const double px,
                                               const double py, const int *__restrict__ ci, const int e0, const int e1,
                                               Weight weight, const int law) {
    double fx = 0.0, fy = 0.0;
    int e = e0, next = -1;  // ci[e], once read
    for (int j = t; j < n; j += D) {
        const double2 q = at(j);
        if (too_close<true>(q.x - px, q.y - py)) {
            if (next < j) {  // on to the first neighbour >= j, in growing steps
                int step = 1;
                for (; e < e1 && ci[min(e + step, e1) - 1] < j; step <<= 1) e = min(e + step, e1);
                int hi = min(e + step, e1);
                while (e < hi) {
                    const int m = (e + hi) >> 1;
                    if (ci[m] < j) e = m + 1; else hi = m;
                }
                next = e < e1 ? ci[e] : 0x7fffffff;
            }
            if (next == j) continue;
        }
        pair_rep<true>(q.x, q.y, px, py, fx, fy);
    }
    for (e = e0 + t; e < e1; e += D) {
        const double2 q = at(ci[e]);
        const double dx = q.x - px, dy = q.y - py;
        correct_pair(law, weight(e), dx, dy, too_close<true>(dx, dy) ? 0.0 : inv_r2<true>(dx, dy), fx, fy);
    }
    return make_double2(fx, fy);
}

// x_i += (F/|F|) * STEP, algorithms.cpp:775-779 / Coordinate.h:57-65.
__device__ __forceinline__ double2 moved(double2 p, double fx, double fy, double step) {
    const double mag = sqrt(fx * fx + fy * fy);
    p.x = p.x + (fx / mag) * step;
    p.y = p.y + (fy / mag) * step;
    return p;
}

}  // namespace bl
