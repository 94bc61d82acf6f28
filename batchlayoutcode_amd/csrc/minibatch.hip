// Minibatch force step of the BatchLayout cache-blocking family on CDNA4 (gfx950).
//
// Reference: sample/algorithms.cpp:715-794 (algo 2), :795-871 (converged variant),
// :874-945 (algo 3, LinLog), :947-1018 (algo 8).  One iteration visits the vertices
// in ceil(n/B) consecutive batches (Gauss-Seidel across batches); inside a batch
// every vertex i sees the positions from the start of the batch step (Jacobi):
//
//   F_i = sum_{j in N(i)} A(x_j - x_i)  -  sum_{j not in N(i), |x_j-x_i|>0} (x_j - x_i)/|x_j - x_i|^2
//   x_i += STEP * F_i/|F_i|,   ENERGY += |F_i|^2,   STEP *= decay after each iteration
//
// where N(i) is the set of column ids the reference's merge pointer meets (:758-762)
// and A is the attraction law (W|d| d, W d, or log2(1+W|d|) d).
//
// Mixed and FP32 modes (the fast path).  Per pair: the FP64 difference d = x_j - x_i, |d|^2 and
// 1/|d|^2 (mixed: FP64, one reciprocal for eight pairs; FP32: v_rcp_f32), and the term -d/|d|^2
// accumulated in FP64 (one FMA per component with the FP64 difference).  The dense loop runs over all j; neighbours are not
// branched on: a correction adds, in FP64, each neighbour's attraction and removes the
// repulsion product the dense loop accumulated for it, for close ones from the same factor bit for bit
// (linked_factor), so that what is left of it is the sum's own rounding.  A vertex with a neighbour closer than 2^-40 has its
// force formed without that neighbour's repulsion (apart_share).
//   * k_step32 (small graphs): one launch per batch step, a workgroup per batch vertex.
//   * k_pairs32 + k_move32: two launches per batch step.  The pair kernel's
//     chunk workgroups write each batch vertex's chunk partials; its correction waves take
//     the neighbour corrections in pieces of at most CORR_PIECE entries (a hub's
//     correction is spread over many waves); k_move32 adds them in a fixed order and moves.
//   * With BL_GRAPH=1, one iteration's launches (every batch step, the energy, STEP *= decay
//     on the device) are captured once as a hipGraph and replayed, one host launch per
//     iteration (measured no faster on this GPU, so not the default).
//
// FP64 mode (reference-grade): the reference's own operations, in its order.  The
// j range is cut into the reference's 512-wide blocks (blocky, :717); each block's
// partial is summed in j order with the merge-pointer branch, and the partials are
// added in block order, so the result reproduces the strict-IEEE reference build.
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <mutex>

#include <hip/hip_ext.h>

#include "bl_internal.h"
#include "pair_math.h"

namespace bl {
namespace {

constexpr int WG = 256;
constexpr int kBlockY = 512;  // the reference's j block, algorithms.cpp:717
constexpr int UNROLL = 16;

// Read-only view of the positions in the constant address space: with a wave-uniform
// index the compiler fetches x_j with scalar loads (one fetch per wave, no VGPRs).  Only
// used by kernels during which the positions do not change.
typedef const __attribute__((address_space(4))) double cdouble;

// x_i += (F/|F|) * STEP and |F|^2, algorithms.cpp:775-779 / Coordinate.h:57-65.
__device__ __forceinline__ void move_one(double2 *pos, int i, double fx, double fy, double step, double *eterm) {
    pos[i] = moved(pos[i], fx, fy, step);
    eterm[i] = fx * fx + fy * fy;
}

// ---------------------------------------------------------------------------------------
// Per-step kernels: the FP32 fallback and the FP64 reference-order path

// Dense FP32 repulsion + neighbour correction (one launch per batch step).
// grid = (G + ncorr, rows), 256 threads.  Workgroups x < G: batch slots [y*IPW, y*IPW+IPW)
// against j chunk x, split over JS = 256/IPW j-subgroups added in LDS in subgroup order.
// Workgroups x >= G (row 0 only): one wave per correction piece of the batch (pieces
// [pc0, pc0+npc): at most CORR_PIECE neighbour entries of one vertex, so a hub's correction
// is spread over many waves instead of holding up the step).
// part[slot * P + x] receives the chunk partial; part[slot * P + G + k] piece k's correction, or a NaN of
// the bits APART and the x of the vertex's whole force, whose y is then in eterm.
constexpr long long APART = 0x7ffa6d6f72746170;
template <int JS, bool REFINE>
__global__ __launch_bounds__(WG) void k_pairs32(const double2 *__restrict__ pos, int n, int b0, int bc, int chunk,
                                                int G, double2 *__restrict__ part, int P,
                                                const int *__restrict__ erp, const int *__restrict__ eci,
                                                const float *__restrict__ ew, double W, int law,
                                                const int *__restrict__ cpre, const int *__restrict__ cpv, int pc0,
                                                int npc, double *__restrict__ eterm) {
    constexpr int IPW = WG / JS;
    __shared__ double2 red[WG];
    const int tid = threadIdx.x;
    if (__builtin_expect((int)blockIdx.x >= G, 0)) {  // its code last: 0.5 us a step with it before the dense sum's
        if (blockIdx.y != 0) return;
        const int w = ((int)blockIdx.x - G) * (WG / 64) + tid / 64;
        const int lane = tid & 63;
        if (w >= npc) return;
        const int pc = pc0 + w;
        const int i = cpv[pc], k = pc - cpre[i];
        const double2 pi = pos[i];
        double cx = 0.0, cy = 0.0;
        const int kbeg = erp[i] + k * CORR_PIECE;
        const int kend = min(erp[i + 1], kbeg + CORR_PIECE);
        const int grouped = n / UNROLL * UNROLL;  // a subgroup's range begins and ends at whole UNROLLs, or at n
        const auto at = [=](int j) { return pos[j]; };
        bool close = false;
        for (int e = kbeg + lane; e < kend; e += 64) {
            const int j = eci[e];
            const double2 pj = pos[j];
            const double dx = pj.x - pi.x, dy = pj.y - pi.y;
            const double inv = linked_factor<REFINE>(at, j < grouped, j & ~(GROUP - 1), j & (GROUP - 1), 1, n, pi.x,
                                                     pi.y, dx, dy);
            correct_pair(law, ew ? W * (double)ew[e] : W, dx, dy, inv, cx, cy);
            close = close || too_close<REFINE>(dx, dy);
        }
        double2 *mine = part + (size_t)(i - b0) * P + G + k;
        if (__ballot(close)) {  // the whole force, for k_move32 to take instead of the sum
            const double2 f = apart_share(at, n, lane, 64, pi.x, pi.y, eci, erp[i], erp[i + 1],
                                          [=](int e) { return ew ? W * (double)ew[e] : W; }, law);
            cx = wave_sum(f.x);
            cy = wave_sum(f.y);
            if (lane == 0) {
                *mine = make_double2(__longlong_as_double(APART), cx);
                eterm[i] = cy;
            }
            return;
        }
        cx = wave_sum(cx);
        cy = wave_sum(cy);
        if (lane == 0) *mine = make_double2(cx, cy);
        return;
    }
    const int li = tid % IPW;
    const int js = __builtin_amdgcn_readfirstlane(tid / IPW);  // IPW is a multiple of 64
    cdouble *cpos = (cdouble *)pos;
    const int slot = (int)blockIdx.y * IPW + li;
    const int i = b0 + (slot < bc ? slot : bc - 1);
    const double px = pos[i].x, py = pos[i].y;
    const int jb = (int)blockIdx.x * chunk;
    const int je = min(n, jb + chunk);
    const int sub = (chunk + JS - 1) / JS;
    const int j0 = min(je, jb + js * sub);
    const int j1 = min(je, j0 + sub);
    double ax, ay;
    // lgkmcnt(0): with arguments still on their way the compiler waits between the loop's scalar loads, in every
    // round (1 us a step)
    __builtin_amdgcn_s_waitcnt(0xc07f);
    dense_sum<REFINE, UNROLL>(cpos, j0, j1, px, py, ax, ay);
    if constexpr (JS > 1) {
        red[tid] = make_double2(ax, ay);
        __syncthreads();
        if (js == 0) {
#pragma unroll
            for (int s = 1; s < JS; ++s) {
                ax += red[s * IPW + li].x;
                ay += red[s * IPW + li].y;
            }
        }
    }
    if (js == 0 && slot < bc) part[(size_t)slot * P + blockIdx.x] = make_double2(ax, ay);
}

// A whole batch step in one launch, a workgroup of NT threads per batch vertex: the dense sum (thread
// t takes positions t, t + NT, ...), the corrections, the move.  No partial leaves the workgroup, so
// the second launch and its loads go; every vertex's workgroup reads all positions itself.  The
// positions are in two arrays: a step reads src, which holds every move before it, and writes dst,
// which lacks the previous batch's (p0, pc) and gets them copied with this batch's.  What bounds a step
// is the launch and two dependent loads (3.8 us); figures at one_launch.
template <int NT, bool REFINE>
__global__ __launch_bounds__(NT) void k_step32(const double2 *__restrict__ src, double2 *__restrict__ dst, int n,
                                               int p0, int pc, int b0, const int *__restrict__ erp,
                                               const int *__restrict__ eci, const float *__restrict__ ew, double W,
                                               int law, const double *__restrict__ stepp, double step,
                                               double *__restrict__ eterm) {
    __shared__ double2 red[NT / 64];
    const int tid = threadIdx.x;
    const int i = b0 + (int)blockIdx.x;
    const double2 pi = src[i];
    const int e0 = erp[i], e1 = erp[i + 1];
    const int jn = e0 + tid < e1 ? eci[e0 + tid] : 0;
    double ax = 0.0, ay = 0.0;
    strided_sum<REFINE, NT>(src, tid, n, pi.x, pi.y, ax, ay);
    double cx = 0.0, cy = 0.0;
    bool close = false;
    const auto at = [=](int j) { return src[j]; };
    for (int e = e0 + tid; e < e1; e += NT) {
        const int j = e == e0 + tid ? jn : eci[e];
        const double2 pj = src[j];
        const double dx = pj.x - pi.x, dy = pj.y - pi.y;
        const int q = j / NT;  // the position's place in thread j % NT
        const double inv = linked_factor<REFINE>(at, true, j - (q & (GROUP - 1)) * NT, q & (GROUP - 1), NT, n, pi.x, pi.y,
                                                 dx, dy);
        correct_pair(law, ew ? W * (double)ew[e] : W, dx, dy, inv, cx, cy);
        close = close || too_close<REFINE>(dx, dy);
    }
    ax = wave_sum(ax + cx);
    ay = wave_sum(ay + cy);
    const double mark = __longlong_as_double(APART);
    if (__ballot(close)) ax = mark;
    if ((tid & 63) == 0) red[tid >> 6] = make_double2(ax, ay);
    __syncthreads();
    if (tid == 64)
        for (int k = (int)blockIdx.x; k < pc; k += (int)gridDim.x) dst[p0 + k] = src[p0 + k];
    if (tid >= 64) return;
    double fx = red[0].x, fy = red[0].y;
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) fx += red[w].x, fy += red[w].y;
    if (REFINE && isnan(fx)) {  // the same in all lanes
        bool apart = false;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) apart = apart || __double_as_longlong(red[w].x) == APART;
        if (apart) {
            const double2 f = apart_share(at, n, tid, 64, pi.x, pi.y, eci, e0, e1,
                                          [=](int e) { return ew ? W * (double)ew[e] : W; }, law);
            fx = wave_sum(f.x);
            fy = wave_sum(f.y);
        }
    }
    if (tid == 0) {
        dst[i] = moved(pi, fx, fy, stepp ? *stepp : step);
        eterm[i] = fx * fx + fy * fy;
    }
}

__global__ __launch_bounds__(WG) void k_copy(const double2 *__restrict__ src, double2 *__restrict__ dst, int n) {
    const int i = (int)blockIdx.x * WG + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

// FP64 reference-order pair kernel.  grid = (ceil(n/512), rows of 16 batch vertices, in y and z);
// block x covers the reference's j block [512x, 512x+512) for a row.
//
// A block's partial is a chain of 512 additions in j order, but the terms don't depend on the chain:
// four waves form the terms of a tile of 64 positions (IEEE division, or the attraction at a
// neighbour) in LDS while the fifth adds the tile before, a lane per vertex and component.  A pair
// that adds nothing has the term 0, which leaves a sum that began with +0 as it is.  The neighbours
// met in the block are bits in LDS, found once.  With one lane a vertex for both (division on the chain,
// 20 workgroups for 10k vertices) a batch step of 10,007 vertices took 82 us, now 14 (18 with tiles of
// 128); the chain is 2 of them.
constexpr int SLOTS64 = 16, TILE64 = 64, ROWS64 = 32768;  // slots a row, positions a tile, rows in y

__global__ __launch_bounds__(64 + WG) void k_pairs64(const double2 *__restrict__ pos, int n, int b0, int bc,
                                                     double2 *__restrict__ part, int P, const int *__restrict__ erp,
                                                     const int *__restrict__ eci, const float *__restrict__ ew,
                                                     double W, int law) {
    __shared__ double2 q[kBlockY];
    __shared__ double2 term[2][TILE64][SLOTS64];
    __shared__ unsigned met[SLOTS64][kBlockY / 32];  // bit u - jb: column u is a neighbour
    __shared__ int first[SLOTS64];                   // the block's first neighbour entry
    const int tid = threadIdx.x;
    const int jb = (int)blockIdx.x * kBlockY, nj = min(n, jb + kBlockY) - jb;
    const int s0 = ((int)blockIdx.z * ROWS64 + (int)blockIdx.y) * SLOTS64;
    if (s0 >= bc) return;
    for (int u = tid; u < kBlockY; u += 64 + WG) q[u] = pos[jb + min(u, nj - 1)];
    for (int k = tid; k < SLOTS64 * (kBlockY / 32); k += 64 + WG) (&met[0][0])[k] = 0;
    if (tid < SLOTS64) first[tid] = 0x7fffffff;
    __syncthreads();
    const int w = tid - 64;  // a producer's number
    const int slot = w & (SLOTS64 - 1), jl = w >> 4;
    const int i = b0 + min(s0 + (slot & (SLOTS64 - 1)), bc - 1);
    double2 v = make_double2(0.0, 0.0);
    if (w >= 0) {
        v = pos[i];
        const int kend = erp[i + 1];
        int lo = erp[i], hi = kend;
        while (hi - lo > 64) {  // first neighbour >= jb (the merge pointer's state at the block start): in [lo, hi]
            const int m = (lo + hi) >> 1;
            if (eci[m] < jb) lo = m + 1; else hi = m;
        }
        for (int e = lo + jl; e < kend; e += WG / SLOTS64) {
            const int c = eci[e] - jb;
            if (c >= nj) break;
            if (c >= 0) {
                atomicOr(&met[slot][c >> 5], 1u << (c & 31));
                atomicMin(&first[slot], e);
            }
        }
    }
    __syncthreads();
    const int tiles = (nj + TILE64 - 1) / TILE64;
    double f = 0.0;
    for (int t = 0; t <= tiles; ++t) {
        if (w >= 0) {
            if (t < tiles) {
                unsigned near = 0;  // neighbours among this thread's positions: one copy of their code, after
#pragma unroll
                for (int k = 0; k < TILE64; k += WG / SLOTS64) {  // :764-768
                    const int u = t * TILE64 + k + jl;
                    const double2 p = q[u];
                    const double dx = p.x - v.x, dy = p.y - v.y;
                    const double dist = dx * dx + dy * dy;
                    const double inv = 1.0 / dist;
                    const bool in = u < nj && dist > 0;
                    term[t & 1][k + jl][slot] = make_double2(in ? -(dx * inv) : 0.0, in ? -(dy * inv) : 0.0);
                    near |= (met[slot][u >> 5] >> (u & 31) & 1) << (k / (WG / SLOTS64));
                }
                for (; near; near &= near - 1) {  // :758-762
                    const int k = __ffs(near) - 1, u = t * TILE64 + k * (WG / SLOTS64) + jl;
                    int e = first[slot] + __popc(met[slot][u >> 5] & ((1u << (u & 31)) - 1));
                    for (int r = 0; r < u >> 5; ++r) e += __popc(met[slot][r]);
                    double tx = 0.0, ty = 0.0;
                    attract64(law, ew ? W * (double)ew[e] : W, q[u].x - v.x, q[u].y - v.y, tx, ty);
                    term[t & 1][k * (WG / SLOTS64) + jl][slot] = make_double2(tx, ty);
                }
            }
        } else if (t > 0) {
            const double *col = &term[(t - 1) & 1][0][0].x + (tid & (2 * SLOTS64 - 1));
#pragma unroll 16
            for (int k = 0; k < TILE64; ++k) f += col[2 * SLOTS64 * k];
        }
        __syncthreads();
    }
    if (tid < 2 * SLOTS64 && s0 + tid / 2 < bc)
        (&part[(size_t)(s0 + tid / 2) * P + blockIdx.x].x)[tid & 1] = f;
}

// FP32 path: one workgroup per batch vertex sums its G chunk partials and its correction
// pieces (FP64, fixed order: strided per thread, then a fixed tree).
__global__ __launch_bounds__(WG) void k_move32(const double2 *__restrict__ part, int P, int G,
                                               const int *__restrict__ cpre, double2 *__restrict__ pos, int b0,
                                               int bc, const double *__restrict__ stepp, double step,
                                               double *__restrict__ eterm) {
    __shared__ double2 red[WG / 64];
    const int slot = (int)blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if (slot >= bc) return;
    const int i = b0 + slot;
    const double2 *row = part + (size_t)slot * P;
    // Loads that wait for nothing are issued together: the vertex's position, its number of
    // correction pieces, and the G chunk partials, which every row has whatever that number;
    // the pieces follow in the same per-thread order (p = tid, tid + WG, ...).
    const double2 x0 = pos[i];
    const int pe = G + (cpre[i + 1] - cpre[i]);
    double sx = 0.0, sy = 0.0;
    int p = tid;
    for (; p < G; p += WG) {
        const double2 v = row[p];
        sx += v.x;
        sy += v.y;
    }
    for (; p < pe; p += WG) {
        const double2 v = row[p];
        sx += v.x;
        sy += v.y;
    }
    sx = wave_sum(sx);
    sy = wave_sum(sy);
    if (lane == 0) red[w] = make_double2(sx, sy);
    __syncthreads();
    if (tid == 0) {
        double fx = (red[0].x + red[1].x) + (red[2].x + red[3].x);
        double fy = (red[0].y + red[1].y) + (red[2].y + red[3].y);
        if (isnan(fx))
            for (p = G; p < pe; ++p)
                if (__double_as_longlong(row[p].x) == APART) fx = row[p].y, fy = eterm[i];
        pos[i] = moved(x0, fx, fy, stepp ? *stepp : step);
        eterm[i] = fx * fx + fy * fy;
    }
}

// FP64 mode: prevCoordinates[i] += f per j block in block order (:771), then the move.  A lane per
// vertex and component, eight partials loaded at a time.
__global__ __launch_bounds__(64) void k_move64(const double2 *__restrict__ part, int P, double2 *__restrict__ pos,
                                               int b0, int bc, const double *__restrict__ stepp, double step,
                                               double *__restrict__ eterm) {
    const int slot = (int)blockIdx.x * 32 + threadIdx.x / 2, c = threadIdx.x & 1;
    const double *row = &part[(size_t)min(slot, bc - 1) * P].x + c;
    double s = 0.0;
#pragma unroll 8
    for (int p = 0; p < P; ++p) s += row[2 * p];
    const double other = __shfl_xor(s, 1);
    if (slot < bc && c == 0) move_one(pos, b0 + slot, s, other, stepp ? *stepp : step, eterm);
}

// STEP for a captured graph lives on the device so that one iteration's launches are the same every
// iteration: set once, then multiplied after each iteration with the host's FP64 operation.
// Otherwise it is an argument of the launches.
__global__ void k_step_set(double *stepp, double v) {
    if (threadIdx.x == 0) *stepp = v;
}
__global__ void k_step_decay(double *stepp, double decay) {
    if (threadIdx.x == 0) *stepp = *stepp * decay;  // :781 (0.999), :934 / :1007 (0.99)
}

}  // namespace

// ---- the non-finite guard -------------------------------------------------------------
__global__ void k_zero_int(int *p) {
    if (threadIdx.x == 0) *p = 0;
}

// One vector atomic per wave that holds a non-finite coordinate.
__global__ __launch_bounds__(256) void k_count_nonfinite(const double2 *__restrict__ pos, int n, int *count) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    bool bad = false;
    if (i < n) {
        const double2 p = pos[i];
        bad = !isfinite(p.x) || !isfinite(p.y);
    }
    const uint64_t m = __ballot(bad);
    if (m && (threadIdx.x & 63) == (int)(__builtin_ctzll(m))) atomicAdd(count, __popcll(m));
}

int count_nonfinite(const double2 *pos, int n, int *d_count, hipStream_t s, int *h_count) {
    hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(64), 0, s, d_count);
    if (n > 0) hipLaunchKernelGGL(k_count_nonfinite, dim3((n + 255) / 256), dim3(256), 0, s, pos, n, d_count);
    BL_HIP(hipGetLastError());
    BL_HIP(hipMemcpyAsync(h_count, d_count, sizeof(int), hipMemcpyDeviceToHost, s));
    BL_HIP(hipStreamSynchronize(s));
    return BL_OK;
}

// ---- energy reductions (shared with the Barnes-Hut path) -------------------------------
// Energy sum_i |F_i|^2 (not FP64 mode's) and the number of positions that are not finite, in two
// fixed-order stages: ENERGY_PARTS workgroups each add a contiguous share (threads strided, then a
// wave and workgroup reduction), then one wave adds the shares in order.  Deterministic.  One copy
// and one wait bring both to the host (EnergyOut); a count of its own took two more launches, a copy and
// a wait, about 20 us of a run.
__global__ __launch_bounds__(256) void k_energy_part(const double *__restrict__ eterm, const double2 *__restrict__ pos,
                                                     int n, EnergyOut *out) {
    __shared__ double red[4];
    __shared__ int bad[4];
    const int ch = (n + ENERGY_PARTS - 1) / ENERGY_PARTS;
    const int i0 = blockIdx.x * ch, i1 = min(n, i0 + ch);
    double a = 0.0, b = 0.0;
    int k = 0;
    auto count = [&](int i) {
        const double2 p = pos[i];
        k += isfinite(p.x) && isfinite(p.y) ? 0 : 1;
    };
    int i = i0 + (int)threadIdx.x;
    for (; i + 256 < i1; i += 512) {
        a += eterm[i];
        b += eterm[i + 256];
        count(i);
        count(i + 256);
    }
    if (i < i1) {
        a += eterm[i];
        count(i);
    }
    a = wave_sum(a + b);
#pragma unroll
    for (int off = 32; off; off >>= 1) k += __shfl_xor(k, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a, bad[threadIdx.x >> 6] = k;
    __syncthreads();
    if (threadIdx.x == 0) {
        out->share[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
        out->bad_share[blockIdx.x] = bad[0] + bad[1] + bad[2] + bad[3];
    }
}

__global__ __launch_bounds__(64) void k_energy_final(EnergyOut *out) {
    double a = 0.0;
    int bad = 0;
    for (int k = threadIdx.x; k < ENERGY_PARTS; k += 64) a += out->share[k], bad += out->bad_share[k];
    a = wave_sum(a);
#pragma unroll
    for (int off = 32; off; off >>= 1) bad += __shfl_xor(bad, off, 64);
    if (threadIdx.x == 0) {
        out->energy = a;
        out->nonfinite = bad;
    }
}

// Sequential sum in vertex order, ENERGY += |F_i|^2 as the reference (FP64 mode): one wave adds a
// tile from LDS while the others load the next, so that the chain of additions is what takes the time
// (10,007 terms: 50 us, 11 cycles a term; 362 with one thread loading each term).
constexpr int SEQ_TILE = 1536;  // 8 loads a thread of three waves
__global__ __launch_bounds__(256) void k_energy_seq(const double *__restrict__ eterm, int n, double *out) {
    __shared__ double buf[2][SEQ_TILE];
    const int w = (int)threadIdx.x - 64;
    const int tiles = (n + SEQ_TILE - 1) / SEQ_TILE;
    double e = 0.0;
    for (int t = 0; t <= tiles; ++t) {
        if (w >= 0) {
#pragma unroll
            for (int k = 0; k < SEQ_TILE / 192; ++k) {
                const int i = t * SEQ_TILE + 192 * k + w;
                buf[t & 1][192 * k + w] = i < n ? eterm[i] : 0.0;  // |F|^2 >= 0: adding 0 changes nothing
            }
        } else if (t > 0) {
            const double *col = buf[(t - 1) & 1];
            double a[16], b[16];  // read one group while the other is added
#pragma unroll
            for (int k = 0; k < 16; ++k) a[k] = col[k];
            for (int g = 0; g < SEQ_TILE; g += 32) {
#pragma unroll
                for (int k = 0; k < 16; ++k) b[k] = col[g + 16 + k];
#pragma unroll
                for (int k = 0; k < 16; ++k) e += a[k];
#pragma unroll
                for (int k = 0; k < 16; ++k) a[k] = col[min(g + 32, SEQ_TILE - 16) + k];
#pragma unroll
                for (int k = 0; k < 16; ++k) e += b[k];
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = e;
}

int launch_energy(const double *eterm, const double2 *pos, int n, EnergyOut *out, int precision, hipStream_t s) {
    hipLaunchKernelGGL(k_energy_part, dim3(ENERGY_PARTS), dim3(256), 0, s, eterm, pos, n, out);
    hipLaunchKernelGGL(k_energy_final, dim3(1), dim3(64), 0, s, out);
    if (precision == BL_PREC_FP64)
        hipLaunchKernelGGL(k_energy_seq, dim3(1), dim3(256), 0, s, eterm, n, &out->energy);
    BL_HIP(hipGetLastError());
    return BL_OK;
}

// ---- the static workspace (bl_run_device_static) ------------------------------------------
// One array per GPU, held until the process ends.  On the host its name stands for a host-side
// placeholder, not device memory, so host code uses only the device address that
// hipGetSymbolAddress returns, looked up once per device with that device current.
static __device__ __align__(256) unsigned char scratch[BL_STATIC_SCRATCH_BYTES];

constexpr int MAX_DEVICES = 64;

static int static_scratch(int device, unsigned char **out) {
    static std::mutex mu;
    static void *addr[MAX_DEVICES] = {};
    if (device < 0 || device >= MAX_DEVICES) return BL_E_DEVICE;
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[device]) {
        int cur = -1;
        BL_HIP(hipGetDevice(&cur));
        if (cur != device) BL_HIP(hipSetDevice(device));
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != device) (void)hipSetDevice(cur);
        if (e != hipSuccess) return device_error(e, "hipGetSymbolAddress(scratch)", __LINE__);
        if (!p) return BL_E_DEVICE;
        addr[device] = p;
    }
    *out = static_cast<unsigned char *>(addr[device]);
    return BL_OK;
}

static size_t round256(size_t b) { return (b + 255) & ~(size_t)255; }

// One launch a step (k_step32) or two (k_pairs32, k_move32).  A step of one launch takes 3.8 us and
// each workgroup's pass over all positions, one of two 6.6 us and its pairs at the whole chip's rate.
// us a step, two launches / one, by n (random geometric graphs):
//   -batch    1,000        4,000        10,000       20,000        40,000
//     64      6.6 / 3.8    6.5 / 3.9    6.8 / 5.2    7.1 / 6.0     7.1 / 7.9
//    256      8.4 / 5.3    7.2 / 5.0    6.8 / 6.2    7.6 / 6.9     8.8 / 8.8
//  1,024     14.9 / 12.2   9.9 / 7.8   11.0 / 9.5   13.7 / 13.7   20.7 / 24.6
// Threads a vertex: 1,024 where 256 would each take many positions and a CU has one vertex (10,000 at
// -batch 256: 6.2 us against 6.3, 20,000: 6.9 against 7.7; 4,000: 5.0 both); with more vertices a CU
// 256 (10,000 at -batch 1,024: 9.5 against 15.9).
constexpr int STEP_ONE_MAX = 20480, STEP_ONE_BATCH = 1024, STEP_WIDE = 8192;
static bool one_launch(int n, int bmax) {
    if (const char *e = getenv("BL_STEP_LAUNCHES"))  // tests
        if (atoi(e) == 2) return false;
    return n <= STEP_ONE_MAX && bmax <= STEP_ONE_BATCH;
}
// The second array never makes a layout too large for the static workspace.
static_assert(4096 + 24u * (STEP_ONE_MAX + 64) <= BL_STATIC_SCRATCH_BYTES, "two arrays exceed the workspace");

int run_minibatch(bl_graph *g, double *d_xy, const bl_params *p, int law, double decay, double step0, int iters,
                  bool converged, bl_stats *st, bool static_ws) {
    const int n = g->n;
    const int B = p->batch;
    const int nb = (n + B - 1) / B;
    const int bmax = B < n ? B : n;
    const bool fp64 = p->precision == BL_PREC_FP64;
    hipStream_t s = g->stream;
    double2 *pos = reinterpret_cast<double2 *>(d_xy);
    const int *erp = g->eff_rowptr.as<int>();
    const int *eci = g->eff_colids.as<int>();
    const float *ew = g->has_w ? g->eff_w.as<float>() : nullptr;

    // launch geometry
    int JS = 1, G = 1, chunk = n, P = 1;
    size_t part_elems = 0;
    if (fp64) {
        G = (n + kBlockY - 1) / kBlockY;
        P = G;
        part_elems = (size_t)bmax * P;
    } else {
        // 64 batch slots x 4 j-subgroups per workgroup: at least ~1024 workgroups (4 per CU),
        // and j chunks of at most ~CHUNK_MAX positions, whose scalar loads the rows of a chunk
        // then mostly share in the scalar cache
        constexpr int CHUNK_MAX = 1024;
        JS = 4;
        const int ipw = WG / JS;
        const int rows = (bmax + ipw - 1) / ipw;
        const int target = std::max(std::max(1, 1024 / rows), (n + CHUNK_MAX - 1) / CHUNK_MAX);
        const int quant = UNROLL * JS;
        chunk = (n + target - 1) / target;
        chunk = ((chunk + quant - 1) / quant) * quant;
        G = (n + chunk - 1) / chunk;
        P = G + g->corr_max_pieces;
        part_elems = (size_t)bmax * P;
    }
    const bool one = !fp64 && one_launch(n, bmax);
    const size_t a_elems = one ? (size_t)n : part_elems;  // the second position array in the partials' place
    double2 *part;
    double *eterm;
    EnergyOut *energy;
    if (static_ws) {
        // [energy shares | partial forces | energy terms]; every word a step reads is written
        // earlier in the same step, so the contents of the previous call do not matter
        static_assert(sizeof(EnergyOut) <= 4096, "energy shares exceed their part");
        const size_t off_part = 4096;
        const size_t off_eterm = off_part + round256(sizeof(double2) * std::max(a_elems, part_elems));
        const size_t need = off_eterm + round256(sizeof(double) * (size_t)n);
        if (need > BL_STATIC_SCRATCH_BYTES) return BL_E_SCRATCH;
        unsigned char *ws = nullptr;
        const int rc = static_scratch(g->device, &ws);
        if (rc) return rc;
        energy = reinterpret_cast<EnergyOut *>(ws);
        part = reinterpret_cast<double2 *>(ws + off_part);
        eterm = reinterpret_cast<double *>(ws + off_eterm);
    } else {
        if (g->part.ensure(sizeof(double2) * a_elems)) return BL_E_NOMEM;
        if (g->eterm.ensure(sizeof(double) * (size_t)n)) return BL_E_NOMEM;
        if (g->energy.ensure(sizeof(EnergyOut))) return BL_E_NOMEM;
        part = g->part.as<double2>();
        eterm = g->eterm.as<double>();
        energy = g->energy.as<EnergyOut>();
    }

    Prof prof;
    prof.on = p->profile != 0;
    prof.s = s;
    const char *genv = getenv("BL_GRAPH");
    const bool want_graph = !prof.on && !static_ws && (converged || iters >= 2) && genv && !strcmp(genv, "1");
    double STEP = step0;
    double *const d_step = want_graph ? &energy->step : nullptr;  // else a launch's argument
    if (want_graph) hipLaunchKernelGGL(k_step_set, dim3(1), dim3(64), 0, s, d_step, step0);
    // One launch a step: the array that the next step reads, and the batch that the other one lacks.
    // The steps' number is known (or made even, each iteration) so that the last one writes pos.
    double2 *const both[2] = {pos, part};
    const bool even_out = converged || want_graph;
    int cur = even_out ? 0 : (int)((int64_t)iters * nb & 1), p0 = 0, pc = 0;
    if (one && (converged || iters > 0))
        hipLaunchKernelGGL(k_copy, dim3((n + WG - 1) / WG), dim3(WG), 0, s, pos, part, n);
    // One iteration's launches: every batch step (pairs, then the move), the energy, STEP *= decay.
    auto emit_iteration = [&](bool energy_seen) -> int {
        for (int b = 0; b < nb; ++b) {
            const int b0 = b * B;
            const int bc = (n - b0) < B ? (n - b0) : B;
            if (one) {
                hipEvent_t e0 = nullptr, e1 = nullptr;
                if (prof.on) prof.ext(0, &e0, &e1);
                const auto go = [&](auto kernel, int threads) {
                    if (prof.on)  // the dispatch records its own start and end
                        hipExtLaunchKernelGGL(kernel, dim3(bc), dim3(threads), 0, s, e0, e1, 0, both[cur],
                                              both[cur ^ 1], n, p0, nb > 1 ? pc : 0, b0, erp, eci, ew, p->weight, law,
                                              d_step, STEP, eterm);
                    else
                        hipLaunchKernelGGL(kernel, dim3(bc), dim3(threads), 0, s, both[cur], both[cur ^ 1], n, p0,
                                           nb > 1 ? pc : 0, b0, erp, eci, ew, p->weight, law, d_step, STEP, eterm);
                };
                const bool wide = n > STEP_WIDE && bmax <= 256;
                if (p->precision == BL_PREC_FP32)
                    wide ? go(k_step32<1024, false>, 1024) : go(k_step32<256, false>, 256);
                else
                    wide ? go(k_step32<1024, true>, 1024) : go(k_step32<256, true>, 256);
                cur ^= 1;
                p0 = b0, pc = bc;
            } else if (fp64) {
                prof.begin(0);
                const int rows = (bc + SLOTS64 - 1) / SLOTS64;
                hipLaunchKernelGGL(k_pairs64, dim3(G, std::min(rows, ROWS64), (rows + ROWS64 - 1) / ROWS64),
                                   dim3(64 + WG), 0, s, pos, n, b0, bc, part, P,
                                   erp, eci, ew, p->weight, law);
                prof.end();
                prof.begin(1);
                hipLaunchKernelGGL(k_move64, dim3((bc + 31) / 32), dim3(64), 0, s, part, P, pos, b0, bc, d_step, STEP,
                                   eterm);
                prof.end();
            } else {
                const int ipw = WG / JS;
                const int pc0 = g->h_cpre[b0], npc = g->h_cpre[b0 + bc] - pc0;
                const dim3 grid(G + (npc + 3) / 4, (bc + ipw - 1) / ipw);
                const int *cpre = g->cpre.as<int>(), *cpv = g->cpv.as<int>();
                if (prof.on) {  // the dispatch records its own start and end
                    hipEvent_t e0, e1;
                    prof.ext(0, &e0, &e1);
                    if (p->precision == BL_PREC_FP32)
                        hipExtLaunchKernelGGL((k_pairs32<4, false>), grid, dim3(WG), 0, s, e0, e1, 0, pos, n, b0, bc,
                                              chunk, G, part, P, erp, eci, ew, p->weight, law, cpre, cpv, pc0, npc, eterm);
                    else
                        hipExtLaunchKernelGGL((k_pairs32<4, true>), grid, dim3(WG), 0, s, e0, e1, 0, pos, n, b0, bc,
                                              chunk, G, part, P, erp, eci, ew, p->weight, law, cpre, cpv, pc0, npc, eterm);
                    prof.ext(1, &e0, &e1);
                    hipExtLaunchKernelGGL(k_move32, dim3(bc), dim3(WG), 0, s, e0, e1, 0, part, P, G, cpre, pos, b0, bc,
                                          d_step, STEP, eterm);
                } else {
                    if (p->precision == BL_PREC_FP32)
                        hipLaunchKernelGGL((k_pairs32<4, false>), grid, dim3(WG), 0, s, pos, n, b0, bc, chunk, G, part,
                                           P, erp, eci, ew, p->weight, law, cpre, cpv, pc0, npc, eterm);
                    else
                        hipLaunchKernelGGL((k_pairs32<4, true>), grid, dim3(WG), 0, s, pos, n, b0, bc, chunk, G, part,
                                           P, erp, eci, ew, p->weight, law, cpre, cpv, pc0, npc, eterm);
                    hipLaunchKernelGGL(k_move32, dim3(bc), dim3(WG), 0, s, part, P, G, cpre, pos, b0, bc, d_step,
                                       STEP, eterm);
                }
            }
        }
        if (one && even_out && cur) {  // the last step wrote the other array: its batch is what pos lacks
            hipLaunchKernelGGL(k_copy, dim3((pc + WG - 1) / WG), dim3(WG), 0, s, part + p0, pos + p0, pc);
            cur = pc = 0;
        } else if (one && want_graph) {  // a replay begins with both arrays complete, as the captured iteration
            hipLaunchKernelGGL(k_copy, dim3((pc + WG - 1) / WG), dim3(WG), 0, s, pos + p0, part + p0, pc);
            pc = 0;
        }
        int rc = BL_OK;
        if (energy_seen) {
            prof.begin(2);
            rc = launch_energy(eterm, pos, n, energy, p->precision, s);
            prof.end();
        }
        if (want_graph) hipLaunchKernelGGL(k_step_decay, dim3(1), dim3(64), 0, s, d_step, decay);
        return rc;
    };
    // BL_GRAPH=1 (and no per-launch timing): one iteration is captured once as a graph and
    // replayed, one host launch per iteration instead of two per batch step.  Not the default:
    // measured on MI355X (ROCm 7) the replay was no faster (64x64 grid 96 vs 95 us per iteration,
    // 32x32 grid 32 vs 28 us, 250k vertices 28.6 vs 28.0 ms): the GPU's own dispatch of
    // dependent small kernels, not the host's launch calls, sets the pace.  The static-workspace
    // path creates no graph (instantiation allocates).
    struct Exec {
        hipGraphExec_t e = nullptr;
        ~Exec() {
            if (e) (void)hipGraphExecDestroy(e);
        }
    } ex;
    if (want_graph && hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) == hipSuccess) {
        const int rc = emit_iteration(true);
        hipGraph_t gr = nullptr;
        const hipError_t ee = hipStreamEndCapture(s, &gr);
        if (rc == BL_OK && ee == hipSuccess && gr) {
            if (hipGraphInstantiate(&ex.e, gr, nullptr, nullptr, 0) != hipSuccess) ex.e = nullptr;
        }
        if (gr) (void)hipGraphDestroy(gr);
        (void)hipGetLastError();  // a failed capture leaves the launches to the loop below
    }
    EnergySeen seen;
    double E = 0.0, E0 = 1.79769313486231570815e+308;
    int loop = 0;
    for (;;) {
        if (converged) {
            if (!(fabs(E0 - E) / E0 > p->engt)) break;  // algorithms.cpp:818
        } else if (loop >= iters) {
            break;
        }
        E0 = E;
        if (ex.e) {
            BL_HIP(hipGraphLaunch(ex.e, s));
        } else {
            const int rc = emit_iteration(converged || want_graph || loop == iters - 1);
            if (rc) return rc;
            prof.flush();
        }
        STEP = STEP * decay;  // the host's copy (the device multiplies its own the same way)
        ++loop;
        if (converged) {
            BL_HIP(hipMemcpyAsync(&seen, energy, sizeof(seen), hipMemcpyDeviceToHost, s));
            BL_HIP(hipStreamSynchronize(s));
            E = seen.energy;
        }
    }
    BL_HIP(hipGetLastError());
    if (!converged && loop > 0) BL_HIP(hipMemcpyAsync(&seen, energy, sizeof(seen), hipMemcpyDeviceToHost, s));
    BL_HIP(hipStreamSynchronize(s));
    if (loop > 0) E = seen.energy;
    prof.report(st);
    if (st) {
        st->energy = loop > 0 ? E : (law == LAW_FR ? 0.0 : 1.79769313486231570815e+308);
        st->iters_done = loop;
        st->step_final = STEP;
        if (loop > 0) {
            st->nonfinite = seen.nonfinite;
        } else if (static_ws) {  // nothing ran: counted here, in the energy block
            int nf = 0;
            const int rc = count_nonfinite(pos, n, &energy->nonfinite, s, &nf);
            if (rc) return rc;
            st->nonfinite = nf;
        }
    }
    return BL_OK;
}

}  // namespace bl
