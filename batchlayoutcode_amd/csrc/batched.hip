// Many small graphs in one persistent launch (bl_run_batched).
//
// Each graph follows the single-graph minibatch algorithm (algorithms.cpp:715-794 for algo 2,
// :947-1018 for algo 8): ceil(n/B) batches per iteration, Jacobi inside a batch, Gauss-Seidel
// across batches, x_i += STEP*F/|F|, STEP *= decay, with the pair arithmetic and neighbour
// correction of pair_math.h.  Workgroups of 1024 threads pull graphs from an atomic work
// queue (largest n^2 first) and run all of a graph's iterations: the graph's FP64
// positions sit in LDS when they fit (read by every lane with the same address, i.e.
// broadcast) and are read from global memory otherwise.
//
// Inside a batch step IPW batch slots (a power of two, 64..1024, per graph) are served at once
// by JS = 1024 / IPW j-subgroups, in rounds of IPW slots.  The j range is cut into NCH fixed
// chunks (16 to 256, by the graph's size and -batch alone) whose partials are combined by one fixed pairwise
// tree, ((c0 + c1) + (c2 + c3)) + ..., whatever the shape: a subgroup sums its consecutive chunks
// as the subtree they form, and the subgroups' subtrees are combined as the rest of the tree.  So
// every shape gives the same bits, and the shape is free to be tuned (run_batched measures the
// candidates per size class of the graphs); the neighbour correction follows.  Results do not
// depend on timing either.
//
// A step has two barriers (after the dense sums, after the moves): the lanes of a row, BT / (slots in one
// round), share its neighbours' corrections, which come from the positions before the step and so go
// first, and combine its subtrees by DPP moves; the next batch's neighbour lists are loaded behind the
// dense sum.  The dense sum is bound by FP64 operations (13.7 pairs a ns and CU); the rest of a step
// takes 4 us (8.6 with a thread per row after the sum and five barriers).
//
// Teams.  One workgroup takes 87 us a step for a graph of 8192 vertices at -batch 128, so a launch
// of few graphs, or of many with a few large ones, waits for its largest graphs while most CUs are
// idle.  The largest graphs are therefore laid out by teams of T workgroups (2 to 16): each member
// holds the whole graph in its own LDS, sums 1/T of the chunks for every slot of the batch, stores
// these partials, waits for the other members', combines all of them in the same tree and moves the
// batch in its own copy.  One hand-off per batch step (about 4.5 us); every member forms the same
// positions, member 0 writes them.  What is handed over is stored with agent-scope stores, which
// the XCD's L2 writes through to memory: once they have completed, a relaxed counter publishes them,
// and a member that has seen the count reads them with agent-scope loads.  Two buffers in turn: a member
// writes a buffer again only after the next step's count, when all have read it.  The teams take the
// first places of the queue and together at most the workgroups that run at once, so their members
// start together.  Where they don't (the device is busy with other launches), a wait ends at a
// deadline, its team gives up (the others go on), and a second launch without teams lays out its graph, whose
// positions in memory are still the initial ones.  Launches of graphs of 64..8192
// vertices, 20 iterations, without and with teams: 16 graphs 97.0 and 16.1 ms, 200 (-batch 64) 108 and
// 35.7, 1,500 107 and 83.9.
#include <math.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <numeric>
#include <tuple>
#include <vector>

#include "bh_common.h"
#include "pair_math.h"
#include "traverse.h"

namespace bl {
namespace {

constexpr int BT = 1024;       // threads per workgroup
constexpr int MAXB = 1024;     // largest batch size of the batched path
constexpr int MAXTEAM = 16;    // largest team

// The slots served at once where a batch of bc takes one round: a power of two from 64.
__host__ __device__ inline int one_round(int bc) {
    int w = 64;
    while (w < bc && w < BT) w <<= 1;
    return w;
}

// Fixed j chunks of the dense sum: 16, at which every shape has one a subgroup; for larger graphs
// with small batches more, of 32 positions or more, up to 16 for each subgroup of the one round, for
// the teams to share.  A chunk costs a little besides its pairs (a step of 4,096 vertices at -batch 128
// takes 49.3 us with 32 positions a chunk, 48.4 with 64), but with fewer chunks teams stay small: 200
// graphs of 64..8192 vertices at -batch 64 take 35.7 ms with 32, 48.1 with 64.
__host__ __device__ inline int chunks_of(int n, int B) {
    const int most = 16 * (BT / one_round(n < B ? n : B));
    int c = 16;
    while (2 * c <= most && 64 * c <= n) c <<= 1;
    return c;
}

struct BatchedArgs {
    const int2 *items;         // the queue: {graph, team member}, largest graphs first
    const int *ipw_of;         // batch slots served at once, per graph (power of two, 64..1024)
    int count;                 // items
    const int *team;           // team size per graph (null: no teams)
    const int *team_at;        // a team's place in parts and arrived
    double2 *parts;            // [team][2][MAXTEAM][B] members' partials, by step parity
    int *arrived;              // [team] members that stored their partials, summed over the steps
    int *err;                  // [team] a wait that ran out
    long long ticks;           // longest wait
    const int *voff;           // vertex offsets [count+1]
    const int *rp;             // row pointers over all vertices (global entry ids)
    const int *rend;           // the end of a row's effective neighbours (k_row_ends)
    const int *ci;             // column ids (graph-local)
    double2 *pos;              // all positions
    int B, iters, law, lds_cap;
    double step0, decay, W;
    double *energies;
    long long *finish;         // wall-clock tick at each graph's completion
    long long *wg_start;       // wall-clock tick at each workgroup's start
    int *queue;
};

typedef __attribute__((address_space(3))) const double lds_double;

// Pairwise combination in a fixed tree: leaves arrive left to right, level l holds the pending
// left subtree of 2^l leaves; after 2^L leaves (L <= 4) level L holds their sum,
// ((v0 + v1) + (v2 + v3)) + ...  Branches on the leaf count k (the same in every lane) skip the levels
// a leaf doesn't reach; a level is set by a select: an else branch that sets another one, or an
// indexed array, goes to scratch memory, whose loads took half the time of a chunk of 32 positions.
struct PairTree {
    double x0 = 0.0, y0 = 0.0, x1 = 0.0, y1 = 0.0, x2 = 0.0, y2 = 0.0, x3 = 0.0, y3 = 0.0, x4 = 0.0, y4 = 0.0;
    int k = 0;
    __device__ __forceinline__ void add(double vx, double vy) {
        double sx = x0 + vx, sy = y0 + vy;  // close the subtrees this leaf completes, left operand first
        x0 = k & 1 ? x0 : vx, y0 = k & 1 ? y0 : vy;
        if (k & 1) {
            vx = sx, vy = sy, sx = x1 + vx, sy = y1 + vy;
            x1 = k & 2 ? x1 : vx, y1 = k & 2 ? y1 : vy;
            if (k & 2) {
                vx = sx, vy = sy, sx = x2 + vx, sy = y2 + vy;
                x2 = k & 4 ? x2 : vx, y2 = k & 4 ? y2 : vy;
                if (k & 4) {
                    vx = sx, vy = sy, sx = x3 + vx, sy = y3 + vy;
                    x3 = k & 8 ? x3 : vx, y3 = k & 8 ? y3 : vy;
                    if (k & 8) x4 = sx, y4 = sy;
                }
            }
        }
        ++k;
    }
    __device__ __forceinline__ double2 total(int L) const {
        const double x = L == 0 ? x0 : L == 1 ? x1 : L == 2 ? x2 : L == 3 ? x3 : x4;
        const double y = L == 0 ? y0 : L == 1 ? y1 : L == 2 ? y2 : L == 3 ? y3 : y4;
        return make_double2(x, y);
    }
};

// The subtree of chunks [c0, c0 + cpt) of `sub` positions (whole groups of 8) for position p.
template <bool REFINE, class Src>
__device__ __forceinline__ double2 chunk_sums(Src src, int n, int c0, int cpt, int sub, double2 p) {
    PairTree t;
    int j = c0 * sub;
    for (int c = 0; c < cpt; ++c) {
        const int j1 = min(n, (c0 + c + 1) * sub);
        double ax = 0.0, ay = 0.0;
        for (; j + 8 <= j1; j += 8) {
            double qx[8], qy[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) qx[k] = src[2 * (j + k)], qy[k] = src[2 * (j + k) + 1];
            pair_rep_group<REFINE, 8>(qx, qy, p.x, p.y, ax, ay);
        }
        if constexpr (REFINE) {
            if (j < j1) add_group<8, false>(interleaved(src), j, 1, j1, p.x, p.y, ax, ay), j = j1;
        } else {
            for (; j < j1; ++j) pair_rep<false>(src[2 * j], src[2 * j + 1], p.x, p.y, ax, ay);
        }
        t.add(ax, ay);
    }
    const double2 v = t.total(__builtin_ctz(cpt));
    if (isfinite(v.x) && isfinite(v.y)) return v;
    PairTree u;  // a group's product left the range: each such chunk again, with care
    for (int c = c0; c < c0 + cpt; ++c) {
        double ax, ay;
        dense_sum<REFINE, 8, true>(src, min(n, c * sub), min(n, (c + 1) * sub), p.x, p.y, ax, ay);
        u.add(ax, ay);
    }
    return u.total(__builtin_ctz(cpt));
}

// v summed over `count` (1, 2, 4, 8 or 16) lanes from a multiple of it, pairwise from neighbours up,
// in each of them.
__device__ __forceinline__ double lanes_sum(double v, int count) {
    if (count > 1) v = dpp_add<0xB1, 0xF>(v);   // quad_perm [1, 0, 3, 2]
    if (count > 2) v = dpp_add<0x4E, 0xF>(v);   // quad_perm [2, 3, 0, 1]
    if (count > 4) v = dpp_add<0x141, 0xF>(v);  // row_half_mirror
    if (count > 8) v = dpp_add<0x140, 0xF>(v);  // row_mirror
    return v;
}

// Waits until `need` arrivals of team `at` are counted (modulo 2^32, which 134 million steps of a team of 16
// reach), in thread 0; false at the deadline or after another member's.
__device__ __forceinline__ bool team_wait(const BatchedArgs &a, int at, unsigned need) {
    const long long t0 = wall_clock64();
    while ((int)((unsigned)__hip_atomic_load(a.arrived + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - need) < 0) {
        if (__hip_atomic_load(a.err + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
        if (wall_clock64() - t0 > a.ticks) {
            atomicOr(a.err + at, 1);
            return false;
        }
        __builtin_amdgcn_s_sleep(1);
    }
    return true;
}

// Lays out graph g as member `me` of its team of T workgroups.
template <bool REFINE>
__device__ void layout_graph(const BatchedArgs &a, int g, int me, int T, double2 *P, double2 *red, double2 *fb,
                             double *eb, int *go) {
    const int tid = threadIdx.x;
    const int v0 = __builtin_amdgcn_readfirstlane(a.voff[g]);
    const int n = __builtin_amdgcn_readfirstlane(a.voff[g + 1]) - v0;
    const bool in_lds = n <= a.lds_cap;  // always with a team
    double2 *gp = in_lds ? P : a.pos + v0;
    if (in_lds) {
        for (int k = tid; k < n; k += BT) P[k] = a.pos[v0 + k];
        __syncthreads();
    }
    const int B = a.B;
    const int ipw = __builtin_amdgcn_readfirstlane(a.ipw_of[g]);
    const int nch = chunks_of(n, B);
    const int JS = BT / ipw, cpt = nch / (JS * T);  // subgroups, chunks per subgroup
    const int li = tid & (ipw - 1), js = tid >> __builtin_ctz(ipw);
    const int c0 = (me * JS + js) * cpt;      // this subgroup's first chunk
    const int sub = ((n + nch - 1) / nch + 7) & ~7;  // chunk c: [c * sub, (c + 1) * sub) within [0, n)
    const int nb = (n + B - 1) / B;
    // the L lanes of a batch slot's row: its neighbours, its subtrees, its move
    const int L = BT / one_round(min(B, n)), row = tid >> __builtin_ctz(L), k = tid & (L - 1);
    const bool rounds = one_round(min(B, n)) > ipw;
    const int at = T > 1 ? __builtin_amdgcn_readfirstlane(a.team_at[g]) : 0;
    double2 *parts = a.parts + (size_t)at * 2 * MAXTEAM * B;
    const int share = max(1, T / L);          // members whose subtrees a lane of a row adds
    unsigned need = 0;
    double step = scalar(a.step0), E = 0.0;  // in scalar registers: the vector ones are short
    auto ends = [&](int b) {  // this row's entries in batch b
        const int i = v0 + min(n - 1, b * B + row);
        return make_int2(a.rp[i], a.rend[i]);
    };
    const auto posn = [=](int j) { return gp[j]; };
    auto first = [&](int2 e) { return e.x + k < e.y ? a.ci[e.x + k] : 0; };
    int2 er = ends(0);
    int jn = first(er);
    for (int it = 0; it < a.iters; ++it) {
        for (int b = 0; b < nb; ++b) {
            const int b0 = b * B, bc = min(B, n - b0);
            const bool mine = row < bc;
            const double2 pr = gp[b0 + (mine ? row : 0)];
            double cx = 0.0, cy = 0.0;
            const int law = a.law == LAW_FA ? LAW_FA : LAW_FR;
            bool close = false;
            for (int e = er.x + k; e < er.y; e += L) {
                const int j = e == er.x + k ? jn : a.ci[e];
                const double2 pj = gp[j];
                const double dx = pj.x - pr.x, dy = pj.y - pr.y;
                const double inv = linked_factor<REFINE>(posn, true, j & ~(GROUP - 1), j & (GROUP - 1), 1, n, pr.x, pr.y,
                                                         dx, dy);  // chunks begin at whole groups
                correct_pair(law, a.W, dx, dy, inv, cx, cy);
                close = close || too_close<REFINE>(dx, dy);
            }
            const bool apart = REFINE && (__ballot(close) >> (tid & 63 & ~(L - 1)) & ((1ull << L) - 1)) != 0;
            if (apart) {
                const double2 f = apart_share(posn, n, k, L, pr.x, pr.y, a.ci, er.x, er.y, [&](int) { return a.W; }, law);
                cx = f.x, cy = f.y;
            }
            // the next batch's entries are loaded behind this batch's dense sum
            er = ends(b + 1 < nb ? b + 1 : 0);
            double2 *part = parts + ((need & 1) * MAXTEAM + me) * B;
            for (int r0 = 0; r0 < bc; r0 += ipw) {  // rounds of ipw slots
                const int slot = r0 + li;
                const bool act = slot < bc;
                const double2 pi = gp[b0 + (act ? slot : 0)];
                // LDS broadcasts, or global memory
                red[tid] = in_lds ? chunk_sums<REFINE>((lds_double *)P, n, c0, cpt, sub, pi)
                                  : chunk_sums<REFINE>(reinterpret_cast<const double *>(gp), n, c0, cpt, sub, pi);
                if (rounds) {
                    __syncthreads();
                    if (js == 0 && act) {
                        PairTree u;  // the subgroups' subtrees, in order
                        for (int q = 0; q < JS; ++q) u.add(red[q * ipw + li].x, red[q * ipw + li].y);
                        fb[slot] = u.total(__builtin_ctz(JS));
                    }
                    __syncthreads();
                }
            }
            jn = first(er);
            cx = lanes_sum(cx, L);
            cy = lanes_sum(cy, L);
            double2 f;
            if (rounds) {
                f = fb[mine ? row : 0];
            } else {  // every position has been read
                __syncthreads();
                f = red[min(k, JS - 1) * ipw + (mine ? row : 0)];
                f.x = lanes_sum(f.x, JS);
                f.y = lanes_sum(f.y, JS);
            }
            if (T > 1) {
                if (mine && k == 0) store_through(part + row, f);
                // each wave's stores have completed before the workgroup's arrival is counted
                __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __syncthreads();
                if (tid == 0) {
                    __hip_atomic_fetch_add(a.arrived + at, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    *go = team_wait(a, at, (unsigned)(need + 1) * (unsigned)T);
                }
                __syncthreads();
                if (!__builtin_amdgcn_readfirstlane(*go)) return;
                // the members' subtrees: the top of the tree
                const double2 *all = parts + ((need & 1) * MAXTEAM + min(k, T / share - 1) * share) * B +
                                     (mine ? row : 0);
                PairTree u;
                for (int m = 0; m < share; ++m) {
                    const double2 v = load_through(all + m * B);
                    u.add(v.x, v.y);
                }
                f = u.total(__builtin_ctz(share));
                f.x = lanes_sum(f.x, T / share);
                f.y = lanes_sum(f.y, T / share);
            }
            f.x = apart ? cx : f.x + cx;
            f.y = apart ? cy : f.y + cy;
            // the move (every force of the batch is formed from the positions before it)
            if (mine && k == 0) gp[b0 + row] = moved(gp[b0 + row], f.x, f.y, step);
            if (it == a.iters - 1) {  // the energy: wave sums, then the 16 wave sums in order
                const double e2 = wave_sum(mine && k == 0 ? f.x * f.x + f.y * f.y : 0.0);
                if ((tid & 63) == 0) eb[tid >> 6] = e2;
            }
            __syncthreads();  // the moves are visible to the next batch
            if (it == a.iters - 1) {
                double eb_sum = 0.0;
#pragma unroll
                for (int q = 0; q < BT / 64; ++q) eb_sum += eb[q];
                E = scalar(E + eb_sum);  // batches added in order
            }
            ++need;
        }
        step = scalar(step * a.decay);
    }
    if (me == 0) {
        if (in_lds) {
            for (int k = tid; k < n; k += BT) a.pos[v0 + k] = P[k];
        }
        // every thread holds the same E (the batch sums come from the same wave sums); all of them
        // store it so that no per-lane branch sits next to the queue loop's back edge
        a.energies[g] = E;
        a.finish[g] = wall_clock64();
    }
    __syncthreads();
}

template <bool REFINE>
__global__ __launch_bounds__(BT) void k_batched(BatchedArgs a) {
    extern __shared__ double2 fb[];  // the batch's forces [B], then the graph's positions when they fit
    double2 *P = fb + a.B;
    __shared__ double2 red[BT];
    __shared__ double eb[BT / 64];
    __shared__ int slot, go;
    const int tid = threadIdx.x;
    if (tid == 0) a.wg_start[blockIdx.x] = wall_clock64();
    for (;;) {
        if (tid == 0) slot = atomicAdd(a.queue, 1);
        __syncthreads();
        // The slot is the same for every thread; readfirstlane makes that visible to the
        // compiler.  Left as a per-lane LDS value, the loop exit looks divergent and the
        // loop may be restructured so that lane 0 (which advances the queue) leaves the
        // per-graph loop while the other lanes of its wave repeat the same graph forever.
        const int q = __builtin_amdgcn_readfirstlane(slot);
        __syncthreads();
        if (q >= a.count) break;
        const int g = __builtin_amdgcn_readfirstlane(a.items[q].x), me = __builtin_amdgcn_readfirstlane(a.items[q].y);
        const int T = a.team ? __builtin_amdgcn_readfirstlane(a.team[g]) : 1;
        layout_graph<REFINE>(a, g, me, T, P, red, fb, eb, &go);
    }
}

// rend[i] = the end of row i's effective neighbours (effective_neighbors): the longest strictly
// increasing prefix of the row; an empty row has the graph's next entry, if any.  A workgroup per
// graph; eight entries of a row loaded at a time.  One entry after another on the host, this and the
// check of the rows (now on several threads) took 20 of the 32 ms that a call with 1,500 graphs and 10M
// entries spent beside its layouts.
__global__ __launch_bounds__(256) void k_row_ends(const int *__restrict__ voff, const int *__restrict__ rp,
                                                  const int *__restrict__ ci, int *__restrict__ rend) {
    const int v0 = voff[blockIdx.x], v1 = voff[blockIdx.x + 1];
    const int gend = rp[v1];
    for (int i = v0 + (int)threadIdx.x; i < v1; i += 256) {
        const int s = rp[i], e = rp[i + 1];
        int end = s < gend ? s + 1 : s;  // the first entry, or the next row's
        if (s < e) {
            int last = ci[s];
            for (bool more = true; more && end < e;) {
                int c[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) c[k] = ci[min(end + k, e - 1)];
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    more = more && end < e && c[k] > last;
                    last = c[k];
                    end += more ? 1 : 0;
                }
            }
        }
        rend[i] = end;
    }
}

// The fixed rule: every batch slot served in one round (the next power of two >= min(B, n)).
int ipw_rule(int n, int B) { return one_round(std::min(B, n)); }

// Tuned shapes per (size class, B, precision, law, positions in LDS), for the process.
struct TuneKey {
    int cls, B, refine, law, lds;
    bool operator<(const TuneKey &o) const {
        return std::tie(cls, B, refine, law, lds) < std::tie(o.cls, o.B, o.refine, o.law, o.lds);
    }
};
std::mutex tune_mu;
std::map<TuneKey, int> tuned;

// Team sizes for graphs of n[k] vertices on `places` workgroups that run at once, WG_RATE / per_cu
// pairs a us each: the graph that would end last gets twice the workgroups while that pays, until
// it is no longer far behind the launch's average.  A step costs STEP_US besides its pairs, a team's
// TEAM_US more (measured at the head of this file).
constexpr double WG_RATE = 13.0e3;  // a workgroup that has a CU to itself
constexpr double STEP_US = 4.0, TEAM_US = 4.5;
std::vector<int> team_sizes(const std::vector<int> &n, const std::vector<int> &ipw, int B, int cap, int places,
                            int per_cu) {
    const int count = (int)n.size();
    std::vector<int> T(count, 1);
    auto time = [&](int k, int t) {  // us per iteration
        const double nb = (n[k] + B - 1) / B;
        return nb * (STEP_US + (t > 1 ? TEAM_US : 0.0)) + (double)n[k] * n[k] * per_cu / (WG_RATE * t);
    };
    double all = 0.0;
    std::vector<std::pair<double, int>> heap(count);  // the latest first
    for (int k = 0; k < count; ++k) heap[k] = {time(k, 1), k}, all += heap[k].first;
    std::make_heap(heap.begin(), heap.end());
    int used = 0;  // places of teams
    while (!heap.empty()) {
        std::pop_heap(heap.begin(), heap.end());
        const double now = heap.back().first;
        const int k = heap.back().second, t = T[k], more = t == 1 ? 2 : t;
        heap.pop_back();
        if (now < 1.1 * all / places) break;
        const double then = time(k, 2 * t);
        if (n[k] > cap || 2 * t > MAXTEAM || 2 * t * (BT / ipw[k]) > chunks_of(n[k], B) || used + more > places ||
            then > 0.85 * now)
            break;  // what is left is no shorter than this one
        used += more;
        all += 2 * t * then - t * now;
        T[k] = 2 * t;
        heap.push_back({then, k});
        std::push_heap(heap.begin(), heap.end());
    }
    return T;
}

}  // namespace

int run_batched(int32_t count, const int32_t *voff, const int64_t *eoff, const int32_t *rowptr, const int32_t *colids,
                double *xy, const bl_params *p, double *energies, double *finish_ms, bl_stats *st) {
    if (p->batch > MAXB) return BL_E_ARG;
    const int N = voff[count];
    const size_t nnz = (size_t)eoff[count];
    // largest graphs first
    std::vector<int> order(count);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
        const long long nx = voff[x + 1] - voff[x], ny = voff[y + 1] - voff[y];
        return nx * nx > ny * ny;
    });

    int dev = 0, cus = 0, khz = 0, maxlds = 0;
    BL_HIP(hipGetDevice(&dev));
    BL_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    BL_HIP(hipDeviceGetAttribute(&maxlds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess || khz <= 0) khz = 100000;
    const int static_lds = (int)(sizeof(double2) * (BT + p->batch) + sizeof(double) * (BT / 64) + 64);
    int maxn = 0;
    for (int k = 0; k < count; ++k) maxn = std::max(maxn, voff[k + 1] - voff[k]);
    const int cap = std::max(0, std::min(maxn, (maxlds - static_lds) / (int)sizeof(double2)));
    const size_t dyn = sizeof(double2) * (size_t)(cap + p->batch);
    void (*const kernel)(BatchedArgs) = p->precision == BL_PREC_MIXED ? k_batched<true> : k_batched<false>;
    if (dyn > 0) BL_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn));
    int per_cu = 0;
    BL_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, BT, dyn));
    per_cu = std::max(1, per_cu);
    const int places = std::max(1, per_cu * cus);
    std::vector<int> sizes(count), ipw(count);
    for (int k = 0; k < count; ++k) {
        sizes[k] = voff[k + 1] - voff[k];
        ipw[k] = ipw_rule(sizes[k], p->batch);
    }
    const char *team_env = getenv("BL_BATCHED_TEAM");  // 1: no teams; 2..16: teams of that size where they fit (tests)
    std::vector<int> team = team_sizes(sizes, ipw, p->batch, cap, places, per_cu);
    if (team_env) {
        const int f = atoi(team_env);
        int used = 0;
        for (int k = 0; k < count; ++k) {
            team[k] = 1;
            if (f > 1 && f <= MAXTEAM && !(f & (f - 1)) && sizes[k] <= cap && f * (BT / ipw[k]) <= chunks_of(sizes[k], p->batch) &&
                used + f <= places)
                team[k] = f, used += f;
        }
    }
    // the queue: the teams' members, then the other graphs, each largest first
    std::vector<int2> items;
    std::vector<int> team_at(count, 0);
    int teams = 0;
    for (int q = 0; q < count; ++q)
        if (team[order[q]] > 1) {
            team_at[order[q]] = teams++;
            for (int m = 0; m < team[order[q]]; ++m) items.push_back(make_int2(order[q], m));
        }
    for (int q = 0; q < count; ++q)
        if (team[order[q]] == 1) items.push_back(make_int2(order[q], 0));
    const int grid = std::max(1, std::min((int)items.size(), places));

    hipStream_t s = nullptr;
    BL_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    struct Buffers {
        void *p = nullptr;
        hipStream_t s = nullptr;
        ~Buffers() {
            if (s) (void)hipStreamSynchronize(s);
            if (p) (void)hipFree(p);
            if (s) (void)hipStreamDestroy(s);
        }
    } buf;
    buf.s = s;
    const size_t b_order = 8 * items.size(), b_voff = 4 * (size_t)(count + 1), b_erp = 4 * (size_t)(N + 1),
                 b_eci = 4 * std::max<size_t>(1, nnz), b_pos = 16 * (size_t)N, b_en = 8 * (size_t)count,
                 b_fin = 8 * (size_t)count, b_wg = 8 * (size_t)grid, b_q = 64, b_ipw = 4 * (size_t)count,
                 b_arr = 4 * (size_t)std::max(1, 2 * teams),
                 b_parts = sizeof(double2) * 2 * MAXTEAM * p->batch * (size_t)teams;
    auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
    const size_t total = al(b_order) + al(b_voff) + 2 * al(b_erp) + al(b_eci) + al(b_pos) + al(b_en) + al(b_fin) +
                         al(b_wg) + al(b_q) + 3 * al(b_ipw) + al(b_order) + al(b_arr) + al(b_parts);
    BL_HIP(hipMalloc(&buf.p, total));
    char *c = static_cast<char *>(buf.p);
    int2 *d_items = reinterpret_cast<int2 *>(c); c += al(b_order);
    int *d_voff = reinterpret_cast<int *>(c); c += al(b_voff);
    int *d_rp = reinterpret_cast<int *>(c); c += al(b_erp);
    int *d_rend = reinterpret_cast<int *>(c); c += al(b_erp);
    int *d_ci = reinterpret_cast<int *>(c); c += al(b_eci);
    double2 *d_pos = reinterpret_cast<double2 *>(c); c += al(b_pos);
    double *d_en = reinterpret_cast<double *>(c); c += al(b_en);
    long long *d_fin = reinterpret_cast<long long *>(c); c += al(b_fin);
    long long *d_wg = reinterpret_cast<long long *>(c); c += al(b_wg);
    int *d_q = reinterpret_cast<int *>(c); c += al(b_q);
    int *d_ipw = reinterpret_cast<int *>(c); c += al(b_ipw);
    int *d_team = reinterpret_cast<int *>(c); c += al(b_ipw);
    int *d_team_at = reinterpret_cast<int *>(c); c += al(b_ipw);
    int *d_arr = reinterpret_cast<int *>(c); c += al(b_arr);  // the teams' counts, then their error flags
    double2 *d_parts = reinterpret_cast<double2 *>(c); c += al(b_parts);
    int2 *d_titems = reinterpret_cast<int2 *>(c);  // a size class's sample graphs (tuning)
    BL_HIP(hipMemcpyAsync(d_items, items.data(), b_order, hipMemcpyHostToDevice, s));
    BL_HIP(hipMemcpyAsync(d_team, team.data(), b_ipw, hipMemcpyHostToDevice, s));
    BL_HIP(hipMemcpyAsync(d_team_at, team_at.data(), b_ipw, hipMemcpyHostToDevice, s));
    BL_HIP(hipMemsetAsync(d_arr, 0, b_arr, s));
    BL_HIP(hipMemcpyAsync(d_voff, voff, b_voff, hipMemcpyHostToDevice, s));
    BL_HIP(hipMemcpyAsync(d_rp, rowptr, b_erp, hipMemcpyHostToDevice, s));
    if (nnz) BL_HIP(hipMemcpyAsync(d_ci, colids, 4 * nnz, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_row_ends, dim3(count), dim3(256), 0, s, d_voff, d_rp, d_ci, d_rend);
    BL_HIP(hipGetLastError());
    BL_HIP(hipMemcpyAsync(d_pos, xy, b_pos, hipMemcpyHostToDevice, s));
    BL_HIP(hipMemsetAsync(d_q, 0, b_q, s));

    BatchedArgs a;
    a.items = d_items;
    a.ipw_of = d_ipw;
    a.count = (int)items.size();
    a.team = d_team;
    a.team_at = d_team_at;
    a.parts = d_parts;
    a.arrived = d_arr;
    a.err = d_arr + teams;
    a.ticks = (long long)khz * 2000;  // 2 s
    if (const char *w = getenv("BL_BATCHED_WAIT_US")) a.ticks = (long long)khz * atoll(w) / 1000;  // tests
    a.voff = d_voff;
    a.rp = d_rp;
    a.rend = d_rend;
    a.ci = d_ci;
    a.pos = d_pos;
    a.B = p->batch;
    a.iters = p->iters;
    a.law = p->algo == BL_ALGO_FA ? LAW_FA : LAW_FR;
    a.lds_cap = cap;
    a.step0 = p->step0;
    a.decay = p->algo == BL_ALGO_FA ? 0.99 : 0.999;
    a.W = p->weight;
    a.energies = d_en;
    a.finish = d_fin;
    a.wg_start = d_wg;
    a.queue = d_q;
    hipEvent_t e0, e1;
    BL_HIP(hipEventCreate(&e0));
    BL_HIP(hipEventCreate(&e1));
    struct Events {
        hipEvent_t *a, *b;
        ~Events() {
            (void)hipEventDestroy(*a);
            (void)hipEventDestroy(*b);
        }
    } evs{&e0, &e1};

    // The shape of each graph: the fixed rule, or, for runs with enough work, the fastest of the
    // candidate shapes per size class (graphs of 2^c .. 2^(c+1) - 1 vertices), measured once per
    // process on up to TUNE_SAMPLE graphs of the class, one iteration each, on a copy of the
    // positions.  All shapes give the same bits.
    double work = 0.0;
    for (int k = 0; k < count; ++k) work += (double)(voff[k + 1] - voff[k]) * (voff[k + 1] - voff[k]);
    work *= std::max(1, p->iters);
    const char *tenv = getenv("BL_TUNE");
    const bool tune = !(tenv && !strcmp(tenv, "0")) && (work >= 2e9 || (tenv && !strcmp(tenv, "1")));
    if (tune) {
        constexpr int TUNE_SAMPLE = 24;
        std::map<int, std::vector<int>> members;  // class -> graph ids in queue order
        for (int q = 0; q < count; ++q) {
            const int k = order[q], nk = voff[k + 1] - voff[k];
            if (nk >= 2) members[31 - __builtin_clz((unsigned)nk)].push_back(k);
        }
        void *tpos = nullptr;
        struct Free {
            void **p;
            ~Free() {
                if (*p) (void)hipFree(*p);
            }
        } free_tpos{&tpos};
        for (auto &cm : members) {
            const std::vector<int> &ids = cm.second;
            int nmax = 0;
            for (int k : ids) nmax = std::max(nmax, voff[k + 1] - voff[k]);
            const TuneKey key{cm.first, p->batch, p->precision == BL_PREC_MIXED, a.law, nmax <= cap ? 1 : 0};
            int best = -1;
            {
                std::lock_guard<std::mutex> lock(tune_mu);
                auto it = tuned.find(key);
                if (it != tuned.end()) best = it->second;
            }
            const int top = ipw_rule(nmax, p->batch);
            if (best < 0 && top > 64) {
                if (!tpos) {
                    BL_HIP(hipMalloc(&tpos, b_pos));
                    BL_HIP(hipMemcpyAsync(tpos, d_pos, b_pos, hipMemcpyDeviceToDevice, s));
                }
                const int m = std::min((int)ids.size(), TUNE_SAMPLE);
                std::vector<int2> sample(m);
                for (int j = 0; j < m; ++j) sample[j] = make_int2(ids[j], 0);
                BL_HIP(hipMemcpyAsync(d_titems, sample.data(), 8 * (size_t)m, hipMemcpyHostToDevice, s));
                BatchedArgs t = a;
                t.items = d_titems;
                t.team = nullptr;
                t.count = m;
                t.iters = 1;
                t.pos = static_cast<double2 *>(tpos);
                float best_ms = 0.f;
                for (int cand = 64; cand <= top; cand <<= 1) {
                    std::vector<int> all(count, cand);
                    BL_HIP(hipMemcpyAsync(d_ipw, all.data(), b_ipw, hipMemcpyHostToDevice, s));
                    float ms = 0.f;
                    for (int rep = 0; rep < 2; ++rep) {  // the second launch is timed
                        BL_HIP(hipMemsetAsync(d_q, 0, b_q, s));
                        BL_HIP(hipEventRecord(e0, s));
                        hipLaunchKernelGGL(kernel, dim3(std::min(m, grid)), dim3(BT), dyn, s, t);
                        BL_HIP(hipGetLastError());
                        BL_HIP(hipEventRecord(e1, s));
                        BL_HIP(hipEventSynchronize(e1));
                        BL_HIP(hipEventElapsedTime(&ms, e0, e1));
                    }
                    if (best < 0 || ms < best_ms) best = cand, best_ms = ms;
                }
                std::lock_guard<std::mutex> lock(tune_mu);
                tuned[key] = best;
            }
            if (best > 0)
                for (int k : ids)  // a team keeps the rule's shape: a smaller one splits j past its chunks
                    if (team[k] == 1) ipw[k] = std::min(best, ipw_rule(voff[k + 1] - voff[k], p->batch));
        }
    }
    if (const char *force = getenv("BL_BATCHED_IPW")) {  // one shape for every graph (tests)
        const int f = atoi(force);
        if (f >= 64 && f <= BT && (f & (f - 1)) == 0)
            for (int k = 0; k < count; ++k)
                if (team[k] == 1) ipw[k] = std::min(f, ipw_rule(voff[k + 1] - voff[k], p->batch));
    }
    BL_HIP(hipMemcpyAsync(d_ipw, ipw.data(), b_ipw, hipMemcpyHostToDevice, s));
    BL_HIP(hipMemsetAsync(d_q, 0, b_q, s));
    BL_HIP(hipMemsetAsync(d_fin, 0, b_fin, s));
    BL_HIP(hipEventRecord(e0, s));
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(BT), dyn, s, a);
    BL_HIP(hipGetLastError());
    std::vector<double> en(count);
    std::vector<long long> fin(count), wg(grid);
    BL_HIP(hipMemcpyAsync(wg.data(), d_wg, b_wg, hipMemcpyDeviceToHost, s));
    if (teams) {
        BL_HIP(hipMemcpyAsync(fin.data(), d_fin, b_fin, hipMemcpyDeviceToHost, s));
        BL_HIP(hipStreamSynchronize(s));
        items.clear();  // the graphs of the teams that gave up, without teams
        for (int q = 0; q < count; ++q)
            if (!fin[order[q]]) items.push_back(make_int2(order[q], 0));
        if (!items.empty()) {
            BL_HIP(hipMemcpyAsync(d_items, items.data(), 8 * items.size(), hipMemcpyHostToDevice, s));
            BL_HIP(hipMemsetAsync(d_q, 0, b_q, s));
            a.count = (int)items.size();
            a.team = nullptr;
            hipLaunchKernelGGL(kernel, dim3(std::min((int)items.size(), grid)), dim3(BT), dyn, s, a);
            BL_HIP(hipGetLastError());
        }
    }
    BL_HIP(hipEventRecord(e1, s));
    int nonfinite = 0;  // the guard's counter in the queue block's spare words
    int rc = count_nonfinite(d_pos, N, d_q + 8, s, &nonfinite);
    if (rc) return rc;
    BL_HIP(hipMemcpyAsync(xy, d_pos, b_pos, hipMemcpyDeviceToHost, s));
    BL_HIP(hipMemcpyAsync(en.data(), d_en, b_en, hipMemcpyDeviceToHost, s));
    BL_HIP(hipMemcpyAsync(fin.data(), d_fin, b_fin, hipMemcpyDeviceToHost, s));
    BL_HIP(hipStreamSynchronize(s));
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    if (energies) std::copy(en.begin(), en.end(), energies);
    if (finish_ms) {
        const long long t0 = *std::min_element(wg.begin(), wg.end());
        for (int k = 0; k < count; ++k) finish_ms[k] = (double)(fin[k] - t0) / (double)khz;
    }
    if (st) {
        memset(st, 0, sizeof(*st));
        st->energy = std::accumulate(en.begin(), en.end(), 0.0);
        st->iters_done = p->iters;
        st->seconds = ms / 1e3;
        double sstep = p->step0;
        for (int it = 0; it < p->iters; ++it) sstep *= a.decay;
        st->step_final = sstep;
        st->kernel_ms[0] = ms;
        st->kernel_launches[0] = 1;
        st->nonfinite = nonfinite;
    }
    return BL_OK;
}

}  // namespace bl
