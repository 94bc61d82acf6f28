// The batch walk of the Barnes-Hut family (algorithms.cpp:1050-1066) by dependence levels.
//
// A vertex's new position is a function of its iteration-start position, its repulsion, the new
// positions of its neighbours in earlier batches ("early") and the iteration-start positions of
// the others ("late").  So the sequential batches are a dependence graph of vertices, not of
// batches: level(i) = 1 + the largest level of an early neighbour (0 without one), and the
// vertices of one level move at once whatever their batches.  There are never more levels than
// batches, and on graphs with unordered ids there are about as many as the longest chain of
// neighbours in increasing batch order: 18 on a triangulation of 1.66M points at -batch 256 (6,497
// batches), 24 on the 250k random geometric graph (976), 199 on the R-MAT graph of scale 20
// at -batch 1024 (534).  The result is the sequential walk's: the late terms are summed first,
// for all vertices (k_level_late), before any vertex moves.
//
//   f_i = (sum over early, in list order) - rep'_i,    rep'_i = rep_i - sum over late
//
// Consecutive levels are one launch (k_level_flow).  Nothing but the new positions orders them: before the
// walk every vertex's entry of `moved` is marked as not there, a move stores its vertex's, and whoever
// needs it reads it until it has come.  So a level costs one store and one load through memory, about
// 2.4 us, where a launch of its own cost 5 (two dependent loads past caches that a launch leaves empty, the
// dispatch, the write-back), and the next levels' rows are loaded while they wait.  Workgroups take their
// level and place in it by a ticket in level order, from one counter: what a workgroup waits for was given to
// one that started before it, so some workgroup can always go on, whatever else runs on the device (with a
// counter for each XCD two launches side by side can each fill the XCD whose next ticket the other waits
// for).  A ticket takes 13 ns, one after another, so a workgroup takes as many rows as its lanes have
// places for.  A wait ends at a deadline, and the run with an error.
//   - rows of up to 4 entries take 4 lanes each, rows of up to 8 take 8, of up to 16 16, at an address that
//     the lane's number gives: a lane forms the factors of one entry, and the lanes' products are added one
//     after another by DPP moves (with rows of 9 to 16 entries one a wave the random geometric graph's walk
//     took 5,183 tickets and 75 us, now 64; R-MAT 486 -> 455);
//   - rows of up to LV_WAVE entries one a wave, longer ones (hubs) one a workgroup.
// What bounds the walk: on R-MAT the hand-off of 188 levels; on the triangulation random 16-byte reads and
// writes (1.66M moves in 198 us).  k_level_flow against a launch a level: R-MAT scale 20 at -batch 1024
// 989 -> 455 us, 250k random geometric graph 111 -> 64, triangulation 215 -> 198.
// Runs of levels of at most LV_RUN vertices without rows beyond 8 entries are one launch of one
// workgroup, which takes the levels one after another with a barrier between them (1.2 to 3 us each) and
// loads a level's vertices and entries two levels ahead.
//
// Walk per iteration, with the late sums, before and after: triangulation of 1.66M points at -batch
// 256 2.65 -> 0.28 ms (lagged walk), 250k random geometric graph 0.54 -> 0.08 ms (lagged walk),
// R-MAT scale 20 at -batch 1024 2.07 -> 0.56 ms (wide walk), a 1000 x 1000 grid in row order at
// -batch 64 7.84 -> 2.17 ms (lagged walk) and at -batch 1024 5.20 -> 0.08 ms (entry-split walk).
//
// Graphs for which the lagged walk (walk_lag.hip) is chosen keep its sums bit for bit: the
// early neighbours at least D groups back ("settled") are summed first, the repulsion is
// subtracted, then the others ("recent", marked in the entry) are added; |d| and the unit vector by rsqrt2
// (late terms by the IEEE square root).  Those for which the wide walk (walk_wide.hip) is chosen have all by
// rsqrt2, as it has.  All others have IEEE roots and divisions, as the row, entry-split and split walks.
#include <math.h>
#include <stdlib.h>

#include <algorithm>
#include <new>
#include <vector>

#include "bh_common.h"
#include "pair_math.h"

namespace bl {
namespace {

constexpr int LV_NARROW = 4, LV_WIDE = 8, LV_BROAD = 16;  // lanes of a short row
constexpr int LV_WAVE = 512;      // longest row of one wave: 8 entries a lane (1, in list order)
constexpr int LV_T = 512;         // threads of a level's workgroups: 8 slices or rows, or one hub
constexpr int LV_WAVES = LV_T / 64;
constexpr int LV_RUN = 2048;      // largest level of a run: 2 slices per wave of 1024 threads
constexpr int LV_RUNS = 8;        // shortest run: a level in it takes 2-3 us, after about 15 us to start
constexpr int LV_TICKET_INTS = 32;  // between the ticket counters of the launches
// Blocks of a level from which a ticket stands for two: the triangulation's walk takes 232 us with one, 198 with
// two, 214 with up to eight (from 256 blocks a ticket more), whose rows then wait for each other.
constexpr int LV_PAIR = 512;
constexpr int LV_MAXLEVELS = 1 << 16;
constexpr int LV_LATE = 32;       // longest row of a slice of the late lists
constexpr int LV_ROW = 64;        // longest row whose sums are kept in list order (the lagged walk's)
constexpr int LV_WINDOW = 4096;   // where rows are longer, these lists are sorted by length within such windows
constexpr unsigned LV_PAD = 0x7fffffffu, LV_RECENT = 0x80000000u;
constexpr int64_t LV_SHORT = (int64_t)1 << 62;  // host: marks a short row's place

// A level in k_level_flow, its `blocks` of 8 waves' work from the last, `per` of them to a workgroup from
// the launch's number `first` on: nn waves of rows of 4 lanes (16 a wave), then nw of rows of 8 (8 a
// wave) and nb of rows of 16, from vertex slot v0 and entry block e0 (64 entries each), then nr rows from
// row r0, one a wave, then hubs, one a workgroup.
struct LevelShape {
    int v0, nn, nw, nb, r0, nr;
    unsigned e0;
    int first, blocks, per;
};

struct LevelArgs {
    const int2 *head;      // late slices: first entry, columns
    const int *vid;        // vertices of the slices and short rows (-1: none)
    const unsigned *ids;   // their entries: column id, LV_RECENT, or LV_PAD; a slice's as [column][64], a
                           // short row's consecutive
    const float *w;
    const int4 *row;       // longer rows: vertex, first entry, past the last
    const unsigned *rids;
    const float *rw;
    const int *lstart;     // the run kernel: first slice of each level in its run
    double W, step;
    double2 *pos, *rep;
    double2 *moved;        // new positions, LV_NONE until they are there
    double *eterm;
    const int *status;
    const int *blk;        // k_level_flow: each workgroup's level
    const LevelShape *shape;
    int *ticket, *err;
    long long ticks;       // the longest wait for a position
};

// "Not moved yet": all ones, a NaN that no stored position is.
constexpr unsigned long long LV_NONE = ~0ull;
__device__ __forceinline__ bool is_none(double x) { return (unsigned long long)__double_as_longlong(x) == LV_NONE; }

// Positions between workgroups: 16 bytes an access, past the XCD's L2 on both sides.  One lane's access to an
// aligned address is one request, so a coordinate is seen whole, and each is looked at by itself.  As two
// 8-byte accesses (load_through, store_through) the walk took 657 us on R-MAT against 462, for twice
// the requests of the waves that wait.
typedef double f64x2 __attribute__((ext_vector_type(2)));
template <int N>
__device__ __forceinline__ void load_moved(const LevelArgs &a, const int *j, double2 *p) {
    f64x2 v[N];
    if constexpr (N == 1) {
        __asm__ volatile("global_load_dwordx4 %0, %1, off sc1\n\ts_waitcnt vmcnt(0)"
                         : "=&v"(v[0])
                         : "v"(a.moved + j[0])
                         : "memory");
    } else {
        static_assert(N == 8, "one or eight positions");
        __asm__ volatile(
            "global_load_dwordx4 %0, %8, off sc1\n\tglobal_load_dwordx4 %1, %9, off sc1\n\t"
            "global_load_dwordx4 %2, %10, off sc1\n\tglobal_load_dwordx4 %3, %11, off sc1\n\t"
            "global_load_dwordx4 %4, %12, off sc1\n\tglobal_load_dwordx4 %5, %13, off sc1\n\t"
            "global_load_dwordx4 %6, %14, off sc1\n\tglobal_load_dwordx4 %7, %15, off sc1\n\ts_waitcnt vmcnt(0)"
            : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
            : "v"(a.moved + j[0]), "v"(a.moved + j[1]), "v"(a.moved + j[2]), "v"(a.moved + j[3]), "v"(a.moved + j[4]),
              "v"(a.moved + j[5]), "v"(a.moved + j[6]), "v"(a.moved + j[7])
            : "memory");
    }
#pragma unroll
    for (int g = 0; g < N; ++g) p[g] = make_double2(v[g].x, v[g].y);
}
__device__ __forceinline__ void store_moved(double2 *p, double2 q) {
    f64x2 v = {q.x, q.y};
    // two wait states before the registers of a 16-byte store may be written again
    __asm__ volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" : : "v"(p), "v"(v) : "memory");
}

// x_i += (F/|F|) * STEP (:1062-1066).  IEEE: root and divisions as the row, entry-split and split walks form
// them; else the unit vector F * rsqrt2(|F|^2), the lagged and the wide walk's operations.
// FLOW: published for the workgroups of the same launch, else for later launches if there are any that
// read it (a.moved).
template <bool FLOW, bool IEEE>
__device__ __forceinline__ void move_vertex(const LevelArgs &a, int i, double2 v, double2 f) {
    const double m2 = f.x * f.x + f.y * f.y;
    double2 q;
    if constexpr (IEEE) {
        q = moved(v, f.x, f.y, a.step);
    } else {
        const double r = rsqrt2(m2) * a.step;
        q = make_double2(fma(f.x, r, v.x), fma(f.y, r, v.y));
    }
    const double2 m = make_double2(is_none(q.x) ? NAN : q.x, is_none(q.y) ? NAN : q.y);
    if constexpr (FLOW) store_moved(a.moved + i, m);
    else if (a.moved) a.moved[i] = m;
    a.pos[i] = q;
    a.eterm[i] = m2;
}

// The new positions of the early neighbours j[g] (of which only those with need[g] must be there), each
// read until it has come.  False: given up, at the deadline or because another wave did.
template <int N>
__device__ __forceinline__ bool moved_pos(const LevelArgs &a, const int *j, const bool *need, double2 *p) {
    load_moved<N>(a, j, p);
    long long t0 = 0;
    for (int k = 0;; ++k) {
        bool wait = false;
#pragma unroll
        for (int g = 0; g < N; ++g) wait = wait || (need[g] && (is_none(p[g].x) || is_none(p[g].y)));
        if (!__any(wait)) return true;
        if (k == 0) t0 = wall_clock64();
        if ((k & 15) == 15 || a.ticks < 0) {
            const bool late = wall_clock64() - t0 > a.ticks;
            if (late) store_through(a.err, 1);
            if (late || load_through(a.err)) return false;
        }
        __builtin_amdgcn_s_sleep(1);
        if (wait) load_moved<N>(a, j, p);
    }
}

// A neighbour's difference and the factor of its attraction W|d| d, |d| by the IEEE square root or rsqrt2.
template <bool IEEE>
__device__ __forceinline__ void factors(double2 pj, double2 v, double Wk, double &dx, double &dy, double &sc) {
    if constexpr (IEEE) {
        dx = pj.x - v.x;
        dy = pj.y - v.y;
        sc = Wk * sqrt(dx * dx + dy * dy);
    } else {
        attr_factors(pj, v, Wk, dx, dy, sc);
    }
}

// The sums so far and one more term, kept if `on`.
template <bool IEEE>
__device__ __forceinline__ void add_if(bool on, double2 pj, double2 v, double Wk, double2 &f) {
    double dx, dy, sc;
    factors<IEEE>(pj, v, Wk, dx, dy, sc);
    const double x = fma(dx, sc, f.x), y = fma(dy, sc, f.y);
    f.x = on ? x : f.x;
    f.y = on ? y : f.y;
}

// Early sum of one vertex: settled entries, then - r at the first recent one (or at the end).
template <bool IEEE>
struct EarlySum {
    double2 f{0.0, 0.0};
    bool less = false;
    __device__ __forceinline__ void subtract(bool on, double2 r) {
        f.x = on ? f.x - r.x : f.x;
        f.y = on ? f.y - r.y : f.y;
        less = less || on;
    }
    __device__ __forceinline__ void add(unsigned c, double2 pj, double2 v, double2 r, double Wk) {
        subtract(c >= LV_RECENT && !less, r);
        add_if<IEEE>(c != LV_PAD, pj, v, Wk, f);
    }
    __device__ __forceinline__ double2 total(double2 r) {
        subtract(!less, r);
        return f;
    }
};

// N columns of a slice from entry e (the lane's in the first column), of which the first `have`
// exist (the last again past them), and the positions they name (padding names the own vertex).
template <bool HAS_W, int N>
__device__ __forceinline__ void slice_ids(const LevelArgs &a, size_t e, int have, unsigned *c, float *w) {
#pragma unroll
    for (int g = 0; g < N; ++g) {
        const size_t k = e + 64 * (size_t)min(g, have - 1);
        c[g] = g < have ? a.ids[k] : LV_PAD;
        w[g] = HAS_W ? a.w[k] : 0.0f;
    }
}
template <int N>
__device__ __forceinline__ void slice_pos(const LevelArgs &a, const unsigned *c, int own, double2 *p) {
#pragma unroll
    for (int g = 0; g < N; ++g) p[g] = a.pos[c[g] == LV_PAD ? own : (int)(c[g] & LV_PAD)];
}

// v of the lane before (row_shr:1; lane 0 of 16 gets 0, and the first lane of a short row takes none).
__device__ __forceinline__ double lane_before(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x111, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x111, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}

// A wave of short rows (false: given up), N lanes each: entry block `block`, the rows' vertices from slot vs.  Lane k
// of a row forms entry k's factors and adds its product to the sum of the lanes before it, in the
// k-th of N steps; the repulsion is subtracted before the first recent entry, else at the end.
template <bool HAS_W, int N, bool IEEE>
__device__ __forceinline__ bool short_rows(const LevelArgs &a, int vs, size_t block) {
    const int lane = threadIdx.x & 63, k = lane & (N - 1);
    const int id = a.vid[vs + lane / N], i = max(id, 0);
    const size_t e = block * 64 + lane;
    const unsigned c = a.ids[e];
    const double Wk = HAS_W ? a.W * (double)a.w[e] : a.W;
    const bool real = c != LV_PAD;
    const double2 v = a.pos[i], r = a.rep[i];
    const int j = real ? (int)(c & LV_PAD) : i;
    double2 pj;
    if (!moved_pos<1>(a, &j, &real, &pj)) return false;
    double dx, dy, sc;
    factors<IEEE>(pj, v, Wk, dx, dy, sc);
    const unsigned rec = (unsigned)(__ballot(c >= LV_RECENT) >> (lane - k)) & ((1u << N) - 1);
    const bool first = rec != 0 && (int)__builtin_ctz(rec) == k;
    const double rx = first ? r.x : 0.0, ry = first ? r.y : 0.0;
    double2 f = make_double2(0.0, 0.0);
#pragma unroll
    for (int g = 0; g < N; ++g) {
        double px = g > 0 ? lane_before(f.x) : 0.0, py = g > 0 ? lane_before(f.y) : 0.0;
        px -= rx;
        py -= ry;
        const double sx = fma(dx, sc, px), sy = fma(dy, sc, py);
        if (k == g) f = make_double2(real ? sx : px, real ? sy : py);
    }
    if (rec == 0) f = make_double2(f.x - r.x, f.y - r.y);
    if (k == N - 1 && id >= 0) move_vertex<true, IEEE>(a, i, v, f);
    return true;
}

// This thread's share of a row's sum: entries t, t + T, ..., eight loads in flight.
// LATE: their iteration-start positions, else the new ones (bad: given up).
template <bool HAS_W, bool LATE, bool IEEE, int T>
__device__ __forceinline__ double2 row_share(const LevelArgs &a, int4 row, int t, double2 v, int &bad) {
    constexpr int N = 8;
    double2 f = make_double2(0.0, 0.0);
    for (int e = row.y + t; e < row.z; e += N * T) {
        int c[N];
        bool on[N];
        double2 p[N];
        float w[N];
#pragma unroll
        for (int g = 0; g < N; ++g) {
            const int k = min(e + g * T, row.z - 1);
            on[g] = e + g * T < row.z;
            c[g] = (int)(a.rids[k] & LV_PAD);
            w[g] = HAS_W ? a.rw[k] : 0.0f;
        }
        if constexpr (LATE) {
#pragma unroll
            for (int g = 0; g < N; ++g) p[g] = a.pos[c[g]];
        } else if (!moved_pos<N>(a, c, on, p)) {
            bad = 1;
            break;
        }
#pragma unroll
        for (int g = 0; g < N; ++g)
            add_if<IEEE>(on[g], p[g], v, HAS_W ? a.W * (double)w[g] : a.W, f);
    }
    return f;
}

__device__ __forceinline__ double lane_of(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}

// The total force of a row of at most 64 entries with its sums in list order, in every lane: lane
// k forms the factors of entry k, then the products are added one after another.
template <bool HAS_W>
__device__ __forceinline__ double2 row_in_order(const LevelArgs &a, int4 row, int lane, double2 v, double2 r, int &bad) {
    const int cnt = row.z - row.y, k = row.y + min(lane, cnt - 1);
    const unsigned c = a.rids[k];
    const double Wk = HAS_W ? a.W * (double)a.rw[k] : a.W;
    const int j = (int)(c & LV_PAD);
    const bool real = true;
    double2 pj;
    if (!moved_pos<1>(a, &j, &real, &pj)) bad = 1;
    double dx, dy, sc;
    attr_factors(pj, v, Wk, dx, dy, sc);
    const uint64_t rec = __ballot(c >= LV_RECENT && lane < cnt);
    const int from = rec ? (int)__builtin_ctzll(rec) : cnt;  // the first recent entry
    double2 f = make_double2(0.0, 0.0);
    for (int e = 0; e < cnt; ++e) {
        if (e == from) f = make_double2(f.x - r.x, f.y - r.y);
        const double s = lane_of(sc, e);
        f.x = fma(lane_of(dx, e), s, f.x);
        f.y = fma(lane_of(dy, e), s, f.y);
    }
    return from == cnt ? make_double2(f.x - r.x, f.y - r.y) : f;
}

// A row's wave or workgroup has its sum f in `one` thread: the late sum, or the move.
template <bool LATE, bool IEEE>
__device__ __forceinline__ void finish_row(const LevelArgs &a, bool one, int i, double2 v, double2 r, double2 f, int bad) {
    if (!one || bad) return;
    if constexpr (LATE)
        a.rep[i] = make_double2(r.x - f.x, r.y - f.y);
    else
        move_vertex<true, IEEE>(a, i, v, make_double2(f.x - r.x, f.y - r.y));
}

// Rows by block b past the slices' blocks: nr rows from row r0 one a wave, then hubs (a
// fixed order of the sums: per lane, over the wave by DPP, over the waves in turn).  False: given up (a
// hub in all waves).
template <bool HAS_W, bool LATE, bool SEQ, bool IEEE>
__device__ __forceinline__ bool long_rows(const LevelArgs &a, int b, int r0, int nr, int bad) {
    __shared__ double2 red[LV_WAVES];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int rb = (nr + LV_WAVES - 1) / LV_WAVES;
    if (b < rb) {
        const int k = b * LV_WAVES + wave;
        if (k >= nr) return true;
        const int4 row = a.row[r0 + k];  // wave-uniform
        const double2 v = a.pos[row.x], r = a.rep[row.x];
        if constexpr (SEQ) {
            const double2 f = row_in_order<HAS_W>(a, row, lane, v, r, bad);
            if (lane == 0 && !bad) move_vertex<true, IEEE>(a, row.x, v, f);
            return !bad;
        }
        double2 f = row_share<HAS_W, LATE, IEEE, 64>(a, row, lane, v, bad);
        bad = __any(bad);
        f.x = wave_sum(f.x);
        f.y = wave_sum(f.y);
        finish_row<LATE, IEEE>(a, lane == 0, row.x, v, r, f, bad);
        return !bad;
    }
    const int4 row = a.row[r0 + nr + b - rb];
    const double2 v = a.pos[row.x], r = a.rep[row.x];
    double2 f = row_share<HAS_W, LATE, IEEE, LV_T>(a, row, (int)threadIdx.x, v, bad);
    f.x = wave_sum(f.x);
    f.y = wave_sum(f.y);
    __syncthreads();  // the hub before has been added up
    if (lane == 0) red[wave] = f;
    bad = __syncthreads_or(bad);
    f = red[0];
#pragma unroll
    for (int k = 1; k < LV_WAVES; ++k) f = add2(f, red[k]);
    finish_row<LATE, IEEE>(a, threadIdx.x == 0, row.x, v, r, f, bad);
    return !bad;
}

// Consecutive levels (SEQ: every row's sum in list order), the longest rows of each first.
template <bool HAS_W, bool SEQ, bool IEEE>
__global__ __launch_bounds__(LV_T) void k_level_flow(LevelArgs a) {
    __shared__ int tk;
    if (threadIdx.x == 0)  // nullptr: a single level, nothing to wait for
        tk = a.ticket ? __hip_atomic_fetch_add(a.ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : (int)blockIdx.x;
    const int bad = *a.status;
    __syncthreads();
    if (bad) return;
    const int t = __builtin_amdgcn_readfirstlane(tk);
    const LevelShape q = a.shape[a.blk[t]];
    const int nsb = (q.nn + q.nw + q.nb + LV_WAVES - 1) / LV_WAVES;
    const int end = q.blocks - (t - q.first) * q.per;
    // hubs first, whose barriers every wave reaches: one that gives up at a row or slice meets no more of them
    for (int b = end - 1; b >= max(0, end - q.per); --b) {
        bool ok = true;
        if (b < nsb) {
            const int k = __builtin_amdgcn_readfirstlane(b * LV_WAVES + ((int)threadIdx.x >> 6));
            constexpr int RN = 64 / LV_NARROW, RW = 64 / LV_WIDE, RB = 64 / LV_BROAD;  // rows a wave
            const int wide = q.v0 + RN * q.nn, broad = wide + RW * q.nw;
            if (k < q.nn)
                ok = short_rows<HAS_W, LV_NARROW, IEEE>(a, q.v0 + RN * k, (size_t)q.e0 + k);
            else if (k < q.nn + q.nw)
                ok = short_rows<HAS_W, LV_WIDE, IEEE>(a, wide + RW * (k - q.nn), (size_t)q.e0 + k);
            else if (k < q.nn + q.nw + q.nb)
                ok = short_rows<HAS_W, LV_BROAD, IEEE>(a, broad + RB * (k - q.nn - q.nw), (size_t)q.e0 + k);
        } else {
            ok = long_rows<HAS_W, false, SEQ, IEEE>(a, b - nsb, q.r0, q.nr, 0);
        }
        if (!ok) return;
    }
}

// What k_level_late leaves for an iteration's k_level_flow: no vertex has moved, no workgroup has a ticket.
struct LevelClear {
    int late;     // k_level_late's workgroups for the late sums; the others clear
    int n, nt;    // vertices and ints of tickets (0, 0 where no launch reads them)
    int *ticket;
    int first;    // the run's first iteration
};
__device__ __forceinline__ void clear_moved(const LevelArgs &a, const LevelClear &q) {
    const double none = __longlong_as_double((long long)LV_NONE);
    const int i = ((int)blockIdx.x - q.late) * LV_T + (int)threadIdx.x;
    if (i < q.n) a.moved[i] = make_double2(none, none);
    for (int k = i; k < q.nt; k += ((int)gridDim.x - q.late) * LV_T) q.ticket[k] = 0;
    if (q.first && i == 0) *a.err = 0;
}

// The late sums of all vertices, folded into the repulsion: ns slices, then the rows.
template <bool HAS_W, bool IEEE>
__global__ __launch_bounds__(LV_T) void k_level_late(LevelArgs a, int ns, int nr, LevelClear q) {
    if ((int)blockIdx.x >= q.late) {
        clear_moved(a, q);
        return;
    }
    const int bad = *a.status;
    const int nsb = (ns + LV_WAVES - 1) / LV_WAVES;
    if ((int)blockIdx.x < nsb) {
        constexpr int N = 4;
        const int lane = threadIdx.x & 63;
        const int s = __builtin_amdgcn_readfirstlane((int)blockIdx.x * LV_WAVES + ((int)threadIdx.x >> 6));
        if (s >= ns) return;
        const int2 h = a.head[s];
        const int id = a.vid[s * 64 + lane], i = max(id, 0);
        const double2 v = a.pos[i], r = a.rep[i];
        double2 f = make_double2(0.0, 0.0);
        for (int k0 = 0; k0 < h.y; k0 += N) {
            unsigned c[N];
            float w[N];
            double2 p[N];
            slice_ids<HAS_W, N>(a, (size_t)h.x + 64 * (size_t)k0 + lane, h.y - k0, c, w);
            slice_pos<N>(a, c, i, p);
#pragma unroll
            for (int g = 0; g < N; ++g)
                add_if<IEEE>(c[g] != LV_PAD, p[g], v, HAS_W ? a.W * (double)w[g] : a.W, f);
        }
        if (id >= 0 && !bad) a.rep[i] = make_double2(r.x - f.x, r.y - f.y);
        return;
    }
    long_rows<HAS_W, true, false, IEEE>(a, (int)blockIdx.x - nsb, 0, nr, bad);
}

// Levels [l0, l1) of at most LV_RUN vertices in slices of 8 columns (the run's first vertex slot is
// v0, its entry block e0), by one workgroup: wave w takes slices w and w + 16 of a level.  What does
// not change during the walk is loaded ahead, the vertices and entries two levels and the vertex's
// own position (only its own level moves it) and repulsion one; after the barrier a level is one
// round trip for its neighbours' positions, the sums and the stores.  The workgroup's waves share
// one L1, so a barrier after the stores is all the order they need.
template <bool HAS_W, bool IEEE>
__global__ __launch_bounds__(1024) void k_level_run(LevelArgs a, int l0, int l1, int v0, unsigned e0) {
    constexpr int PER = LV_RUN / 1024, G = LV_WIDE;
    if (__builtin_amdgcn_readfirstlane(*a.status)) return;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    struct Slice {
        int id = -1;
        unsigned c[G];
        float w[G];
    } cur[PER], nxt[PER];
    double2 v[PER], r[PER];
    auto entries = [&](int l, Slice *x) {
        const int b = l < l1 ? a.lstart[l] : 0, e = l < l1 ? a.lstart[l + 1] : 0;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int s = b + wv + 16 * j;
            x[j].id = -1;
            if (s < e) {
                x[j].id = a.vid[v0 + s * 64 + lane];
                slice_ids<HAS_W, G>(a, ((size_t)e0 + (size_t)G * s) * 64 + lane, G, x[j].c, x[j].w);
            } else {
#pragma unroll
                for (int g = 0; g < G; ++g) x[j].c[g] = LV_PAD, x[j].w[g] = 0.0f;
            }
        }
    };
    auto own = [&](const Slice *x) {
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int i = max(x[j].id, 0);
            v[j] = a.pos[i];
            r[j] = a.rep[i];
        }
    };
    entries(l0, cur);
    own(cur);
    entries(l0 + 1, nxt);
    for (int l = l0; l < l1; ++l) {
        double2 f[PER], vo[PER];
        int ido[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            ido[j] = cur[j].id;
            vo[j] = v[j];
            f[j] = make_double2(0.0, 0.0);
            if (__builtin_amdgcn_readfirstlane(__ballot(ido[j] >= 0) != 0)) {
                double2 p[G];
                slice_pos<G>(a, cur[j].c, max(ido[j], 0), p);
                EarlySum<IEEE> sum;
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    if (!__ballot(cur[j].c[g] != LV_PAD)) break;  // rows fill the columns in order
                    sum.add(cur[j].c[g], p[g], v[j], r[j], HAS_W ? a.W * (double)cur[j].w[g] : a.W);
                }
                f[j] = sum.total(r[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < PER; ++j) cur[j] = nxt[j];
        own(cur);
        entries(l + 2, nxt);
#pragma unroll
        for (int j = 0; j < PER; ++j)
            if (ido[j] >= 0) move_vertex<false, IEEE>(a, ido[j], vo[j], f[j]);
        __syncthreads();
    }
}

template <class T>
bool put(DevBuf &d, const std::vector<T> &h) {
    if (d.ensure(sizeof(T) * std::max<size_t>(h.size(), 64))) return false;
    return h.empty() || hipMemcpy(d.p, h.data(), sizeof(T) * h.size(), hipMemcpyHostToDevice) == hipSuccess;
}

// The slices' heads and vertices and the longer rows, as on the device, and room for their entries
// (k_level_fill).
struct Lists {
    std::vector<int2> head;
    std::vector<int32_t> vid;
    std::vector<int4> row;
    bool upload(LevelLists &d, bool has_w, int64_t nid, int64_t nrid, hipStream_t s) const {
        const size_t a = 4 * (size_t)std::max<int64_t>(nid, 64), b = 4 * (size_t)std::max<int64_t>(nrid, 64);
        if (!put(d.head, head) || !put(d.vid, vid) || !put(d.row, row) || d.ids.ensure(a) || d.rids.ensure(b)) return false;
        if (has_w && (d.w.ensure(a) || d.rw.ensure(b) || hipMemsetAsync(d.w.p, 0, a, s) != hipSuccess)) return false;
        return hipMemsetD32Async((hipDeviceptr_t)d.ids.p, (int)LV_PAD, a / 4, s) == hipSuccess;
    }
};

// Where a vertex's entries go: a slice's column (stride 64), a short row or a longer row (consecutive).
struct FillList {
    const int64_t *slot;
    unsigned *ids, *rids;
    float *w, *rw;
    __device__ __forceinline__ void put(int64_t sl, int k, unsigned id, const float *gw, int e) const {
        const int64_t r = ~sl;
        const bool row = sl < 0 && !(r & LV_SHORT);
        const int64_t at = sl >= 0 ? sl + 64 * (int64_t)k : (r & ~LV_SHORT) + k;
        (row ? rids : ids)[at] = id;
        if (gw) (row ? rw : w)[at] = gw[e];
    }
};

// The entries of the lists from the CSR: a vertex's late entries (same or a later batch), its settled early
// ones, then the recent ones (D > 0: groups later than its own less D), each in CSR order.  A lane per
// vertex; rows of more than 32 entries by the whole wave, one after another.  On the host, with the
// lists' pages touched for the first time, this took 28 of the 66 ms of a first pass over the R-MAT graph of
// scale 20 and 17 of 92 on the 1.66M-vertex triangulation.
__global__ __launch_bounds__(256) void k_level_fill(int n, int B, int D, const int *__restrict__ rp,
                                                    const int *__restrict__ ci, const float *__restrict__ gw,
                                                    const int *__restrict__ go, FillList early, FillList late) {
    const int i = (int)blockIdx.x * 256 + threadIdx.x, lane = threadIdx.x & 63;
    const bool in = i < n;
    const int s = in ? rp[i] : 0, e = in ? rp[i + 1] : 0;
    const int b0 = i / B * B, lim = in && D > 0 ? go[i] - D : 0;
    const int64_t es = in ? early.slot[i] : 0, ls = in ? late.slot[i] : 0;
    const bool wide = e - s > 32;
    if (!wide) {
        int ke = 0, kl = 0;
        bool recent = false;
        for (int x = s; x < e; ++x) {
            const int j = ci[x];
            if (j >= b0) late.put(ls, kl++, (unsigned)j, gw, x);
            else if (D > 0 && go[j] > lim) recent = true;
            else early.put(es, ke++, (unsigned)j, gw, x);
        }
        for (int x = s; recent && x < e; ++x) {
            const int j = ci[x];
            if (j < b0 && go[j] > lim) early.put(es, ke++, (unsigned)j | LV_RECENT, gw, x);
        }
    }
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    for (uint64_t todo = __ballot(wide); todo; todo &= todo - 1) {
        const int from = (int)__builtin_ctzll(todo);
        const int rs = __shfl(s, from, 64), re = __shfl(e, from, 64), rb = __shfl(b0, from, 64);
        const int rl = __shfl(lim, from, 64);
        const int64_t te = __shfl((long long)es, from, 64), tl = __shfl((long long)ls, from, 64);
        int ke = 0, kl = 0;
        uint64_t any = 0;
        for (int pass = 0; pass < 2; ++pass) {  // settled and late entries, then the recent ones
            if (pass && !any) break;
            for (int x0 = rs; x0 < re; x0 += 64) {
                const int x = x0 + lane;
                const int j = x < re ? ci[x] : 0;
                const bool is_late = x < re && j >= rb;
                const bool recent = x < re && !is_late && D > 0 && go[j] > rl;
                const bool settled = x < re && !is_late && !recent;
                const uint64_t me = __ballot(pass ? recent : settled), ml = __ballot(is_late);
                if (pass ? recent : settled)
                    early.put(te, ke + __popcll(me & lt), (unsigned)j | (pass ? LV_RECENT : 0u), gw, x);
                if (!pass && is_late) late.put(tl, kl + __popcll(ml & lt), (unsigned)j, gw, x);
                ke += __popcll(me);
                kl += __popcll(ml);
                any |= __ballot(recent);
            }
        }
    }
}

}  // namespace

namespace {
int level_blocks(int slices, int rows, int hubs) {
    return (slices + LV_WAVES - 1) / LV_WAVES + (rows + LV_WAVES - 1) / LV_WAVES + hubs;
}

// Classes of a level's rows: of 4, 8 and 16 lanes, of a wave, hubs.
constexpr int LV_CLASSES = 5;
int row_class(int early) {
    return early <= LV_NARROW ? 0 : early <= LV_WIDE ? 1 : early <= LV_BROAD ? 2 : early <= LV_WAVE ? 3 : 4;
}
int count(const bl_graph *g, int l, int c) {
    const int32_t *f = g->lev_first.data() + (size_t)l * LV_CLASSES + c;
    return f[1] - f[0];
}
// The end of the run of small levels without rows of more than 8 entries from level l on.
int run_end(const bl_graph *g, int l) {
    const auto small = [&](int e) {
        return count(g, e, 0) + count(g, e, 1) <= LV_RUN && count(g, e, 2) + count(g, e, 3) + count(g, e, 4) == 0;
    };
    while (l < g->lev_count && small(l)) ++l;
    return l;
}

// Levels and numbers of early entries of all vertices, and the rows of each level and class.
bool scan_levels(bl_graph *g, int B) {
    const int n = g->n;
    if ((int)g->h_rowptr.size() != n + 1 || (int64_t)g->h_colids.size() != g->nnz) return false;
    const int32_t *rp = g->h_rowptr.data(), *ci = g->h_colids.data();
    g->lev_of.resize(n);
    g->lev_early_n.resize(n);
    int32_t *lev = g->lev_of.data(), *ec = g->lev_early_n.data();
    int nl = 0;
    for (int b0 = 0; b0 < n; b0 += B)
        for (int i = b0; i < std::min(n, b0 + B); ++i) {
            int top = -1, c = 0;
            for (int e = rp[i]; e < rp[i + 1]; ++e)
                if (ci[e] < b0) {
                    top = std::max(top, lev[ci[e]]);
                    ++c;
                }
            lev[i] = top + 1;
            ec[i] = c;
            nl = std::max(nl, top + 2);
        }
    if (nl > LV_MAXLEVELS) return false;
    g->lev_count = nl;
    g->lev_first.assign((size_t)nl * LV_CLASSES + 1, 0);
    int32_t *first = g->lev_first.data();
    for (int i = 0; i < n; ++i) ++first[(size_t)lev[i] * LV_CLASSES + row_class(ec[i]) + 1];
    for (size_t k = 0; k < (size_t)nl * LV_CLASSES; ++k) first[k + 1] += first[k];
    g->lev_big = g->lev_small = 0;
    for (int l = 0; l < nl;) {
        const int e = run_end(g, l);
        if (e - l >= LV_RUNS) g->lev_small += e - l, l = e;
        else ++g->lev_big, ++l;
    }
    return true;
}

// A plan's host lists, which the launches don't need.
void forget_levels(bl_graph *g) {
    for (std::vector<int32_t> *v : {&g->lev_of, &g->lev_early_n, &g->lev_first}) std::vector<int32_t>().swap(*v);
}

bool build_plan(bl_graph *g, int B, int D) {
    const int n = g->n, nl = g->lev_count;
    if (D > 0 && g->max_row > LV_ROW) return false;  // the lagged walk's rows, whose sums stay in list order
    const int32_t *rp = g->h_rowptr.data(), *lev = g->lev_of.data(), *ec = g->lev_early_n.data();
    const float *gw = g->h_w.empty() ? nullptr : g->h_w.data();
    const std::vector<int32_t> go = D > 0 ? lag_walk_groups(g, B) : std::vector<int32_t>();
    const std::vector<int32_t> &first = g->lev_first;
    std::vector<int32_t> order(n);
    {
        std::vector<int32_t> at(first.begin(), first.end() - 1);
        for (int i = 0; i < n; ++i) order[at[(size_t)lev[i] * LV_CLASSES + row_class(ec[i])]++] = i;
    }
    constexpr int64_t cap = ((int64_t)1 << 31) - 1;
    // Where every vertex's entries go: slot >= 0 the first of its column in a slice (stride 64), < 0
    // ~ the first of a longer row, or of a short row (marked LV_SHORT).
    struct Build {
        Lists L;
        std::vector<int64_t> slot;
        int64_t nid = 0, nrid = 0;
        void slices(const int32_t *vs, int m, int W) {
            const size_t vat = L.vid.size();
            L.vid.resize(vat + (size_t)(m + 63) / 64 * 64, -1);
            for (int t = 0; t < m; ++t) {
                L.vid[vat + t] = vs[t];
                slot[vs[t]] = nid + (int64_t)(t >> 6) * W * 64 + (t & 63);
            }
            nid += (int64_t)((m + 63) / 64) * W * 64;
        }
        // short rows of W lanes, to whole waves; their number of waves
        int short_rows(const int32_t *vs, int m, int W) {
            const int per = 64 / W, waves = (m + per - 1) / per;
            const size_t vat = L.vid.size();
            L.vid.resize(vat + (size_t)waves * per, -1);
            for (int t = 0; t < m; ++t) {
                L.vid[vat + t] = vs[t];
                slot[vs[t]] = ~((nid + (int64_t)t * W) | LV_SHORT);
            }
            nid += (int64_t)waves * 64;
            return waves;
        }
        void row(int i, int len) {
            slot[i] = ~nrid;
            L.row.push_back(make_int4(i, (int)nrid, (int)(nrid + len), 0));
            nrid += len;
        }
    } E, L;
    E.slot.resize(n);
    L.slot.resize(n);
    // the levels' launches: on their own, or runs of small levels without longer rows
    std::vector<int32_t> start;  // of each level of the runs, its first slice in its run, and the run's end
    std::vector<LevelShape> shape;
    std::vector<int32_t> blk;  // of each workgroup of k_level_flow, its level
    g->lev_launch.clear();
    for (int l = 0; l < nl;) {
        const int e = run_end(g, l);
        const int v0 = (int)E.L.vid.size();
        const uint32_t e0 = (uint32_t)(E.nid / 64);
        const int32_t *vs = order.data() + first[(size_t)l * LV_CLASSES];
        if (e - l >= LV_RUNS) {
            LevelLaunch q{};
            q.v0 = v0;
            q.e0 = e0;
            q.l0 = (int)start.size();
            q.l1 = q.l0 + e - l;
            int at = 0;  // slices of the run
            for (; l < e; ++l) {
                const int m = count(g, l, 0) + count(g, l, 1);
                start.push_back(at);
                E.slices(order.data() + first[(size_t)l * LV_CLASSES], m, LV_WIDE);
                at += (m + 63) / 64;
            }
            start.push_back(at);
            g->lev_launch.push_back(q);
        } else {
            LevelShape q{};
            q.v0 = v0;
            q.e0 = e0;
            q.nn = E.short_rows(vs, count(g, l, 0), LV_NARROW);
            q.nw = E.short_rows(vs += count(g, l, 0), count(g, l, 1), LV_WIDE);
            q.nb = E.short_rows(vs += count(g, l, 1), count(g, l, 2), LV_BROAD);
            vs += count(g, l, 2);
            q.r0 = (int)E.L.row.size();
            q.nr = count(g, l, 3);
            const int nh = count(g, l, 4);
            for (int t = 0; t < q.nr + nh; ++t) E.row(vs[t], ec[vs[t]]);
            if (g->lev_launch.empty() || g->lev_launch.back().l1 > g->lev_launch.back().l0) {
                LevelLaunch f{};
                f.b0 = (int)blk.size();
                g->lev_launch.push_back(f);
            }
            LevelLaunch &f = g->lev_launch.back();
            q.first = f.blocks;
            q.blocks = level_blocks(q.nn + q.nw + q.nb, q.nr, nh);
            q.per = q.blocks < LV_PAIR ? 1 : 2;
            f.blocks += (q.blocks + q.per - 1) / q.per;
            blk.insert(blk.end(), (size_t)(f.blocks - q.first), (int32_t)shape.size());
            shape.push_back(q);
            ++f.levels;
            ++l;
        }
        if (E.nid > cap * 32 || (int64_t)E.L.vid.size() > cap) return false;
    }
    // the late lists: slices in vertex order, sorted by length within windows where rows are long (the lagged
    // walk's sums all in slices, which add in list order)
    const int sliced = D > 0 ? LV_ROW : LV_LATE;
    std::vector<int32_t> win, rows, hubs;
    auto late_len = [&](int i) { return rp[i + 1] - rp[i] - ec[i]; };
    const bool sorted = g->max_row > LV_LATE;
    for (int w0 = 0; w0 < n; w0 += LV_WINDOW) {
        win.clear();
        for (int i = w0; i < std::min(n, w0 + LV_WINDOW); ++i) {
            const int c = late_len(i);
            if (c > LV_WAVE) hubs.push_back(i);
            else if (c > sliced) rows.push_back(i);
            else if (c > 0) win.push_back(i);
        }
        if (sorted)
            std::stable_sort(win.begin(), win.end(), [&](int x, int y) { return late_len(x) < late_len(y); });
        for (size_t t = 0; t < win.size(); t += 64) {
            const int m = (int)std::min<size_t>(64, win.size() - t);
            int W = 0;
            for (int q = 0; q < m; ++q) W = std::max(W, late_len(win[t + q]));
            L.L.head.push_back(make_int2((int)L.nid, W));
            L.slices(win.data() + t, m, W);
        }
        if (L.nid > cap - 2 * LV_WINDOW * LV_ROW) return false;
    }
    for (int i : rows) L.row(i, late_len(i));
    for (int i : hubs) L.row(i, late_len(i));
    const char *penv = getenv("BL_LEVEL_PAD_GIB");  // tests: more than there is
    const size_t pad = penv ? (size_t)std::max(0, atoi(penv)) << 30 : 0;
    hipStream_t st = g->stream;
    struct Temp {
        DevBuf e, l, go;
        ~Temp() { e.release(), l.release(), go.release(); }
    } t;
    if (!E.L.upload(g->lev_early, gw, E.nid, E.nrid, st) || !L.L.upload(g->lev_late, gw, L.nid, L.nrid, st) ||
        !put(g->lev_start, start) || !put(g->lev_blk, blk) || !put(g->lev_shape, shape) ||
        g->lev_moved.ensure(sizeof(double2) * (size_t)n + pad) ||
        g->lev_ticket.ensure(4 * (g->lev_launch.size() + 1) * LV_TICKET_INTS) || !put(t.e, E.slot) ||
        !put(t.l, L.slot) || !put(t.go, go))
        return false;
    const auto fill = [&](const DevBuf &slot, const LevelLists &d) {
        return FillList{slot.as<int64_t>(), d.ids.as<unsigned>(), d.rids.as<unsigned>(),
                        gw ? d.w.as<float>() : nullptr, gw ? d.rw.as<float>() : nullptr};
    };
    hipLaunchKernelGGL(k_level_fill, dim3((n + 255) / 256), dim3(256), 0, st, n, B, D, g->rowptr.as<int>(),
                       g->colids.as<int>(), gw ? g->w_edge.as<float>() : nullptr, t.go.as<int>(),
                       fill(t.e, g->lev_early), fill(t.l, g->lev_late));
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess) return false;
    g->lev_late_slices = (int)L.L.head.size();
    g->lev_late_rows = (int)rows.size();
    g->lev_late_hubs = (int)hubs.size();
    return true;
}
}  // namespace

// The levels for batches of B vertices, in g->lev_big (of launches of consecutive levels) and g->lev_small (of
// runs); cached per batch size.  False: too many.  What the plan's making takes beyond it is spent only
// where the levels are chosen.
bool level_walk_levels(bl_graph *g, int B) {
    if (g->lev_scan == B && (!g->lev_scan_ok || g->lev_batch == B || !g->lev_of.empty())) return g->lev_scan_ok;
    g->lev_scan = B;
    try {
        g->lev_scan_ok = scan_levels(g, B);
    } catch (const std::bad_alloc &) {
        g->lev_scan_ok = false;
    }
    if (!g->lev_scan_ok) forget_levels(g);
    return g->lev_scan_ok;
}

void level_walk_release(bl_graph *g) {
    g->lev_early.release();
    g->lev_late.release();
    for (DevBuf *b : {&g->lev_start, &g->lev_blk, &g->lev_shape, &g->lev_moved, &g->lev_ticket}) b->release();
}

// The plan for batches of B vertices (cached per batch size and lag): levels, their slices and
// hubs, the late lists, and the launches.  D > 0: the sums of the lagged walk with lag D and
// the groups of lag_walk_groups.  False: lists past 2^31 entries, or no memory for them, and then no memory held.
bool level_walk_plan(bl_graph *g, int B, int D) {
    if (g->lev_batch == B && g->lev_d == D) return g->lev_ok;
    g->lev_batch = 0;  // scanned again if the last plan has used the levels up
    if (!level_walk_levels(g, B)) return false;
    try {
        g->lev_ok = build_plan(g, B, D);
    } catch (const std::bad_alloc &) {
        g->lev_ok = false;
    }
    g->lev_batch = B;
    g->lev_d = D;
    forget_levels(g);
    if (!g->lev_ok) {
        level_walk_release(g);
        (void)hipGetLastError();  // the walk in its place runs without it
    }
    return g->lev_ok;
}

namespace {
LevelArgs level_args(const bl_graph *g, const LevelLists &d, double2 *pos, const bl_params *p, double step) {
    LevelArgs a;
    a.head = d.head.as<int2>();
    a.vid = d.vid.as<int>();
    a.ids = d.ids.as<unsigned>();
    a.w = g->has_w ? d.w.as<float>() : nullptr;
    a.row = d.row.as<int4>();
    a.rids = d.rids.as<unsigned>();
    a.rw = g->has_w ? d.rw.as<float>() : nullptr;
    a.lstart = g->lev_start.as<int>();
    a.W = p->weight;
    a.step = step;
    a.pos = pos;
    a.rep = g->bh.rep.as<double2>();
    a.moved = g->lev_moved.as<double2>();
    a.eterm = g->eterm.as<double>();
    a.status = g->bh.misc.as<int>();
    a.blk = nullptr;
    a.shape = g->lev_shape.as<LevelShape>();
    a.ticket = nullptr;
    a.err = g->bh.misc.as<int>() + BH_LEVEL_ERR;
    int khz = 0;
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, g->device) != hipSuccess || khz <= 0)
        khz = 100000;
    a.ticks = (long long)khz * 10000;  // 10 s
    if (const char *w = getenv("BL_LEVEL_WAIT_US")) a.ticks = (long long)khz * atoll(w) / 1000;  // tests
    return a;
}
bool is_flow(const LevelLaunch &q) { return q.blocks > 0; }
}  // namespace

// The late sums, before any vertex moves (and the marks for k_level_flow).  fast: the wide walk's operations.
int launch_level_late(bl_graph *g, double2 *pos, const bl_params *p, bool fast, int it, hipStream_t s) {
    const LevelArgs a = level_args(g, g->lev_late, pos, p, 0.0);
    const int ns = g->lev_late_slices, nr = g->lev_late_rows;
    LevelClear q{level_blocks(ns, nr, g->lev_late_hubs), 0, 0, g->lev_ticket.as<int>(), it == 0};
    const int flows = (int)std::count_if(g->lev_launch.begin(), g->lev_launch.end(), is_flow);
    if (flows) {
        q.n = g->n;
        q.nt = flows * LV_TICKET_INTS;
    }
    const int grid = q.late + (q.n + LV_T - 1) / LV_T;
    if (grid > 0) {
        auto k = g->has_w ? (fast ? k_level_late<true, false> : k_level_late<true, true>)
                          : (fast ? k_level_late<false, false> : k_level_late<false, true>);
        hipLaunchKernelGGL(k, dim3(grid), dim3(LV_T), 0, s, a, ns, nr, q);
    }
    BL_HIP(hipGetLastError());
    return BL_OK;
}

// One iteration's walk (after launch_level_late).
int launch_walk_level(bl_graph *g, double2 *pos, const bl_params *p, bool fast, double step, hipStream_t s) {
    LevelArgs a = level_args(g, g->lev_early, pos, p, step);
    int left = (int)std::count_if(g->lev_launch.begin(), g->lev_launch.end(), is_flow);
    int *ticket = g->lev_ticket.as<int>();
    const bool seq = g->lev_d > 0, ieee = !seq && !fast;
    auto k = g->has_w ? (seq    ? k_level_flow<true, true, false>
                         : fast ? k_level_flow<true, false, false>
                                : k_level_flow<true, false, true>)
                      : (seq    ? k_level_flow<false, true, false>
                         : fast ? k_level_flow<false, false, false>
                                : k_level_flow<false, false, true>);
    auto run = g->has_w ? (ieee ? k_level_run<true, true> : k_level_run<true, false>)
                        : (ieee ? k_level_run<false, true> : k_level_run<false, false>);
    for (const LevelLaunch &q : g->lev_launch) {
        if (is_flow(q)) {
            a.blk = g->lev_blk.as<int>() + q.b0;
            a.ticket = q.levels > 1 ? ticket : nullptr;
            ticket += LV_TICKET_INTS;
            --left;
            hipLaunchKernelGGL(k, dim3(q.blocks), dim3(LV_T), 0, s, a);
        } else {
            if (!left) a.moved = nullptr;
            hipLaunchKernelGGL(run, dim3(1), dim3(1024), 0, s, a, q.l0, q.l1, q.v0, q.e0);
        }
    }
    BL_HIP(hipGetLastError());
    return BL_OK;
}

}  // namespace bl
