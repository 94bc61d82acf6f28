// What the tree traversals of one wave share (64 Morton-consecutive queries and one stack).
//
// What bounds a traversal is the instructions its steps issue, vector and scalar alike: a SIMD takes
// four cycles for either (the four SIMDs of a CU share one scalar unit), and at 8 waves per SIMD the
// loads are hidden.  (Counted on the monopole traversal of a triangulation of 1.66M points at theta
// 0.4: 94% of the cycles vector instructions; with some of them turned into twice as many scalar
// ones, 85% scalar instructions and a longer run.)  So the stack lives in registers, the lanes'
// masks are combined on the scalar unit, nothing is computed twice, and the two kinds are kept in
// balance.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bl {

// A wave-uniform value in scalar registers.
__device__ __forceinline__ int scalar(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ double scalar(double v) {
    return __hiloint2double(scalar(__double2hiint(v)), scalar(__double2loint(v)));
}

// v_writelane_b32 with a uniform value and lane (no builtin for it in this compiler)
extern "C" __device__ __attribute__((const)) int bl_writelane(int value, int lane, int old) __asm(
    "llvm.amdgcn.writelane.i32");

// A wave's stack of (node, lanes): entry e in lane e of three registers, entry 0 the end
// mark.  Pushes and pops are lane writes and reads, where a stack in LDS took an exec mask,
// addresses and a round trip.  An opened node pushes its children without a branch: every child is
// written at the top, which only an internal one raises.  At most 3 siblings wait on each of 32
// levels; past 60 entries the oldest 31 go to LDS until the others are done.
constexpr int WAVE_STACK_SAVE = 128;  // LDS ints per register
constexpr int WAVE_STACK_END = -1;    // popped when no entry is left in the registers

struct WaveStack {
    int node, lo = 0, hi = 0;
    int sp = 1, saved = 0;  // sp: the top entry's lane
    int lane;
    int *save;  // [3][WAVE_STACK_SAVE], this wave's
    __device__ __forceinline__ WaveStack(int lane_, int *save_, int root, uint64_t lanes) : lane(lane_), save(save_) {
        node = lane == 0 ? WAVE_STACK_END : root;
        lo = (int)(unsigned)lanes;
        hi = (int)(unsigned)(lanes >> 32);
    }
    __device__ __forceinline__ int pop(uint64_t &lanes) {
        const int v = __builtin_amdgcn_readlane(node, sp);
        lanes = ((uint64_t)(unsigned)__builtin_amdgcn_readlane(hi, sp) << 32) |
                (unsigned)__builtin_amdgcn_readlane(lo, sp);
        --sp;
        return v;
    }
    // after the end mark: brings entries back from LDS; false when there is none
    __device__ __forceinline__ bool more() {
        if (saved == 0) return false;
        saved -= 31;
        const int e = saved + max(lane - 1, 0) % 31;
        node = lane == 0 ? WAVE_STACK_END : save[e];
        lo = save[WAVE_STACK_SAVE + e];
        hi = save[2 * WAVE_STACK_SAVE + e];
        sp = 31;
        return true;
    }
    // an opened node's internal children, the first quadrant on top
    __device__ __forceinline__ void push_children(int4 ch, uint64_t lanes) {
        if (sp > 59) put_away();
        if (__builtin_amdgcn_inverse_ballot_w64(0x1Eull << scalar(sp))) {
            lo = (int)(unsigned)lanes;
            hi = (int)(unsigned)(lanes >> 32);
        }
        const int c[4] = {ch.w, ch.z, ch.y, ch.x};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int x = scalar(c[q]);
            node = bl_writelane(x, scalar(sp) + 1, node);
            sp += x >= 0;
        }
    }
    // entries 1 .. 31 to LDS, the others down by 31
    __device__ __forceinline__ void put_away() {
        if (lane > 0 && lane < 32) {
            const int e = saved + lane - 1;
            save[e] = node;
            save[WAVE_STACK_SAVE + e] = lo;
            save[2 * WAVE_STACK_SAVE + e] = hi;
        }
        const int from = lane == 0 ? 0 : min(lane + 31, 63);
        node = __shfl(node, from, 64);
        lo = __shfl(lo, from, 64);
        hi = __shfl(hi, from, 64);
        saved += 31;
        sp -= 31;
        __builtin_amdgcn_wave_barrier();
    }
};

// The traversal loop itself, in assembly.  Written in C++ the loop carried twice as many
// instructions as it needs: its sums and stack copied between registers around every branch, masks
// turned into vector registers and back, scalar selects.  One block runs until it meets the end mark,
// a full stack or a case for the caller (TRAV_NEAR), with every lane of the wave active on entry and
// on exit.  A step: pop a node, add the term of the lanes that accept it; for the others its leaves'
// terms, last quadrant first, then push its other children.  Its waits: each scalar load is waited
// for before its first use, in the block.  Its fixed registers: s80 the entry, s[84:85] its lanes,
// s[86:87] those that accept, s[88:89] those that do not, s[64:79] the node, s[90:91] the squared
// side over MAXMIN (s81 and s90 zero throughout).
//
// Wait states of gfx950 that an assembler does not insert: one between a reciprocal (or root) and its
// use, one between the write of a vector register and its v_readlane, two between a vector
// instruction's scalar result and its use as a vector operand; none of these pairs is closer here.
// Four between a vector instruction's scalar result and its use as the lane of a v_readlane: %[sp]
// comes in by v_readfirstlane, so the block begins with them; inside it %[sp] and m0 are the
// scalar unit's.
enum TravStop : int { TRAV_END = 0, TRAV_FULL = 1, TRAV_NEAR = 2 };

#define BL_TRAV_POP                          \
    "s_nop 3\n\t"                            \
    "s_mov_b32 s81, 0\n\t"                   \
    "s_mov_b32 s90, 0\n\t"                   \
    "s_mov_b32 %[why], 0\n"                  \
    "Lpop%=:\n\t"                            \
    "v_readlane_b32 s80, %[node], %[sp]\n\t" \
    "v_readlane_b32 s84, %[lo], %[sp]\n\t"   \
    "v_readlane_b32 s85, %[hi], %[sp]\n\t"   \
    "s_sub_u32 %[sp], %[sp], 1\n\t"          \
    "s_cmp_lt_i32 s80, 0\n\t"                \
    "s_cbranch_scc1 Lout%=\n\t"

// (dx, dy) = c - p, r2 = dx^2 + dy^2 for c in s[64:67]
#define BL_TRAV_DIST                           \
    "v_add_f64 %[dx], s[64:65], -%[px]\n\t"    \
    "v_add_f64 %[dy], s[66:67], -%[py]\n\t"    \
    "v_mul_f64 %[r2], %[dx], %[dx]\n\t"        \
    "v_fma_f64 %[r2], %[dy], %[dy], %[r2]\n\t"

// the lanes that accept a node of depth s75 by its side, 4^-depth < `open` r2, and the others (scc: any)
#define BL_TRAV_TEST(open)                          \
    "s_lshl_b32 s91, s75, 21\n\t"                   \
    "s_sub_u32 s91, 0x3ff00000, s91\n\t"            \
    "v_mul_f64 %[t], " open ", %[r2]\n\t"           \
    "v_cmp_lt_f64 vcc, s[90:91], %[t]\n\t"          \
    "s_and_b64 s[86:87], vcc, s[84:85]\n\t"         \
    "s_andn2_b64 s[88:89], s[84:85], s[86:87]\n\t"

// the accepting lanes' term
#define BL_TRAV_TAKE(term)             \
    "s_mov_b64 exec, s[86:87]\n\t"     \
    "s_cbranch_execz Lopen%=\n\t" term \
    "Lopen%=:\n\t"

// the term of the opened node's child c if it is a leaf, for the lanes away from it (c in s[64:67])
#define BL_TRAV_LEAF(c, term)                  \
    "s_cmp_gt_i32 " c ", -2\n\t"               \
    "s_cbranch_scc1 Lno" c "%=\n\t"            \
    "s_sub_u32 s80, -2, " c "\n\t"             \
    "s_lshl_b64 s[82:83], s[80:81], 4\n\t"     \
    "s_add_u32 s82, s82, %[spos0]\n\t"         \
    "s_addc_u32 s83, s83, %[spos1]\n\t"        \
    "s_load_dwordx4 s[64:67], s[82:83], 0\n\t" \
    "s_mov_b64 exec, s[88:89]\n\t"             \
    "s_waitcnt lgkmcnt(0)\n\t" BL_TRAV_DIST    \
    "v_cmp_lt_f64 vcc, 0, %[r2]\n\t"           \
    "s_and_b64 exec, vcc, s[88:89]\n\t" term   \
    "Lno" c "%=:\n\t"

// one internal child to the next lane, which it keeps
#define BL_TRAV_CHILD(c)                        \
    "v_writelane_b32 %[node], " c ", m0\n\t"    \
    "s_cmp_gt_i32 " c ", -1\n\t"                \
    "s_addc_u32 m0, m0, 0\n\t"

// the node is opened for s[88:89]: its leaves, then its children on the stack, the first one on top; on,
// unless the stack may not hold another node's children.  c0 .. c3: past the registers of a leaf's
// position.
#define BL_TRAV_OPEN(c0, c1, c2, c3, term)                                             \
    "s_mov_b64 exec, -1\n\t"                                                           \
    "s_cmp_eq_u64 s[88:89], 0\n\t"                                                     \
    "s_cbranch_scc1 Lpop%=\n\t"                                                        \
    BL_TRAV_LEAF(c3, term) BL_TRAV_LEAF(c2, term)                                      \
    BL_TRAV_LEAF(c1, term) BL_TRAV_LEAF(c0, term)                                      \
    "s_lshl_b64 exec, 30, %[sp]\n\t"                                                   \
    "v_mov_b32 %[lo], s88\n\t"                                                         \
    "v_mov_b32 %[hi], s89\n\t"                                                         \
    "s_mov_b64 exec, -1\n\t"                                                           \
    "s_add_u32 m0, %[sp], 1\n\t"                                                       \
    BL_TRAV_CHILD(c3) BL_TRAV_CHILD(c2) BL_TRAV_CHILD(c1) BL_TRAV_CHILD(c0)            \
    "s_sub_u32 %[sp], m0, 1\n\t"                                                       \
    "s_cmp_lt_i32 %[sp], 60\n\t"                                                       \
    "s_cbranch_scc1 Lpop%=\n\t"                                                        \
    "s_mov_b32 %[why], 1\n\t"                                                          \
    "s_branch Lout%=\n"

// %[s] = 1 / r2 by the hardware's estimate and one Newton step, `between` in the estimate's shadow
#define BL_TRAV_RECIP(between)                 \
    "v_rcp_f64 %[s], %[r2]\n\t" between        \
    "v_fma_f64 %[t], -%[r2], %[s], 1.0\n\t"    \
    "v_fma_f64 %[s], %[s], %[t], %[s]\n\t"

// %[s] = 1 / sqrt(r2): the FP32 estimate q and one FP64 Newton step q (3/2 - (r2/2) q^2)
#define BL_TRAV_RSQRT                          \
    "v_cvt_f32_f64 %[q], %[r2]\n\t"            \
    "v_rsq_f32 %[q], %[q]\n\t"                 \
    "v_mul_f64 %[t], -0.5, %[r2]\n\t"          \
    "v_cvt_f64_f32 %[s], %[q]\n\t"             \
    "v_mul_f64 %[t], %[t], %[s]\n\t"           \
    "v_fma_f64 %[t], %[t], %[s], %[c15]\n\t"   \
    "v_mul_f64 %[s], %[s], %[t]\n\t"

#define BL_TRAV_ADD                            \
    "v_fma_f64 %[fx], %[dx], %[s], %[fx]\n\t"  \
    "v_fma_f64 %[fy], %[dy], %[s], %[fy]\n\t"

#define BL_TRAV_CLOBBERS                                                                                     \
    "vcc", "scc", "m0", "s64", "s65", "s66", "s67", "s68", "s69", "s70", "s71", "s72", "s73", "s74", "s75",  \
    "s76", "s77", "s78", "s79", "s80", "s81", "s82", "s83", "s84", "s85", "s86", "s87", "s88", "s89", "s90", \
    "s91", "s92"

}  // namespace bl
