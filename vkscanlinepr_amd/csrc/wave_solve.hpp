// wave_solve.hpp -- the crossings of a chain solved one after another by a whole wave (gfx950).
//
// A chain's crossings depend on each other, and a lane takes 0.7 to 1.1 us for one: 24 halvings, one
// evaluation after another.  Where no guess of a later start comes true (k_curves.hip), a wave
// does the halvings six at a time: its lanes are the nodes of a tree of six levels, each halves the
// bracket along its own path, exactly as the sequential bisection would, and evaluates its midpoint; a
// ballot of the decisions names the path taken.  0.4 to 0.5 us a crossing, for 13 times the arithmetic:
// it pays where few chains are left to wait for.
#pragma once

#include "device_common.hpp"

namespace spr {

// Where a lane stands: node `lane` of the tree (node 1 is the root, nodes 2n and 2n + 1 are left and right of
// node n).  left[l], right[l]: the way from the root turns there at level l; above, turns: the nodes on the way to
// a lowest node, and those where it turns right.
constexpr int kTreeLevels = 6;
static_assert(kCubicIters % kTreeLevels == 0 && (1 << kTreeLevels) == 64, "rounds of a wave's tree");
struct TreeNode {
    bool left[kTreeLevels - 1], right[kTreeLevels - 1];
    unsigned long long above, turns;
};
__device__ inline TreeNode tree_node(int lane) {
    TreeNode n;
    const int depth = lane ? 31 - __clz(lane) : 0;
    n.above = 0ull;
    n.turns = depth == kTreeLevels - 1 ? 0ull : 1ull;  // node 0 decides nothing: no match for the inner nodes
#pragma unroll
    for (int l = 0; l < kTreeLevels - 1; ++l) {
        const bool on = l < depth, r = on && ((lane >> (depth - 1 - l)) & 1) != 0;
        n.left[l] = on && !r;
        n.right[l] = r;
        const unsigned long long at = on ? 1ull << (lane >> (depth - l)) : 0ull;
        n.above |= at;
        n.turns |= r ? at : 0ull;
    }
    return n;
}

// The halvings of one crossing by a wave; all arguments are the same in all lanes.  right(v): the bracket's upper
// half goes on from a midpoint of value v.  The last midpoint and its value go to tm and vm.
template <uint32_t T, class F>
__device__ inline void halve_wave(const TreeNode& N, const CurveAxis& ax, float t_min, float t1, float& tm, float& vm,
                                  F&& right) {
    float t_lo = t_min, t_hi = t1, m = 0.0f, v = 0.0f;
    int node = 0;
    auto from = [&](float x) { return bitsf((uint32_t)__builtin_amdgcn_readlane((int)fbits(x), node)); };
#pragma unroll 2
    for (int round = 0; round < kCubicIters / kTreeLevels; ++round) {
        float lo = t_lo, hi = t_hi;
#pragma unroll
        for (int l = 0; l < kTreeLevels - 1; ++l) {
            m = (lo + hi) * 0.5f;
            lo = N.right[l] ? m : lo;
            hi = N.left[l] ? m : hi;
        }
        m = (lo + hi) * 0.5f;
        v = eval_axis(T, m, ax.c[0], ax.c[1], ax.c[2], ax.c[3]);
        const bool r = right(v);
        lo = r ? m : lo;
        hi = r ? hi : m;
        const unsigned long long d = __ballot(r);
        node = __ffsll((long long)__ballot((d & N.above) == N.turns)) - 1;
        t_lo = from(lo);
        t_hi = from(hi);
    }
    tm = from(m);
    vm = from(v);
}

// Crossings 0..n-1 of a chain by a whole wave: put(k, v) takes value k (the parameter with its two low bits
// replaced by the side), in order and in every lane.  The usual case takes bisect_below's one compare
// under the conditions of ChainSolver, the others bisect_axis's signs.
template <uint32_t T, class F>
__device__ inline void solve_wave(const TreeNode& N, const CurveAxis& a, float line0, float step, uint32_t side, float t1,
                                  int n, float tstart, F&& put) {
    const bool fast = fast_axis(T, a) && fast_t(t1), neg = fast && step < 0.0f;
    const CurveAxis an = neg ? negated(a) : a;
    bool known = false;
    float tprev = tstart, line = line0;  // lines are small integers: exact
#pragma unroll 1
    for (int k = 0; k < n; ++k) {
        float tm = tprev, vm;
        const bool in_range = fast && fast_t(tprev);
        if (T != kArc && in_range && known) {
            const float cn = neg ? -line : line, cut = neg ? next_up(cn) : cn;
            halve_wave<T>(N, an, tprev, t1, tm, vm, [&](float v) { return v < cut; });
            known = !(fabsf(vm - cn) > 1.0f);
            tm = known ? tm : tprev;
        } else {
            const float d0 = eval_axis(T, tprev, a.c[0], a.c[1], a.c[2], a.c[3]) - line;
            known = in_range;
            if (d0 != 0.0f) {
                const uint32_t s0 = fbits(d0) & 0x80000000u;
                halve_wave<T>(N, a, tprev, t1, tm, vm,
                              [&](float v) { return (fbits(v - line) & 0x80000000u) == s0; });
                const bool ok = !(fabsf(vm - line) > 1.0f);
                known = in_range && ok && (s0 != 0u) == (step > 0.0f);
                tm = ok ? tm : tprev;
            }
        }
        tprev = bitsf((fbits(tm) & 0xFFFFFFFCu) | side);
        put(k, tprev);
        line += step;
    }
}

// For a curve type known at run time (no line).
template <class F>
__device__ inline void solve_wave_any(const TreeNode& N, uint32_t type, const CurveAxis& a, float line0, float step,
                                      uint32_t side, float t1, int n, float tstart, F&& put) {
    if (type == kCubic) solve_wave<kCubic>(N, a, line0, step, side, t1, n, tstart, put);
    else if (type == kQuad) solve_wave<kQuad>(N, a, line0, step, side, t1, n, tstart, put);
    else solve_wave<kArc>(N, a, line0, step, side, t1, n, tstart, put);
}

// About how many of a chain's n crossings lie before parameter tau.
__device__ inline int crossings_before(uint32_t type, const CurveAxis& a, float line0, bool neg, float t0, float tau, int n) {
    if (!(t0 < tau)) return 0;
    const float d = eval_axis(type, tau, a.c[0], a.c[1], a.c[2], a.c[3]) - line0;
    const float k = (neg ? -d : d) * 0.5f + 2.0f;
    return k >= (float)n ? n : (k > 0.0f ? (int)k : 0);
}

// A chain has a long start when many crossings lie near t = 0, where two runs of the bisection from different starts
// hardly ever fall together (k_curves.hip): more than kLongHead before 1/32 of its end parameter, or more than
// kLongEighth before 1/8.
constexpr int kLongHead = 64, kLongEighth = 224;
constexpr float kHeadTau = 0.03125f, kEighth = 0.125f;
__device__ inline bool long_start(uint32_t type, const CurveAxis& a, float line0, bool neg, float t0, float t1, int n) {
    return n > kLongHead && t0 < kEighth * t1 &&
           (crossings_before(type, a, line0, neg, t0, kEighth * t1, n) > kLongEighth ||
            crossings_before(type, a, line0, neg, t0, kHeadTau * t1, n) > kLongHead);
}

}  // namespace spr
