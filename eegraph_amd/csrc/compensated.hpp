// Compensated FP32 arithmetic of the PageRank kernels.
#pragma once

#include "device.hpp"

namespace eeg {

struct Comp {  // value s with the rounding error e that s + e represents exactly
    float s, e;
};
__device__ __forceinline__ Comp two_sum(float a, float b) {
    const float s = a + b;
    const float bb = s - a;
    const float err = (a - (s - bb)) + (b - bb);
    return Comp{s, err};
}
__device__ __forceinline__ Comp comp_add(Comp a, Comp b) {
    const Comp t = two_sum(a.s, b.s);
    return Comp{t.s, t.e + (a.e + b.e)};
}

// Value of lane (this lane + OFF) of the same 16-lane row: a DPP row shift (one VALU move, no
// LDS permute) for OFF < 16, a shuffle beyond.  Lanes whose partner lies outside the row get 0.
template <int OFF>
__device__ __forceinline__ float lane_down(float v) {
    if constexpr (OFF < 16) {
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x100 + OFF, 0xF, 0xF, false));
    } else {
        return __shfl_down(v, OFF, WAVE);
    }
}

// Compensated sum of the x of a group of K aligned lanes, valid in the group's first lane:
// a pairwise tree, ((x0 + x1) + (x2 + x3)) + ((x4 + x5) + (x6 + x7)) for K = 8, each step a
// TwoSum with the error terms carried.  The tree and the operand order are fixed, so the bits
// do not depend on the schedule.
template <int K, int OFF = 1>
__device__ __forceinline__ Comp group_reduce_step(Comp c) {
    if constexpr (OFF >= K) {
        return c;
    } else {
        Comp o;
        o.s = lane_down<OFF>(c.s);
        o.e = lane_down<OFF>(c.e);
        return group_reduce_step<K, 2 * OFF>(comp_add(c, o));
    }
}
template <int K>
__device__ __forceinline__ Comp group_sum_first_lane(float x) {
    // first level: the inputs carry no error term
    const Comp c = two_sum(x, lane_down<1>(x));
    return group_reduce_step<K, 2>(c);
}

// New rank base + d * sum kept as an FP32 pair (hi, lo): the product d*s is split exactly with
// an FMA, base + d*s with TwoSum, and the small terms folded into lo.  The pair carries ~46
// bits.  No contraction: the compiler would put d*s into an FMA with the base, whose TwoSum error
// then holds the rounding error of the product that pe adds again.
__device__ __forceinline__ void rank_pair(float base, float d, Comp sum, float* hi, float* lo) {
#pragma clang fp contract(off)
    const float p = d * sum.s;
    const float pe = fmaf(d, sum.s, -p);
    const Comp q = two_sum(base, p);
    const float small = q.e + (pe + d * sum.e);
    const float h = q.s + small;            // fast two-sum: |q.s| >= |small|
    *hi = h;
    *lo = small - (h - q.s);
}

// The contribution of a rank to each out-neighbour.
__device__ __forceinline__ float contribution(float hi, float lo, uint32_t od) {
    return od ? (hi + lo) / (float)od : 0.0f;
}
// The contribution c with the last rounding error *e added; *e receives the error of the sum.  What c
// itself lost is the remainder of its division (an FMA gives it exactly).
__device__ __forceinline__ float fed_contribution(float c, float hi, float lo, uint32_t od, float* e) {
    if (!od) return 0.0f;  // (nothing gathers it)
    const float d = (float)od;
    const float t = (fmaf(-c, d, hi) + lo) * __builtin_amdgcn_rcpf(d) + *e;
    const float f = c + t;  // fast two-sum: |c| >= |t|, a few roundings of it
    *e = t - (f - c);
    return f;
}

// Rounding errors of contributions are fed back from an iteration on whose L1 change r follows
// - r <= FEED_FROM / (1 - d): what single floats leave adds up to some 2^-24 / (1 - d),
// - r > (d + (1 - d) / 4) * the change before (`last`): it falls by d or more but for rounding,
// while r > FEED_TO; below, they are dropped, and the iteration settles on a fixed point for smaller
// stops.  (CPU runs: grids and bipartite graphs, d = 0.5 .. 0.99, meet the 1e-7 stop at most a few
// iterations after FP64 does; RMAT graphs are left alone.)
constexpr double FEED_FROM = 1.5e-7, FEED_TO = 5e-8;
enum Feed : uint32_t { FEED_WRITE = 1, FEED_READ = 2 };  // what an iteration does with the errors
struct FeedRule {  // the two bounds for a damping
    double factor, from;
    explicit FeedRule(double d) : factor(d + 0.25 * (1.0 - d)), from(FEED_FROM / (1.0 - d)) {}
};
// Feed bits of the next iteration; `was`: of the one that ended, `wrote`: whether it could follow them.
__device__ __forceinline__ uint32_t next_feed(double r, double last, const FeedRule& f, uint32_t was, bool wrote) {
    if (!(r > FEED_TO && r <= f.from && ((was & FEED_WRITE) || r > f.factor * last))) return 0u;
    return FEED_WRITE | ((was & FEED_WRITE) && wrote ? FEED_READ : 0u);
}

}  // namespace eeg
