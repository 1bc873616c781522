// Device functions of the scalar grouped-scale codec, shared by the kernels that fit, search, encode and
// decode (scalar_codec.hip) and the ones that do it in one pass (scalar_round.hip).  Everything is compared bit for
// bit with IEEE binary32 tensor arithmetic: compile with -ffp-contract=off.
#pragma once

#include "mk_common.h"
#include "packed_matvec_impl.h"   // lane_exchange

namespace mk_scalar {

constexpr int kMaxTable = 256;
constexpr int kThreads = 256;

// Index of the first table entry >= x by bisection over a table padded with +inf, then
// the nearer of that entry and the one below it; equal distances pick the lower entry.
__device__ __forceinline__ int nearest_entry(float x, const float *table, int count, int steps) {
    int lower = 0, upper = count;
    for (int s = 0; s < steps; ++s) {
        const int middle = (lower + upper) >> 1;
        const float candidate = middle < count ? table[middle] : __builtin_inff();
        const bool right = candidate < x;
        lower = right ? middle + 1 : lower;
        upper = right ? upper : middle;
    }
    const int above = lower < count - 1 ? lower : count - 1;
    const int below = above > 0 ? above - 1 : 0;
    const float below_distance = fabsf(__fsub_rn(x, table[below]));
    const float above_distance = fabsf(__fsub_rn(x, table[above]));
    return below_distance <= above_distance ? below : above;
}

__device__ __forceinline__ float nearest_integer(float x, float minimum, float maximum) {
    return fminf(fmaxf(rintf(x), minimum), maximum);
}

__device__ __forceinline__ int bisection_steps(int count) {
    int steps = 0;
    while ((1 << steps) < count + 1) ++steps;
    return steps;
}

__device__ __forceinline__ void stage_table(float *shared, const float *values, int count) {
    for (int i = threadIdx.x; i < count; i += blockDim.x) shared[i] = values[i];
    __syncthreads();
}

// Scale of a group from its extrema, before storage rounding; `zero`: the offset of an asymmetric grid.
__device__ __forceinline__ float range_scale(float low, float high, int asym, float reciprocal, float value_minimum, float &zero) {
    if (asym) {
        const float scale = __fmul_rn(fmaxf(__fsub_rn(high, low), 1e-12f), reciprocal);
        zero = __fsub_rn(low, __fmul_rn(value_minimum, scale));
        return scale;
    }
    zero = 0.0f;
    return __fmul_rn(fmaxf(fmaxf(high, -low), 1e-12f), reciprocal);
}

// Storage rounding of an offset: its magnitude as a scale's, its sign kept.
__device__ __forceinline__ float rounded_offset(float zero, int format) {
    const float magnitude = mk_rounded_scale(fmaxf(fabsf(zero), 1e-12f), format);
    return zero > 0.0f ? magnitude : (zero < 0.0f ? -magnitude : 0.0f);
}

// Minimum, maximum and "all finite" over the LANES adjacent lanes of a team, by vector-ALU
// lane moves (an LDS permute per step cost more than the loads of the group).
template <int LANES>
__device__ __forceinline__ void team_range(float &low, float &high, bool &finite, int lane) {
    float bad = finite ? 0.0f : 1.0f;
    auto stage = [&](auto s) __attribute__((always_inline)) {
        constexpr int S = decltype(s)::value;
        if constexpr ((1 << S) < LANES) {
            low = fminf(low, mk_matvec::lane_exchange<S>(low, lane));
            high = fmaxf(high, mk_matvec::lane_exchange<S>(high, lane));
            bad = fmaxf(bad, mk_matvec::lane_exchange<S>(bad, lane));
        }
    };
    stage(std::integral_constant<int, 0>{});
    stage(std::integral_constant<int, 1>{});
    stage(std::integral_constant<int, 2>{});
    stage(std::integral_constant<int, 3>{});
    stage(std::integral_constant<int, 4>{});
    stage(std::integral_constant<int, 5>{});
    finite = bad == 0.0f;
}

}  // namespace mk_scalar
