// Rounding a weight matrix to a scaled scalar grid in one pass: range, stored scale and offset, optional search of a
// shrunken scale, codes.  The weight is read once, in its own type; a group stays in registers from its range to its
// codes.  Same values as mk_fit_scales -> mk_search_scales -> mk_scalar_encode on the FP32 matrix, bit for bit.
//
// Covers what /root/reference/src/mlkit spreads over formats/grouped_scaling.py:132-175,274-289 (range fit, storage
// rounding), kernels/scalar_encode.py:261-304 (search_scales) and :110-146 (encode).
//
// Without a search the pass is bound by HBM (2 or 4 bytes in, 1 out per weight).  Five instead of about ten
// instructions per quotient keep the vector ALUs below that: a lane divides once per group, and Markstein's
// two corrections with the correctly rounded reciprocal give the correctly rounded quotient.
// 4096 x 14336 fp16 to INT4 g128 with offsets: 43 us = 4.1 TB/s (a device copy: 5.1), against 163 us for the
// conversion to FP32, the range fit and the encoding as passes of their own (53 + 58 + 52).
// A search is bound by the vector ALUs: 21 candidates, each a quotient and a rounding per weight.  4096 x 4096 on
// seven values, g64: 131 us, against 496 us with an IEEE division and a bisection of the table per candidate and
// weight, and 236 us with thresholds kept in registers and the exact error of every candidate; groups of 64 columns and
// more on integers or at most eight values now work out an estimate for each candidate (7 instructions a weight where the
// values lie symmetrically about zero) and the exact error only where the estimate leaves the choice open.

#include "scalar_codec_impl.h"

using namespace mk_scalar;

namespace {

struct RoundArgs {
    const void *value;
    const float *values;
    const float *fractions;
    float *scales;
    float *zeros;
    uint8_t *codes;
    int *flag;
    int rows, width, group, groups_per_row, total_groups;
    int dtype, n_values, n_fractions, format, asym, aligned;
    uint32_t row_multiplier;   // identifier / groups_per_row = umulhi(identifier, multiplier) >> shift
    int row_shift;
    float reciprocal, minimum, maximum;
};

// How a normalized value becomes a code: consecutive integers, a table of at most eight values whose thresholds are
// kept in registers, or a longer table bisected in LDS.
enum Rounding { kInteger, kFewValues, kTable };

constexpr int kFew = 8;

// x / divisor, correctly rounded.  `reciprocal` is 1 / divisor rounded to nearest.  The first product may be off by 1.5
// units in the last place; one correction leaves it faithful, its remainder is then exact, and a second
// correction rounds correctly (Markstein, "IA-64 and Elementary Functions", 2000, the division theorem).  The
// caller keeps divisors whose reciprocals leave the normal range off this path; quotients so small that a remainder
// underflows round to the same code either way.
__device__ __forceinline__ float corrected_quotient(float x, float divisor, float reciprocal) {
    float q = __fmul_rn(x, reciprocal);
    q = __fmaf_rn(__fmaf_rn(-q, divisor, x), reciprocal, q);
    return __fmaf_rn(__fmaf_rn(-q, divisor, x), reciprocal, q);
}

__device__ __forceinline__ uint32_t ordered_bits(float x) {
    const uint32_t bits = __float_as_uint(x);
    return bits & 0x80000000u ? ~bits : bits | 0x80000000u;
}

__device__ __forceinline__ float from_ordered_bits(uint32_t ordered) {
    return __uint_as_float(ordered & 0x80000000u ? ordered & 0x7fffffffu : ~ordered);
}

// The largest float that nearest_entry() gives a code of at most `k`: between two entries the rounded distances
// are monotone, so bisection over the floats finds it.
__device__ float upper_threshold(const float *table, int k) {
    const float below = table[k], above = table[k + 1];
    if (!(below < above)) return below;   // equal entries: the first one answers up to its value
    uint32_t inside = ordered_bits(below), outside = ordered_bits(above);
    while (outside - inside > 1) {
        const uint32_t middle = inside + (outside - inside) / 2;
        const float x = from_ordered_bits(middle);
        const bool lower = fabsf(__fsub_rn(x, below)) <= fabsf(__fsub_rn(x, above));
        inside = lower ? middle : inside;
        outside = lower ? outside : middle;
    }
    return from_ordered_bits(inside);
}

// Minimum and maximum that keep NaNs (three operands an instruction on gfx950).
__device__ __forceinline__ float smallest(float a, float b) { return __builtin_elementwise_minimum(a, b); }
__device__ __forceinline__ float largest(float a, float b) { return __builtin_elementwise_maximum(a, b); }

template <int LANES>
__device__ __forceinline__ void team_extrema(float &low, float &high, int lane) {
    auto stage = [&](auto s) __attribute__((always_inline)) {
        constexpr int S = decltype(s)::value;
        if constexpr ((1 << S) < LANES) {
            low = smallest(low, mk_matvec::lane_exchange<S>(low, lane));
            high = largest(high, mk_matvec::lane_exchange<S>(high, lane));
        }
    };
    stage(std::integral_constant<int, 0>{});
    stage(std::integral_constant<int, 1>{});
    stage(std::integral_constant<int, 2>{});
}

// rint and clamp; one instruction each where fminf / fmaxf take two.
__device__ __forceinline__ float nearest_grid_integer(float x, float minimum, float maximum) {
    return __builtin_amdgcn_fmed3f(rintf(x), minimum, maximum);
}

// A team of TEAM lanes owns a group of TEAM * 8 * TRIPS values; lane q holds values 8 q ... 8 q + 7 of every
// TEAM * 8.  The squared errors of a candidate are added as search_kernel of scalar_codec.hip adds them: TEAM * 8
// partial sums over the trips, folded pairwise (values 1, 2, 4 apart inside the lane, then lanes 1, 2, 4 apart).
template <int ROUNDING, bool SEARCH, int TEAM, int TRIPS>
__global__ void __launch_bounds__(kThreads) round_groups_kernel(const RoundArgs a) {
    constexpr int kSpan = TEAM * 8;
    constexpr int kTeams = kThreads / TEAM;
    __shared__ float table[kMaxTable];
    __shared__ float threshold[kMaxTable];
    __shared__ float fraction[64];
    float few_threshold[kFew - 1], few_value[kFew];
    int steps = 0;
    // Quotients up to which the thresholds say what nearest_entry() does.  Past the last entry that one takes the entry
    // below it once both distances round to one number (or the two are equal), which 2^21 of their distance keep well away.
    float limit = __builtin_inff();
    auto uniform = [](float x) __attribute__((always_inline)) -> float {   // in a scalar register
        return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
    };
    if constexpr (ROUNDING != kInteger) {
        stage_table(table, a.values, a.n_values);
        for (int k = threadIdx.x; k < a.n_values; k += kThreads)
            threshold[k] = k + 1 < a.n_values ? upper_threshold(table, k) : __builtin_inff();
        __syncthreads();
        if (a.n_values > 1) limit = uniform(table[a.n_values - 1] + (table[a.n_values - 1] - table[a.n_values - 2]) * 0x1p21f);
        if constexpr (ROUNDING == kFewValues) {
#pragma unroll
            for (int k = 0; k < kFew - 1; ++k) few_threshold[k] = k < a.n_values ? threshold[k] : __builtin_inff();
#pragma unroll
            for (int k = 0; k < kFew; ++k) few_value[k] = table[k < a.n_values ? k : a.n_values - 1];
        } else {
            while ((1 << steps) < a.n_values) ++steps;
        }
    }
    // Searched scales, teams of eight: a first pass over the candidates with a cheaper error (see `prune`).
    constexpr bool kPruned = SEARCH && TEAM == 8 && ROUNDING != kTable;
    __shared__ float estimate[kPruned ? kTeams : 1][64 + 1];
    bool symmetric = ROUNDING == kFewValues;   // uniform
    float magnitude[kFew / 2];                 // then: the values from zero up
    if constexpr (kPruned && ROUNDING == kFewValues) {
        for (int k = 0; k < a.n_values; ++k) symmetric = symmetric && table[k] == -table[a.n_values - 1 - k];
#pragma unroll
        for (int k = 0; k < kFew / 2; ++k) magnitude[k] = table[min(a.n_values / 2 + k, a.n_values - 1)];
    }
    bool ordinary_fractions = true;
    float least_fraction = 1.0f;
    if constexpr (SEARCH) {
        for (int i = threadIdx.x; i < a.n_fractions; i += kThreads) fraction[i] = a.fractions[i];
        __syncthreads();
        for (int i = 0; i < a.n_fractions; ++i) {
            ordinary_fractions = ordinary_fractions && fraction[i] > 0x1p-10f && fraction[i] < 0x1p10f;
            least_fraction = fminf(least_fraction, fraction[i]);
        }
        least_fraction = uniform(least_fraction);
    }
    const int lane_in_team = threadIdx.x % TEAM;

    // The code of a normalized value (tables), and its value on the grid.
    auto code_of = [&](float x) __attribute__((always_inline)) -> int {
        if constexpr (ROUNDING == kFewValues) {
            int code = 0;
#pragma unroll
            for (int k = 0; k < kFew - 1; ++k) code += x > few_threshold[k] ? 1 : 0;
            return code;
        } else {
            int code = 0;   // entries whose threshold lies below x
            for (int s = steps - 1; s >= 0; --s) {
                const int next = code + (1 << s);
                code = next <= a.n_values - 1 && x > threshold[next - 1] ? next : code;
            }
            return code;
        }
    };
    // The same for any quotient (see `limit`).
    auto below_the_last = [&](float x) __attribute__((always_inline)) -> bool {
        const float last = table[a.n_values - 1], before = table[max(a.n_values - 2, 0)];
        return x > last && a.n_values > 1 && fabsf(__fsub_rn(x, before)) <= fabsf(__fsub_rn(x, last));
    };
    auto value_of = [&](float x) __attribute__((always_inline)) -> float {
        if constexpr (ROUNDING == kInteger) {
            return nearest_grid_integer(x, a.minimum, a.maximum);
        } else if constexpr (ROUNDING == kFewValues) {
            float value = few_value[0];
#pragma unroll
            for (int k = 0; k < kFew - 1; ++k) value = x > few_threshold[k] ? few_value[k + 1] : value;
            return value;
        } else {
            return table[code_of(x)];
        }
    };

    for (int first = blockIdx.x * kTeams; first < a.total_groups; first += gridDim.x * kTeams) {
        const int wanted = first + threadIdx.x / TEAM;
        const int identifier = wanted < a.total_groups ? wanted : a.total_groups - 1;
        const int row = a.groups_per_row == 1 ? identifier : static_cast<int>(__umulhi(identifier, a.row_multiplier) >> a.row_shift);
        const int start = (identifier - row * a.groups_per_row) * a.group + 8 * lane_in_team;
        const size_t base = static_cast<size_t>(row) * a.width;
        float sample[TRIPS][8];
        if (a.aligned) {   // uniform: every lane's eight values are inside the row together
#pragma unroll
            for (int t = 0; t < TRIPS; ++t) {
                const int column = start + t * kSpan;
                const size_t from = base + (column < a.width ? column : 0);
                if (a.dtype == MK_F32) {
                    const float4 *source = reinterpret_cast<const float4 *>(static_cast<const float *>(a.value) + from);
                    const float4 low = source[0], high = source[1];
                    sample[t][0] = low.x; sample[t][1] = low.y; sample[t][2] = low.z; sample[t][3] = low.w;
                    sample[t][4] = high.x; sample[t][5] = high.y; sample[t][6] = high.z; sample[t][7] = high.w;
                } else {
                    const uint4 raw = *reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(a.value) + from);
                    const uint32_t word[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if (a.dtype == MK_F16) {
                            sample[t][2 * i] = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(word[i])));
                            sample[t][2 * i + 1] = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(word[i] >> 16)));
                        } else {
                            sample[t][2 * i] = __uint_as_float(word[i] << 16);
                            sample[t][2 * i + 1] = __uint_as_float(word[i] & 0xffff0000u);
                        }
                    }
                }
            }
        } else {
#pragma unroll
            for (int t = 0; t < TRIPS; ++t)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int column = start + t * kSpan + i;
                    sample[t][i] = mk_load_as_float(a.value, base + (column < a.width ? column : 0), a.dtype);
                }
        }
        const bool whole = start + (TRIPS - 1) * kSpan + 8 <= a.width;   // all of this lane's values are inside the row
        float low, high;
        auto range = [&](auto careful_) __attribute__((always_inline)) {
            constexpr bool kCareful = decltype(careful_)::value;
            low = __builtin_inff();
            high = -__builtin_inff();
#pragma unroll
            for (int t = 0; t < TRIPS; ++t)
#pragma unroll
                for (int i = 0; i < 8; i += 2) {
                    float v[2] = {sample[t][i], sample[t][i + 1]};
                    if constexpr (kCareful) {   // past the row: any of the lane's own values, or of the group's first
                        v[0] = start + t * kSpan + i < a.width ? v[0] : sample[0][0];
                        v[1] = start + t * kSpan + i + 1 < a.width ? v[1] : sample[0][0];
                    }
                    low = smallest(smallest(low, v[0]), v[1]);
                    high = largest(largest(high, v[0]), v[1]);
                }
            if constexpr (kCareful) {
                if (start >= a.width) {   // nothing of this lane is inside
                    low = __builtin_inff();
                    high = -__builtin_inff();
                }
            }
        };
        const bool all_whole = __all(whole);
        if (all_whole) range(std::integral_constant<bool, false>{});
        else range(std::integral_constant<bool, true>{});
        team_extrema<TEAM>(low, high, threadIdx.x & 63);
        const bool finite = low - low == 0.0f && high - high == 0.0f;
        float zero;
        float scale = mk_rounded_scale(range_scale(low, high, a.asym, a.reciprocal, a.minimum, zero), a.format);
        if (!finite || !(scale - scale == 0.0f)) {
            if (lane_in_team == 0) *a.flag = 1;
            scale = 1.0f;   // nothing below reads the weights as numbers any more: the caller raises
        }
        if constexpr (!SEARCH) {
            if (a.asym) zero = rounded_offset(zero, a.format);
        }
        if (a.asym) {
#pragma unroll
            for (int t = 0; t < TRIPS; ++t)
#pragma unroll
                for (int i = 0; i < 8; ++i) sample[t][i] = __fsub_rn(sample[t][i], zero);
        }
        if constexpr (SEARCH) {
            // `careful`: some lane's divisor or quotients are extreme, or some lane has columns past the row
            auto error_of = [&](float s, auto careful_) __attribute__((always_inline)) -> float {
                constexpr bool kCareful = decltype(careful_)::value;
                const float inverse = __fdiv_rn(1.0f, s);
                float partial[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) partial[i] = 0.0f;
#pragma unroll
                for (int t = 0; t < TRIPS; ++t)
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const float x = sample[t][i];
                        float q;
                        if constexpr (kCareful) q = __fdiv_rn(x, s);
                        else q = corrected_quotient(x, s, inverse);
                        float nearest = value_of(q);
                        if constexpr (kCareful && ROUNDING != kInteger) nearest = below_the_last(q) ? table[max(a.n_values - 2, 0)] : nearest;
                        float difference = __fsub_rn(__fmul_rn(nearest, s), x);
                        if constexpr (kCareful) difference = start + t * kSpan + i < a.width ? difference : 0.0f;
                        partial[i] = __fadd_rn(partial[i], __fmul_rn(difference, difference));
                    }
                float sum = __fadd_rn(__fadd_rn(__fadd_rn(partial[0], partial[1]), __fadd_rn(partial[2], partial[3])),
                                      __fadd_rn(__fadd_rn(partial[4], partial[5]), __fadd_rn(partial[6], partial[7])));
                if constexpr (TEAM >= 2) sum = __fadd_rn(sum, mk_matvec::lane_exchange<0>(sum, threadIdx.x & 63));
                if constexpr (TEAM >= 4) sum = __fadd_rn(sum, mk_matvec::lane_exchange<1>(sum, threadIdx.x & 63));
                if constexpr (TEAM >= 8) sum = __fadd_rn(sum, mk_matvec::lane_exchange<2>(sum, threadIdx.x & 63));
                return sum;
            };
            const float base_scale = scale;
            auto search = [&](auto careful_) __attribute__((always_inline)) {
                float best = error_of(base_scale, careful_);
                for (int c = 0; c < a.n_fractions; ++c) {
                    const float candidate = mk_rounded_scale(__fmul_rn(base_scale, fraction[c]), a.format);
                    const float error = error_of(candidate, careful_);
                    scale = error < best ? candidate : scale;
                    best = fminf(best, error);
                }
            };
            // The candidates whose error can be the least, from a first pass with contracted arithmetic: the distance to
            // the nearest multiple of the scale, or to the nearest scaled value, without the correctly rounded quotient.
            // Against the error of `error_of` a distance d of a value x may be off by a few 2^-24 (|x| + |d|), so a sum by
            // less than 2^-20 sqrt(E X) + 2^-40 X + 2^-18 E, X the sum of x^2; the margin below is at least four times that on
            // either side.  What remains, one or two candidates as a rule, goes through `error_of` in order.
            auto prune = [&](auto symmetric_) __attribute__((always_inline)) {
                constexpr bool kSymmetric = decltype(symmetric_)::value;
                auto over_team = [&](float sum) __attribute__((always_inline)) -> float {
                    sum += mk_matvec::lane_exchange<0>(sum, threadIdx.x & 63);
                    sum += mk_matvec::lane_exchange<1>(sum, threadIdx.x & 63);
                    return sum + mk_matvec::lane_exchange<2>(sum, threadIdx.x & 63);
                };
                auto estimated = [&](float s) __attribute__((always_inline)) -> float {
                    float sum[2] = {0.0f, 0.0f};
                    const float inverse = __builtin_amdgcn_rcpf(s);
                    float scaled[kFew];
                    if constexpr (ROUNDING == kFewValues) {
#pragma unroll
                        for (int k = 0; k < (kSymmetric ? kFew / 2 : kFew); ++k) scaled[k] = (kSymmetric ? magnitude[k] : few_value[k]) * s;
                    }
#pragma unroll
                    for (int t = 0; t < TRIPS; ++t)
#pragma unroll
                        for (int i = 0; i < 8; ++i) {
                            const float x = sample[t][i];
                            float distance;
                            if constexpr (ROUNDING == kInteger) {
                                distance = __builtin_fmaf(-nearest_grid_integer(x * inverse, a.minimum, a.maximum), s, x);
                            } else {
                                const float from = kSymmetric ? fabsf(x) : x;
                                distance = fabsf(from - scaled[0]);
#pragma unroll
                                for (int k = 1; k < (kSymmetric ? kFew / 2 : kFew); ++k) distance = fminf(distance, fabsf(from - scaled[k]));
                            }
                            sum[i & 1] = __builtin_fmaf(distance, distance, sum[i & 1]);
                        }
                    return over_team(sum[0] + sum[1]);
                };
                float *const estimates = estimate[threadIdx.x / TEAM];
                const float base_scale = scale, of_base = estimated(base_scale);
                float least = of_base;
                for (int c = 0; c < a.n_fractions; ++c) {
                    const float error = estimated(mk_rounded_scale(__fmul_rn(base_scale, fraction[c]), a.format));
                    if (lane_in_team == 0) estimates[c] = error;
                    least = fminf(least, error);
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                float squares = 0.0f;
#pragma unroll
                for (int t = 0; t < TRIPS; ++t)
#pragma unroll
                    for (int i = 0; i < 8; ++i) squares = __builtin_fmaf(sample[t][i], sample[t][i], squares);
                squares = over_team(squares);
                // (two roots: the product of the sums leaves the normal range for scales below 2^-32 or so)
                const float bound = least + (0x1p-14f * least + (0x1p-17f * (sqrtf(least) * sqrtf(squares)) + 0x1p-36f * squares));
                unsigned long long open = 0;
                for (int c = 0; c < a.n_fractions; ++c) open |= static_cast<unsigned long long>(estimates[c] <= bound) << c;
                float best = __builtin_inff();
                if (__any(of_base <= bound)) {
                    const float error = error_of(base_scale, std::integral_constant<bool, false>{});
                    best = of_base <= bound ? error : best;
                }
                while (__any(open != 0)) {   // at most n_fractions turns: each clears a bit of every team that has one
                    const float candidate = mk_rounded_scale(__fmul_rn(base_scale, fraction[open ? __builtin_ctzll(open) : 0]), a.format);
                    const float error = error_of(candidate, std::integral_constant<bool, false>{});
                    if (open && error < best) {
                        best = error;
                        scale = candidate;
                    }
                    open &= open - 1;
                }
                __builtin_amdgcn_wave_barrier();   // the estimates have been read
            };
            // (2^40: no square of the first pass leaves the normal range, nor 2^-36 of a sum of them)
            const float smallest_scale = fminf(base_scale, mk_rounded_scale(__fmul_rn(base_scale, least_fraction), a.format));
            const bool within = all_whole && ordinary_fractions && __all((a.asym ? high - zero : high) <= limit * smallest_scale);
            const bool moderate = kPruned && within && __all(base_scale > 0x1p-40f && base_scale < 0x1p40f);
            if constexpr (kPruned) {
                if (moderate) {
                    if constexpr (ROUNDING == kFewValues) {
                        if (symmetric) prune(std::integral_constant<bool, true>{});
                        else prune(std::integral_constant<bool, false>{});
                    } else {
                        prune(std::integral_constant<bool, false>{});
                    }
                }
            }
            // candidates are fractions of the base (or the smallest value of the storage format)
            if (moderate) {
            } else if (within && __all(base_scale > 0x1p-90f && base_scale < 0x1p90f))
                search(std::integral_constant<bool, false>{});
            else
                search(std::integral_constant<bool, true>{});
            if (a.asym) {
                // the offset is stored after the search: undo it in the values, exactly as the separate passes see them
                const float stored = rounded_offset(zero, a.format);
#pragma unroll
                for (int t = 0; t < TRIPS; ++t)
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const int column = start + t * kSpan + i;
                        sample[t][i] = __fsub_rn(mk_load_as_float(a.value, base + (column < a.width ? column : 0), a.dtype), stored);
                    }
                zero = stored;
            }
        }
        uint32_t packed[TRIPS][2];
        auto encode = [&](auto careful_) __attribute__((always_inline)) {
            const float inverse = __fdiv_rn(1.0f, scale);
#pragma unroll
            for (int t = 0; t < TRIPS; ++t) {
                packed[t][0] = packed[t][1] = 0;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    float q;
                    if constexpr (decltype(careful_)::value) q = __fdiv_rn(sample[t][i], scale);
                    else q = corrected_quotient(sample[t][i], scale, inverse);
                    if constexpr (ROUNDING == kInteger)   // exact: the value is an integer between 0 and 255
                        packed[t][i / 4] = __builtin_amdgcn_cvt_pk_u8_f32(
                            __fsub_rn(nearest_grid_integer(q, a.minimum, a.maximum), a.minimum), i % 4, packed[t][i / 4]);
                    else
                        packed[t][i / 4] |= static_cast<uint32_t>(decltype(careful_)::value && below_the_last(q) ? a.n_values - 2 : code_of(q)) << (8 * (i % 4));
                }
            }
        };
        if (__all(scale > 0x1p-100f && scale < 0x1p100f && (a.asym ? high - zero : high) <= limit * scale))
            encode(std::integral_constant<bool, false>{});
        else encode(std::integral_constant<bool, true>{});
        if (wanted >= a.total_groups) continue;
        if (lane_in_team == 0) {
            a.scales[identifier] = scale;
            if (a.zeros) a.zeros[identifier] = zero;
        }
        if (a.aligned) {
#pragma unroll
            for (int t = 0; t < TRIPS; ++t) {
                const int column = start + t * kSpan;
                if (column < a.width) *reinterpret_cast<uint2 *>(a.codes + base + column) = make_uint2(packed[t][0], packed[t][1]);
            }
        } else {
#pragma unroll
            for (int t = 0; t < TRIPS; ++t)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int column = start + t * kSpan + i;
                    if (column < a.width) a.codes[base + column] = static_cast<uint8_t>(packed[t][i / 4] >> (8 * (i % 4)));
                }
        }
    }
}

template <int ROUNDING, bool SEARCH, int TEAM, int TRIPS>
void launch_round(const RoundArgs &a, hipStream_t stream) {
    // eight workgroups of a CU's worth at most, so that the thresholds of a table are worked out a few thousand times
    int blocks = mk_cdiv(a.total_groups, kThreads / TEAM);
    if (blocks > 256 * 8) blocks = 256 * 8;
    hipLaunchKernelGGL((round_groups_kernel<ROUNDING, SEARCH, TEAM, TRIPS>), dim3(blocks), dim3(kThreads), 0, stream, a);
}

template <int ROUNDING, bool SEARCH>
void dispatch_group(const RoundArgs &a, hipStream_t stream) {
    switch (a.group) {
        case 8: launch_round<ROUNDING, SEARCH, 1, 1>(a, stream); break;
        case 16: launch_round<ROUNDING, SEARCH, 2, 1>(a, stream); break;
        case 32: launch_round<ROUNDING, SEARCH, 4, 1>(a, stream); break;
        case 64: launch_round<ROUNDING, SEARCH, 8, 1>(a, stream); break;
        case 128: launch_round<ROUNDING, SEARCH, 8, 2>(a, stream); break;
        default: launch_round<ROUNDING, SEARCH, 8, 4>(a, stream); break;
    }
}

}  // namespace

extern "C" int mk_round_matrix(const void *value, int dtype, const float *values, int n_values, const float *fractions,
                               int n_fractions, float *scales, float *zeros, uint8_t *codes, int *flag, int rows,
                               int width, int group, int asym, int integer, float minimum, float maximum,
                               float reciprocal, int scale_format, void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MK_REQUIRE(value && scales && codes && flag && (!asym || zeros), MK_ERR_INVALID, "mk_round_matrix: null tensor pointer");
    MK_REQUIRE(rows >= 1 && width >= 1, MK_ERR_INVALID, "mk_round_matrix: sizes must be positive");
    MK_REQUIRE(mk_dtype_valid(dtype), MK_ERR_INVALID, "mk_round_matrix: unknown dtype code");
    MK_REQUIRE(group >= 8 && group <= 256 && (group & (group - 1)) == 0, MK_ERR_UNSUPPORTED,
               "mk_round_matrix: groups of 8, 16, 32, 64, 128 or 256 columns, not %d", group);
    MK_REQUIRE(scale_format >= 0 && scale_format <= 4, MK_ERR_INVALID, "mk_round_matrix: unknown scale format code");
    MK_REQUIRE(n_fractions >= 0 && n_fractions <= 64 && (n_fractions == 0 || fractions), MK_ERR_INVALID,
               "mk_round_matrix: at most 64 candidate fractions");
    if (integer)
        MK_REQUIRE(maximum >= minimum && maximum - minimum <= 255.0f, MK_ERR_INVALID,
                   "mk_round_matrix: integer grid must span at most 256 codes");
    else
        MK_REQUIRE(values && n_values >= 1 && n_values <= kMaxTable, MK_ERR_INVALID,
                   "mk_round_matrix: a value table of 1..256 entries is required");
    const int groups_per_row = mk_cdiv(width, group);
    MK_REQUIRE(static_cast<long long>(rows) * groups_per_row < (1ll << 31) - 256 * 8 * kThreads, MK_ERR_INVALID,
               "mk_round_matrix: too many scale groups");
    RoundArgs a{};
    a.value = value; a.values = values; a.fractions = fractions; a.scales = scales; a.zeros = asym ? zeros : nullptr;
    a.codes = codes; a.flag = flag; a.rows = rows; a.width = width; a.group = group; a.groups_per_row = groups_per_row;
    a.total_groups = rows * groups_per_row; a.dtype = dtype; a.n_values = integer ? 1 : n_values;
    a.n_fractions = n_fractions; a.format = scale_format; a.asym = asym;
    a.aligned = width % 8 == 0 && (reinterpret_cast<uintptr_t>(value) & 15u) == 0 && (reinterpret_cast<uintptr_t>(codes) & 7u) == 0;
    a.reciprocal = reciprocal; a.minimum = minimum; a.maximum = maximum;
    if (groups_per_row > 1) {   // exact for identifiers below 2^31: the multiplier exceeds 2^(32 + shift) / d by less than one
        int bits = 0;
        while ((1 << bits) < groups_per_row) ++bits;
        a.row_shift = bits - 1;
        a.row_multiplier = static_cast<uint32_t>(((1ull << (31 + bits)) + groups_per_row - 1) / groups_per_row);
    }
    const int rounding = integer ? kInteger : n_values <= kFew ? kFewValues : kTable;
    const bool search = n_fractions > 0;
    if (rounding == kInteger) search ? dispatch_group<kInteger, true>(a, stream) : dispatch_group<kInteger, false>(a, stream);
    else if (rounding == kFewValues) search ? dispatch_group<kFewValues, true>(a, stream) : dispatch_group<kFewValues, false>(a, stream);
    else search ? dispatch_group<kTable, true>(a, stream) : dispatch_group<kTable, false>(a, stream);
    MK_LAUNCH_CHECK("mk_round_matrix");
    return MK_OK;
}
