// Packed weight x several rows of activations on the matrix cores of gfx950: kernel template.
//
// y[m, n] = sum_k dequant(code[n, k]) * x[m, k] (+ bias[n]) for nine rows of x and more; fp16 or bf16 x, codes of 2, 3,
// 4 or 8 bits, fp16 or bf16 scales, scale groups of 64 columns, of a multiple of 128, or of the whole row.
//
// Codes go straight from HBM to the matrix cores.  v_mfma_f32_16x16x32 takes a 16 x 32 piece of the weight as eight
// values per lane; lane (n, q) loads the quarter of row n's scale group that the instructions of the group give to
// lanes (., q), so a load is 16 rows of a whole group, and no code moves between lanes.  Codes become small exact
// numbers of x's type (arithmetic for uniform 4- and 8-bit grids, an LDS table of several values per lookup
// otherwise); the group's products are summed first and scaled in fp32 afterwards:
//     y += s * sum(operand * x) + b * sum(x),   b = s * (grid minimum - operand of code 0) + zero,
// with sum(x) from a multiplication by ones where b is not zero.
//
// Table values that x's type cannot hold (NF4, fitted codebooks) are two operands (SPLIT), the value rounded and what the
// rounding left of it: all weights of one code share its error, which adds up over x with a mean where errors of single weights
// cancel (NF4, 14336 columns of relu(normal) x: 3.1e-2 of y in bf16 and 2.1e-3 in fp16 with the rounded value alone, 2.8e-3
// and 3.4e-4 with a decoded weight rounded as a whole, 1.7e-3 and 2.1e-4 -- the rounding of y -- with both).  A table is
// multiplied by a power of two that puts its largest value at 2^14, the scales by the inverse, so that in fp16 neither part
// runs out of range: the two hold a value to 2^-23 of it, or 2^-39 of the largest; in bf16 to 2^-17 of it.  Without SPLIT every
// wavefront makes sure that x's type holds its table; outputs over one that it does not hold come from plain_outputs.
//
// A workgroup owns 16 * RT rows of the weight and 16 * MT rows of x; its wavefronts take the row's steps of 128 columns
// in turn, so a step's activations are read by one wavefront only.  They pass through a stretch of LDS of its own (no
// barriers): loaded as rows, read back as operands, 16-byte pieces swizzled by row so that neither side has
// bank conflicts.  The wavefronts' sums meet in LDS at the end, in a fixed order.
//
// INT4 g128 with offsets and bf16 x, us per launch over weights that no cache holds (decoding the weight and a library
// product before): 4096 x 14336, 16 / 32 / 64 / 128 rows of x 15.5 / 20.1 / 26.5 / 37.6 (54 / 55 / 67 / 90);
// 14336 x 4096 12.2 / 14.9 / 25.2 / 44.0 (53 / 55 / 57 / 60); 896 x 896 3.7 / 3.6 / 3.7 / 4.4 (9 to 11).
// Bound by instruction fetches and latency on small layers (a launch runs its code a few times: every loop that was
// unrolled for prefetching made it slower), by the LDS traffic of the activations from 64 rows of x on, and by
// codes arriving and being multiplied in turn rather than at the same time in between (the loads alone take 8 us of
// 14336 x 4096's 12.2, the arithmetic alone 8).
#pragma once

#include <atomic>
#include <type_traits>

#include "mk_common.h"

namespace mk_matmul {

constexpr int kStep = 128;        // columns per step
constexpr int kMaxWaves = 8;

enum Format { kUniform4, kTable4, kTable3, kTable2, kUniform8 };

struct MatmulArgs {
    const void *x;
    const uint8_t *packed;
    const uint16_t *scales;
    const uint16_t *zeros;    // or null
    const float *values;
    const void *bias;         // or null
    void *y;
    int samples, rows, width, groups, group;
    int steps;                // ceil(width / 128)
    int steps_per_group;      // SUB == 1: steps that share a scale
    uint32_t group_multiplier;   // step / steps_per_group = umulhi(step, multiplier) >> shift, where that is above one
    int group_shift;
    int n_values, uniform, scale_bf16, bias_dtype, need_sums;
    int whole_quads;          // four adjacent outputs of a row of y are one aligned store
    float grid_min, grid_step;
};

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));

template <int XT>
__device__ __forceinline__ f32x4 mfma(mk_u32x4 a, mk_u32x4 b, f32x4 c) {
    if constexpr (XT == MK_F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a), __builtin_bit_cast(h8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, b), c, 0, 0, 0);
}

template <int XT>
__device__ __forceinline__ uint32_t pair_of(float low, float high) {
    if constexpr (XT == MK_F16)
        return __builtin_bit_cast(uint32_t, mk_h2{static_cast<_Float16>(low), static_cast<_Float16>(high)});
    else
        return __builtin_bit_cast(uint32_t, mk_bf2{static_cast<__bf16>(low), static_cast<__bf16>(high)});
}

// What a format is made of: the dwords a lane holds of CH consecutive codes, and the operand of codes 8 j ... 8 j + 7.
// Behind the kTableWords dwords of a table of values there are as many of what their rounding left (SPLIT).
template <int FORMAT, int XT, int CH>
struct Codes;

// Four-bit codes of a uniform grid: one of a dword's four nibble pairs is where the mantissa of a power of two has its
// units (128 + code in bf16, 64 + code in fp16), the others are shifted there.  The eight values of a dword come in
// the order 0, 4, 1, 5, 2, 6, 3, 7.
template <int XT, int CH>
struct Codes<kUniform4, XT, CH> {
    static constexpr int kBits = 4, kWords = CH / 8;
    static constexpr bool kInterleaved = true;
    static constexpr float kOffset = XT == MK_F16 ? 64.0f : 128.0f;   // operand = code + offset
    static constexpr int kTableWords = 0;
    uint32_t mask = XT == MK_F16 ? 0x00f000f0u : 0x000f000fu, base = XT == MK_F16 ? 0x54005400u : 0x43004300u;
    // (in registers, one of each kind: as literals they would not share an instruction)
    __device__ __forceinline__ Codes() { asm("" : "+s"(mask)); asm("" : "+v"(base)); }
    __device__ __forceinline__ mk_u32x4 operand(const uint32_t (&raw)[kWords], int j, const uint32_t *, uint32_t) const {
        const uint32_t w = raw[j];
        if constexpr (XT == MK_F16)
            return {((w << 4) & mask) | base, (w & mask) | base, ((w >> 4) & mask) | base, ((w >> 8) & mask) | base};
        else
            return {(w & mask) | base, ((w >> 4) & mask) | base, ((w >> 8) & mask) | base, ((w >> 12) & mask) | base};
    }
};

// Eight-bit codes of a uniform grid; the operand is code - 128 in fp16 and the code itself in bf16 (both exact).
template <int XT, int CH>
struct Codes<kUniform8, XT, CH> {
    static constexpr int kBits = 8, kWords = CH / 4;
    static constexpr bool kInterleaved = false;
    static constexpr float kOffset = XT == MK_F16 ? -128.0f : 0.0f;
    static constexpr int kTableWords = 0;
    __device__ __forceinline__ mk_u32x4 operand(const uint32_t (&raw)[kWords], int j, const uint32_t *, uint32_t) const {
        mk_u32x4 out;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t w = raw[2 * j + h];
            if constexpr (XT == MK_F16) {
                const mk_h2 bias = {static_cast<_Float16>(-1152.0f), static_cast<_Float16>(-1152.0f)};
                const mk_h2 low = __builtin_bit_cast(mk_h2, __builtin_amdgcn_perm(0x64646464u, w, 0x07010700u)) + bias;
                const mk_h2 high = __builtin_bit_cast(mk_h2, __builtin_amdgcn_perm(0x64646464u, w, 0x07030702u)) + bias;
                out[2 * h] = __builtin_bit_cast(uint32_t, low);
                out[2 * h + 1] = __builtin_bit_cast(uint32_t, high);
            } else {
                out[2 * h] = pair_of<XT>(static_cast<float>(w & 255u), static_cast<float>((w >> 8) & 255u));
                out[2 * h + 1] = pair_of<XT>(static_cast<float>((w >> 16) & 255u), static_cast<float>(w >> 24));
            }
        }
        return out;
    }
};

// Four-bit codes of any table: a byte is two codes, an entry of the LDS table their two values.
template <int XT, int CH>
struct Codes<kTable4, XT, CH> {
    static constexpr int kBits = 4, kWords = CH / 8;
    static constexpr bool kInterleaved = false;
    static constexpr float kOffset = 0.0f;
    static constexpr int kTableWords = 256;
    __device__ __forceinline__ mk_u32x4 operand(const uint32_t (&raw)[kWords], int j, const uint32_t *table, uint32_t) const {
        const uint32_t w = raw[j];
        return {table[w & 255u], table[(w >> 8) & 255u], table[(w >> 16) & 255u], table[w >> 24]};
    }
};

// Three-bit codes: six bits are two codes.  A lane's 32 codes are three dwords, its 16 codes 48 bits of the two dwords
// around them (`shift`: 0 or 16).
template <int XT, int CH>
struct Codes<kTable3, XT, CH> {
    static constexpr int kBits = 3, kWords = CH == 32 ? 3 : 2;
    static constexpr bool kInterleaved = false;
    static constexpr float kOffset = 0.0f;
    static constexpr int kTableWords = 64;
    __device__ __forceinline__ mk_u32x4 operand(const uint32_t (&raw)[kWords], int j, const uint32_t *table, uint32_t shift) const {
        uint32_t w;   // bits 24 j ... 24 j + 23 of the lane's codes
        if constexpr (CH == 32) {
            if (j == 0) w = raw[0];
            else if (j == 1) w = static_cast<uint32_t>((static_cast<uint64_t>(raw[1]) << 32 | raw[0]) >> 24);
            else if (j == 2) w = static_cast<uint32_t>((static_cast<uint64_t>(raw[2]) << 32 | raw[1]) >> 16);
            else w = raw[2] >> 8;
        } else {
            const uint64_t all = (static_cast<uint64_t>(raw[1]) << 32 | raw[0]) >> shift;
            w = static_cast<uint32_t>(all >> (24 * j));
        }
        return {table[w & 63u], table[(w >> 6) & 63u], table[(w >> 12) & 63u], table[(w >> 18) & 63u]};
    }
};

// Two-bit codes: a byte is four codes, two dwords of the table.
template <int XT, int CH>
struct Codes<kTable2, XT, CH> {
    static constexpr int kBits = 2, kWords = CH / 16;
    static constexpr bool kInterleaved = false;
    static constexpr float kOffset = 0.0f;
    static constexpr int kTableWords = 512;
    __device__ __forceinline__ mk_u32x4 operand(const uint32_t (&raw)[kWords], int j, const uint32_t *table, uint32_t) const {
        const uint32_t w = raw[j / 2] >> (16 * (j & 1));
        const mk_u32x2 low = reinterpret_cast<const mk_u32x2 *>(table)[w & 255u];
        const mk_u32x2 high = reinterpret_cast<const mk_u32x2 *>(table)[(w >> 8) & 255u];
        return {low[0], low[1], high[0], high[1]};
    }
};

__device__ __forceinline__ float table_value(const MatmulArgs &a, int code) {
    return a.uniform ? a.grid_min + static_cast<float>(code) * a.grid_step : a.values[code < a.n_values ? code : a.n_values - 1];
}

// Outputs of a tile by their definition, for sums that are not finite (and for tables, see above): an infinite activation times operand and offset gives
// infinities of both signs where its product with the decoded weight has one.  Lane (c, q) of the wavefront holds the
// sums of rows row + 4 q ... + 3 with sample `sample` + c; `open`: the lanes whose four are wanted.
//
// The wavefront works on one sample at a time, each lane on eight adjacent columns of every 512.  One look at the
// activations comes first: a NaN makes every output one, and beside infinities finite terms do not matter (pieces of 512
// columns without one are passed over).  32 rows of x, one of them with a NaN / an infinity, 4096 x 14336 INT4: 29 / 52 us (19
// without; 19.3 ms with a thread to an output).
template <int FORMAT, int XT>
__device__ __forceinline__ void plain_outputs(const MatmulArgs &a, unsigned long long open, int row, int sample, const float *biases,
                                              f32x4 &value, int lane) {
    constexpr int kBits = Codes<FORMAT, XT, 32>::kBits;
    constexpr uint32_t kInfinite = XT == MK_F16 ? 0x7c00u : 0x7f80u;
    const int side_type = a.scale_bf16 ? MK_BF16 : MK_F16;
    const size_t row_bytes = static_cast<size_t>(a.width / 8) * kBits;
#pragma unroll 1
    while (open) {   // uniform: each turn clears the bits of one sample
        const int column = __builtin_ctzll(open) & 15;
        const unsigned long long wanted = open & (0x0001000100010001ull << column);
        open &= ~wanted;
        const uint16_t *x = static_cast<const uint16_t *>(a.x) + static_cast<size_t>(sample + column) * a.width;
        bool undefined = false;
        unsigned long long pieces = 0;   // of 512 columns with an infinity; the last bit stands for all further ones too
#pragma unroll 1
        for (int four = 0; four < a.width && !undefined; four += 2048) {   // (pieces past the row: its last columns again)
            bool not_a_number = false;
#pragma unroll
            for (int first = four; first < four + 2048; first += 512) {
                bool here = false;
                const mk_u32x4 eight = *reinterpret_cast<const mk_u32x4 *>(x + min(first + 8 * lane, a.width - 8));   // (16-byte aligned)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const uint32_t magnitude = eight[i] >> (16 * h) & 0x7fffu;
                        not_a_number |= magnitude > kInfinite;
                        here |= magnitude == kInfinite;
                    }
                if (__any(here)) pieces |= 1ull << min(first >> 9, 63);
            }
            undefined = __any(not_a_number);
        }
        const bool infinite = pieces != 0;
        if (!infinite) pieces = ~0ull;   // finite activations, whose products overflowed
#pragma unroll 1
        for (int q = 0; q < 4; ++q) {
            const int owner = column + 16 * q;
            if (!(wanted >> owner & 1)) continue;   // uniform
            f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
            if (undefined) {
                sum = f32x4{__builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""), __builtin_nanf("")};
            } else {
#pragma unroll 1
                for (int first = 0; first < a.width; first += 512) {
                    const int k = first + 8 * lane;
                    if (!(pieces >> min(first >> 9, 63) & 1) || k >= a.width) continue;
                    const int group = a.group >= a.width ? 0 : k / a.group;   // (whole groups of eight columns)
                    uint32_t matters = 0;
#pragma unroll
                    for (int c = 0; c < 8; ++c) matters |= !infinite || (x[k + c] & 0x7fffu) == kInfinite ? 1u << c : 0u;
                    if (!matters) continue;
#pragma unroll 1
                    for (int i = 0; i < 4; ++i) {
                        const size_t at = min(row + 4 * q + i, a.rows - 1);
                        const uint8_t *source = a.packed + at * row_bytes + static_cast<size_t>(k / 8) * kBits;
                        uint64_t codes = 0;
#pragma unroll
                        for (int b = 0; b < kBits; ++b) codes |= static_cast<uint64_t>(source[b]) << (8 * b);
                        const float scale = mk_load_as_float(a.scales, at * a.groups + group, side_type);
                        const float zero = a.zeros ? mk_load_as_float(a.zeros, at * a.groups + group, side_type) : 0.0f;
                        float part = 0.0f;
#pragma unroll 1
                        for (int c = 0; c < 8; ++c) {
                            if (!(matters >> c & 1)) continue;
                            const int code = static_cast<int>(codes >> (kBits * c) & ((1u << kBits) - 1));
                            const float weight = __fadd_rn(__fmul_rn(table_value(a, code), scale), zero);   // as it is decoded
                            part = __builtin_fmaf(weight, mk_load_as_float(x, k + c, XT), part);
                        }
#pragma unroll
                        for (int r = 0; r < 4; ++r) sum[r] += r == i ? part : 0.0f;
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) sum[r] = mk_segment_sum<64>(sum[r]);
            }
            if (lane == owner) {
#pragma unroll
                for (int r = 0; r < 4; ++r) value[r] = sum[r] + biases[4 * q + r];
            }
        }
    }
}

// Dynamic LDS of a workgroup, in bytes; the sums of the wavefronts reuse the activations' stretch.
template <int FORMAT, int RT, int MT, bool SPLIT>
constexpr size_t lds_bytes(int waves, int scale_groups, bool sums_needed) {
    constexpr int table = Codes<FORMAT, MK_F16, 32>::kTableWords * (SPLIT ? 8 : 4);
    const size_t stage = static_cast<size_t>(waves) * MT * 16 * 256;
    const size_t sums = static_cast<size_t>(waves) * RT * MT * 1024;
    return (stage > sums ? stage : sums) + table + 64 * RT + static_cast<size_t>(scale_groups) * 16 * RT * 4 * (sums_needed ? 2 : 1);
}

template <int FORMAT, int XT, int RT, int MT, int SUB, bool SUMS, bool SPLIT>
__global__ void __launch_bounds__(64 * kMaxWaves) packed_matmul_kernel(const MatmulArgs a) {
    constexpr int kChunk = 32 / SUB;          // codes of a lane per scale group
    constexpr int kProducts = kChunk / 8;     // matrix instructions per scale group
    using C = Codes<FORMAT, XT, kChunk>;
    constexpr int kWords = C::kWords;
    constexpr int kRows = 16 * RT;
    constexpr int kPieces = MT * 4;           // 16-byte pieces of activations per lane and step

    extern __shared__ mk_u32x4 lds[];
    const int lane = threadIdx.x & 63, waves = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // steps and their offsets stay scalar
    const int column = lane & 15, quarter = lane >> 4;
    const int first_row = blockIdx.x * kRows, first_sample = blockIdx.y * (16 * MT);
    const size_t stage_bytes = static_cast<size_t>(waves) * MT * 16 * 256, sum_bytes = static_cast<size_t>(waves) * RT * MT * 1024;
    mk_u32x4 *stage = lds + wave * (MT * 16 * 16);
    uint32_t *table = reinterpret_cast<uint32_t *>(reinterpret_cast<char *>(lds) + (stage_bytes > sum_bytes ? stage_bytes : sum_bytes));
    float *biases = reinterpret_cast<float *>(table + (SPLIT ? 2 : 1) * C::kTableWords);
    float *scales = biases + kRows;

    // -- loads of a step: the codes of this lane's rows, the pieces of activations this lane passes on ---------------
    // (a uniform base, 32-bit offsets: a workgroup's rows span less than 4 GB, the activations too)
    const int row_bytes = a.width / 8 * C::kBits;
    const uint8_t *codes = a.packed + static_cast<size_t>(first_row) * row_bytes;
    unsigned row_offset[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
        row_offset[rt] = static_cast<unsigned>(min(rt * 16 + column, a.rows - 1 - first_row)) * static_cast<unsigned>(row_bytes);
    const int quarter_bytes = quarter * (kChunk / 8 * C::kBits) & ~3;
    const int last_bytes = row_bytes - 4 * kWords;   // past the row: any codes, the activations there are zero
    auto load_codes = [&](uint32_t (&raw)[RT][SUB][kWords], int step) __attribute__((always_inline)) {
#pragma unroll
        for (int sub = 0; sub < SUB; ++sub) {
            const int in_row = min((step * kStep + sub * (kStep / SUB)) / 8 * C::kBits + quarter_bytes, last_bytes);
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const uint32_t *source = reinterpret_cast<const uint32_t *>(codes + (row_offset[rt] + static_cast<unsigned>(in_row)));
                if constexpr (kWords == 8) {
                    const mk_u32x4 low = __builtin_nontemporal_load(reinterpret_cast<const mk_u32x4 *>(source));
                    const mk_u32x4 high = __builtin_nontemporal_load(reinterpret_cast<const mk_u32x4 *>(source) + 1);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        raw[rt][sub][i] = low[i];
                        raw[rt][sub][4 + i] = high[i];
                    }
                } else if constexpr (kWords == 4) {
                    const mk_u32x4 loaded = __builtin_nontemporal_load(reinterpret_cast<const mk_u32x4 *>(source));
#pragma unroll
                    for (int i = 0; i < 4; ++i) raw[rt][sub][i] = loaded[i];
                } else if constexpr (kWords == 2 && FORMAT != kTable3) {
                    const mk_u32x2 loaded = __builtin_nontemporal_load(reinterpret_cast<const mk_u32x2 *>(source));
                    raw[rt][sub][0] = loaded[0];
                    raw[rt][sub][1] = loaded[1];
                } else {
#pragma unroll
                    for (int i = 0; i < kWords; ++i) raw[rt][sub][i] = __builtin_nontemporal_load(source + i);
                }
            }
        }
    };
    const char *x = static_cast<const char *>(a.x);
    unsigned sample_offset[kPieces];
#pragma unroll
    for (int p = 0; p < kPieces; ++p)
        sample_offset[p] = static_cast<unsigned>(min(first_sample + 4 * p + quarter, a.samples - 1)) * static_cast<unsigned>(2 * a.width);
    auto load_activations = [&](mk_u32x4 (&piece)[kPieces], int step) __attribute__((always_inline)) {
        const int in_row = min(step * (2 * kStep) + 16 * column, 2 * a.width - 16);
#pragma unroll
        for (int p = 0; p < kPieces; ++p)
            piece[p] = *reinterpret_cast<const mk_u32x4 *>(x + (sample_offset[p] + static_cast<unsigned>(in_row)));
    };
    auto pass_activations = [&](mk_u32x4 (&piece)[kPieces], int step) __attribute__((always_inline)) {
        if (__builtin_expect(step * kStep + kStep > a.width, 0)) {   // uniform: the row ends inside this step
            const bool inside = step * kStep + 8 * column < a.width;
#pragma unroll
            for (int p = 0; p < kPieces; ++p) piece[p] = inside ? piece[p] : mk_u32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int p = 0; p < kPieces; ++p) {
            const int row = 4 * p + quarter;
            mk_u32x4 value = piece[p];
            if constexpr (C::kInterleaved)
                value = mk_u32x4{__builtin_amdgcn_perm(value[2], value[0], 0x05040100u), __builtin_amdgcn_perm(value[2], value[0], 0x07060302u),
                                 __builtin_amdgcn_perm(value[3], value[1], 0x05040100u), __builtin_amdgcn_perm(value[3], value[1], 0x07060302u)};
            stage[row * 16 + (column ^ (row & 15))] = value;
        }
    };

    uint32_t raw[RT][SUB][kWords];
    mk_u32x4 piece[kPieces];
    load_activations(piece, wave);
    load_codes(raw, wave);

    // -- tables and scales into LDS, once ---------------------------------------------------------------------------
    bool held = true;            // uniform: x's type holds the table, or there is a second operand
    float table_inverse = 1.0f;  // the inverse of the table's power of two, for the scales
    if constexpr (C::kTableWords > 0) {
        constexpr int kCodes = 1 << C::kBits;
        float largest = 0.0f;
#pragma unroll
        for (int code = 0; code < kCodes; ++code) largest = fmaxf(largest, fabsf(table_value(a, code)));
        int exponent = (__float_as_int(largest) >> 23) - (127 + 14);
        exponent = largest > 0.0f && largest < __builtin_inff() ? min(max(exponent, -100), 100) : 0;
        table_inverse = __int_as_float((127 + exponent) << 23);
        const float factor = __int_as_float((127 - exponent) << 23);
        auto rounded = [&](float value) __attribute__((always_inline)) -> float {
            if constexpr (XT == MK_F16) return static_cast<float>(static_cast<_Float16>(value));
            else return static_cast<float>(static_cast<__bf16>(value));
        };
        if constexpr (!SPLIT) {
            const float own = table_value(a, lane % kCodes) * factor;
            held = __all(rounded(own) == own);
        }
        for (int i = threadIdx.x; i < C::kTableWords; i += blockDim.x) {
            const int codes = FORMAT == kTable2 ? (i >> 1) >> (4 * (i & 1)) : i;
            const float low = table_value(a, codes & (kCodes - 1)) * factor;
            const float high = table_value(a, (codes >> C::kBits) & (kCodes - 1)) * factor;
            table[i] = pair_of<XT>(low, high);
            if constexpr (SPLIT) table[C::kTableWords + i] = pair_of<XT>(low - rounded(low), high - rounded(high));
        }
    }
    float *offsets = scales + a.groups * kRows;
    {
        // 64 * waves / kRows threads to a row, four loads of a thread in flight.  Branch-free: past the last group its
        // value is written again, and masks stand for the choices that are the same for every thread.
        constexpr bool kArithmetic = C::kTableWords == 0;
        constexpr int kBatch = 4;
        uint32_t bf16_mask = a.scale_bf16 ? ~0u : 0u, zero_mask = a.zeros ? 0xffffu : 0u;
        asm("" : "+v"(bf16_mask), "+v"(zero_mask));
        auto side_value = [&](uint32_t bits) __attribute__((always_inline)) -> float {
            const uint32_t half = __float_as_uint(static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(bits))));
            return __uint_as_float((bits << 16 & bf16_mask) | (half & ~bf16_mask));
        };
        const int per_row = blockDim.x / kRows, local_row = threadIdx.x / per_row, lane_in_row = threadIdx.x - local_row * per_row;
        const size_t base = static_cast<size_t>(min(first_row + local_row, a.rows - 1)) * a.groups;
        const uint16_t *stored_scales = a.scales + base, *stored_zeros = (a.zeros ? a.zeros : a.scales) + base;
#pragma unroll 1
        for (int first = lane_in_row; first < a.groups; first += kBatch * per_row) {
            uint32_t stored[kBatch], zero[kBatch];
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                const int group = min(first + i * per_row, a.groups - 1);
                stored[i] = stored_scales[group];
                if constexpr (SUMS) zero[i] = stored_zeros[group];
            }
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                const int slot = min(first + i * per_row, a.groups - 1) * kRows + local_row;
                const float scale = side_value(stored[i]);
                scales[slot] = kArithmetic ? scale * a.grid_step : scale * table_inverse;
                if constexpr (SUMS) {
                    const float offset = side_value(zero[i] & zero_mask);
                    offsets[slot] = kArithmetic ? __builtin_fmaf(scale, a.grid_min - C::kOffset * a.grid_step, offset) : offset;
                }
            }
        }
        if (threadIdx.x < kRows) {
            const int row = min(first_row + static_cast<int>(threadIdx.x), a.rows - 1);
            biases[threadIdx.x] = a.bias ? mk_load_as_float(a.bias, row, a.bias_dtype) : 0.0f;
        }
    }
    __syncthreads();

    f32x4 total[RT][MT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) total[rt][mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const uint32_t one = XT == MK_F16 ? 0x3c003c00u : 0x3f803f80u;
    const mk_u32x4 ones = {one, one, one, one};
    const C format;

    auto multiply = [&](const uint32_t (&raw)[RT][SUB][kWords], int step) __attribute__((always_inline)) {
#pragma unroll
        for (int sub = 0; sub < SUB; ++sub) {
            f32x4 product[RT][MT], sum[MT];
            const uint32_t shift = FORMAT == kTable3 && kChunk == 16 ? (quarter & 1) * 16u : 0u;
#pragma unroll
            for (int j = 0; j < kProducts; ++j) {
                mk_u32x4 activations[MT];
                const int chunk = sub * (16 / SUB) + quarter * kProducts + j;
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) activations[mt] = stage[(mt * 16 + column) * 16 + (chunk ^ column)];
                const f32x4 none = {0.0f, 0.0f, 0.0f, 0.0f};
                if constexpr (SUMS) {
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) sum[mt] = mfma<XT>(ones, activations[mt], j == 0 ? none : sum[mt]);
                }
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    const mk_u32x4 weights = format.operand(raw[rt][sub], j, table, shift);
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
                        product[rt][mt] = mfma<XT>(weights, activations[mt], j == 0 ? none : product[rt][mt]);
                    if constexpr (SPLIT) {
                        const mk_u32x4 rest = format.operand(raw[rt][sub], j, table + C::kTableWords, shift);
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) product[rt][mt] = mfma<XT>(rest, activations[mt], product[rt][mt]);
                    }
                }
            }
            int group = step * SUB + sub;
            if constexpr (SUB == 1) {
                if (a.steps_per_group > 1) group = static_cast<int>(__umulhi(step, a.group_multiplier) >> a.group_shift);
            } else {
                group = min(group, a.groups - 1);   // past the row: products of zeros
            }
            const int slot = group * kRows + 4 * quarter;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const f32x4 scale = *reinterpret_cast<const f32x4 *>(scales + slot + rt * 16);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) total[rt][mt][i] = __builtin_fmaf(scale[i], product[rt][mt][i], total[rt][mt][i]);
                if constexpr (SUMS) {
                    const f32x4 offset = *reinterpret_cast<const f32x4 *>(offsets + slot + rt * 16);
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                        for (int i = 0; i < 4; ++i) total[rt][mt][i] = __builtin_fmaf(offset[i], sum[mt][i], total[rt][mt][i]);
                }
            }
        }
    };
    auto wave_fence = []() __attribute__((always_inline)) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    // One copy of the step's code, the next step's loads issued as its registers come free: copies for deeper prefetching
    // cost more in instruction fetches (a launch runs every line a few times only) than they hide.
#pragma unroll 1
    for (int step = wave; step < a.steps; step += waves) {
        wave_fence();   // the previous step's operands have been read
        pass_activations(piece, step);
        const int next = min(step + waves, a.steps - 1);
        load_activations(piece, next);
        wave_fence();
        multiply(raw, step);
        load_codes(raw, next);
    }

    // -- the wavefronts' sums, in wavefront order --------------------------------------------------------------------
    __syncthreads();
    f32x4 *sums = reinterpret_cast<f32x4 *>(lds);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) sums[(wave * RT * MT + rt * MT + mt) * 64 + lane] = total[rt][mt];
    __syncthreads();
#pragma unroll 1
    for (int item = threadIdx.x; item < RT * MT * 64; item += blockDim.x) {
        const int tile = item >> 6, rt = tile / MT, mt = tile - rt * MT, from = item & 63;
        const int local_row = rt * 16 + 4 * (from >> 4);
        const int row = first_row + local_row, sample = first_sample + mt * 16 + (from & 15);
        f32x4 value = *reinterpret_cast<const f32x4 *>(biases + local_row);
#pragma unroll 1
        for (int w = 0; w < waves; ++w) value += sums[w * RT * MT * 64 + item];
        const bool inside = sample < a.samples && row < a.rows;
        const float all = (value[0] + value[1]) + (value[2] + value[3]);
        if (const unsigned long long open = __ballot(inside && (!held || all - all != 0.0f)); __builtin_expect(open != 0, 0))   // (whole wavefronts take a turn)
            plain_outputs<FORMAT, XT>(a, open, first_row + rt * 16, first_sample + mt * 16, biases + rt * 16, value, lane);
        if (!inside) continue;
        const size_t at = static_cast<size_t>(sample) * a.rows + row;
        const int valid = min(4, a.rows - row);
        uint16_t *target = static_cast<uint16_t *>(a.y) + at;
        const mk_u32x2 packed = {pair_of<XT>(value[0], value[1]), pair_of<XT>(value[2], value[3])};
        if (a.whole_quads) *reinterpret_cast<mk_u32x2 *>(target) = packed;
        else
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (i < valid) target[i] = static_cast<uint16_t>(packed[i / 2] >> (16 * (i & 1)));
    }
}

// How a launch is cut.
struct MatmulPlan {
    int row_tiles, sample_tiles, waves, sub;   // RT, MT, wavefronts per workgroup, SUB
    bool split;                                // SPLIT
};

}  // namespace mk_matmul
