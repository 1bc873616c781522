// Vector grids on gfx950: nearest-codeword search (any codebook of 2-, 4-, 8- or
// 16-dimensional codewords; the structured search of the E8P lattice) and the LDL
// error-feedback tile that rounds blocks of `dimension` columns.
//
// One wavefront owns a row (or a vector): its 64 lanes share out the codebook entries -- four
// E8P magnitude patterns per lane, or every 64th codeword -- and the winner is the entry of the
// smallest cost, the lower index on ties, which is what a search in ascending order with a
// strict comparison returns.  Costs are formed in fp32 without fused multiply-adds (but where
// the product is exact), coordinates in ascending order.  The magnitude patterns, and any
// codebook of up to 48 KiB, are staged in LDS once per workgroup.
//
// What is done for each entry takes every lane; what is done once for a coordinate (its
// distance to either coset, its square, the winner's signs, its reconstruction and deviation)
// takes one lane per coordinate, and what is one number for the row is scalar.
//
// In the feedback tile everything a row needs of the tile lives in the wavefront's registers,
// lane l holding columns 2 l and 2 l + 1 (and, in tiles of more than 128 columns, those 128
// further).  A block's values are read out of them with wavefront-uniform lane reads, its
// coefficient rows are requested before its search so that their latency hides behind it, and
// reconstructions, deviations and codes wait in LDS for coalesced writes.
// An E8P point is rebuilt from its pattern, sign bits and coset instead of being fetched from
// the 2 MiB table.
//
// Replaces, in /root/reference/src/mlkit:
//   kernels/lattice_search.py:10-70       nearest_lattice_code / nearest_lattice -> mk_vector_nearest
//   kernels/error_feedback.py:146-274     round_vector_feedback_tile / round_vector_tile
//                                                                   -> mk_feedback_round_vector_tile

#include "mk_common.h"

namespace {

constexpr int kPatternsPerLane = 4;   // 256 E8P magnitude patterns over 64 lanes
constexpr int kPatternFloats = 256 * 8;
constexpr int kWaveRows = 4;          // wavefronts (rows) per workgroup
constexpr int kStagedBytes = 48 * 1024;

extern __shared__ __align__(16) float staged[];

__device__ __forceinline__ float lane_value(float value, int lane) {   // v_readlane: `lane` is wavefront-uniform
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, value), lane));
}

template <int CONTROL, int ROWS = 0xf>
__device__ __forceinline__ int moved(int bits) {
    return __builtin_amdgcn_update_dpp(bits, bits, CONTROL, ROWS, 0xf, ROWS == 0xf);
}

// The smallest of the 64 lanes' values, none of them NaN: as integers of the same order, for which a lane move and a minimum
// are one instruction.
__device__ __forceinline__ float wave_minimum(float value) {
    int key = __builtin_bit_cast(int, value);
    key ^= (key >> 31) & 0x7fffffff;
    key = min(key, moved<0x128>(key));        // row_ror:8, 4, 2, 1
    key = min(key, moved<0x124>(key));
    key = min(key, moved<0x122>(key));
    key = min(key, moved<0x121>(key));
    key = min(key, moved<0x142, 0xa>(key));   // row_bcast:15 into rows 1 and 3
    key = min(key, moved<0x143, 0xc>(key));   // row_bcast:31 into rows 2 and 3
    key = __builtin_amdgcn_readlane(key, 63);
    return __builtin_bit_cast(float, key ^ ((key >> 31) & 0x7fffffff));
}

// This lane's four magnitude patterns (pattern lane + 64 j), their squared norms, what a flip of their cheapest coordinate
// is to be multiplied by when the signs are even, and the parities of their sums (bit `lane` of parity[j]).
struct LanePatterns {
    float value[kPatternsPerLane][8];
    float norm[kPatternsPerLane], factor[kPatternsPerLane];
    uint64_t parity[kPatternsPerLane];
};

struct __attribute__((packed, aligned(4))) Pair {   // one 8-byte load at any float's address
    float value[2];
};

struct __attribute__((packed, aligned(4))) Quad {
    float value[4];
};

// `patterns`: the 256 x 8 table in global memory (not in LDS: these loads and the staging are in flight together).
__device__ __forceinline__ void load_patterns(LanePatterns &p, const float *patterns, int lane) {
#pragma unroll
    for (int j = 0; j < kPatternsPerLane; ++j)
#pragma unroll
        for (int d = 0; d < 8; d += 4) {
            const Quad quad = *reinterpret_cast<const Quad *>(patterns + (lane + 64 * j) * 8 + d);
#pragma unroll
            for (int i = 0; i < 4; ++i) p.value[j][d + i] = quad.value[i];
        }
#pragma unroll
    for (int j = 0; j < kPatternsPerLane; ++j) {
        float norm = 0.0f, total = 0.0f;   // (a sum of half-integers: exact)
#pragma unroll
        for (int d = 0; d < 8; ++d) {
            const float value = p.value[j][d];
            total += value;
            norm = __fadd_rn(norm, __fmul_rn(value, value));
        }
        const bool odd = static_cast<int>(total) & 1;
        p.norm[j] = norm;
        p.factor[j] = odd ? 4.0f : 0.0f;
        p.parity[j] = __ballot(odd);
    }
}

// Code of the E8P point nearest to the vector whose coordinate `lane & 7` is `own`, and that coordinate of the point.  For
// either coset every lane scores its four patterns -- the flip of the cheapest coordinate priced in when the pattern's parity
// disagrees with the signs of the vector -- and the first (coset, j, lane) of the smallest cost wins: the lowest index
// 256 coset + 64 j + lane, so that the -1/4 coset stays on a tie.  Only then are the winner's parity correction and its first
// cheapest coordinate worked out.
__device__ __forceinline__ int nearest_lattice_code(float own, const LanePatterns &p, const float *patterns, int lane, float &point) {
    // lanes 0 to 7 stand for the coset of -1/4, lanes 8 to 15 for that of +1/4
    const float centered_here = __fsub_rn(own, (lane & 8) ? 0.25f : -0.25f);
    const float absolute_here = __builtin_fabsf(centered_here), square = __fmul_rn(centered_here, centered_here);
    const uint32_t below = static_cast<uint32_t>(__ballot(centered_here < 0.0f));   // (a difference of equal numbers is +0)
    float squares = square;   // lanes 7 and 15: the sum in ascending order
#pragma unroll
    for (int d = 1; d < 8; ++d) squares = __fadd_rn(__builtin_bit_cast(float, moved<0x111>(__builtin_bit_cast(int, squares))), square);   // row_shr:1
    float cost[2 * kPatternsPerLane], smallest = __builtin_inff();
#pragma unroll
    for (int coset = 0; coset < 2; ++coset) {
        const float sum = lane_value(squares, 8 * coset + 7);
        const float odd = (__builtin_popcount((below >> (8 * coset)) & 255u) & 1) ? 4.0f : 0.0f;
        float absolute[8];
#pragma unroll
        for (int d = 0; d < 8; ++d) absolute[d] = lane_value(absolute_here, 8 * coset + d);
#pragma unroll
        for (int j = 0; j < kPatternsPerLane; ++j) {
            float dots = __fmul_rn(absolute[0], p.value[j][0]), cheapest = dots;
#pragma unroll
            for (int d = 1; d < 8; ++d) {
                const float product = __fmul_rn(absolute[d], p.value[j][d]);
                dots = __fadd_rn(dots, product);
                cheapest = __builtin_fminf(cheapest, product);
            }
            // products with 2 and 4 are exact; 0 times the cheapest adds nothing (it is finite wherever the rest is)
            float candidate = __builtin_fmaf(-2.0f, dots, __fadd_rn(sum, p.norm[j]));
            candidate = __builtin_fmaf(__builtin_fabsf(__fsub_rn(p.factor[j], odd)), cheapest, candidate);
            cost[kPatternsPerLane * coset + j] = candidate;
            smallest = __builtin_fminf(smallest, candidate);   // (NaN is never the smaller)
        }
    }
    smallest = wave_minimum(smallest);
    // no cost below infinity (NaN): pattern 0, no sign bits, the +1/4 coset
    const bool found = smallest < __builtin_inff();
    uint64_t lanes = 1;
    int slot = kPatternsPerLane;
#pragma unroll
    for (int k = 2 * kPatternsPerLane - 1; k >= 0; --k) {
        const uint64_t equal = __ballot(cost[k] == smallest);
        if (found && equal) {
            lanes = equal;
            slot = k;
        }
    }
    const int holder = __builtin_ctzll(lanes), j = slot & (kPatternsPerLane - 1), pattern = 64 * j + holder;
    const uint64_t odd = j == 0 ? p.parity[0] : j == 1 ? p.parity[1] : j == 2 ? p.parity[2] : p.parity[3];
    const int parity = static_cast<int>(odd >> holder) & 1;
    const float shift = slot < kPatternsPerLane ? -0.25f : 0.25f;
    const float row = patterns[pattern * 8 + (lane & 7)];
    const float centered = __fsub_rn(own, shift), product = __fmul_rn(__builtin_fabsf(centered), row);
    const int magnitude = __builtin_bit_cast(int, product);   // (not negative: ordered as integers)
    int cheapest = min(magnitude, moved<0xB1>(magnitude));    // quad_perm [1,0,3,2]
    cheapest = min(cheapest, moved<0x4E>(cheapest));          // quad_perm [2,3,0,1]
    cheapest = min(cheapest, moved<0x141>(cheapest));         // row_half_mirror
    const int axis = __builtin_ctz(static_cast<uint32_t>(__ballot(magnitude == cheapest)) | 256u);   // the first minimum
    const uint32_t negative = static_cast<uint32_t>(__ballot(centered < 0.0f)) & 255u;
    const bool flips = parity != (__builtin_popcount(negative) & 1) && axis < 7;
    const uint32_t signs = found ? (negative & 127u) ^ (flips ? 1u << axis : 0u) : 0u;
    const uint32_t all = signs | ((__builtin_popcount(signs) + parity) & 1) << 7;
    const uint32_t minus = (all << (31 - (lane & 7))) & 0x80000000u;
    point = __fadd_rn(__uint_as_float(__float_as_uint(row) ^ minus), shift);
    return found ? pattern * 128 + static_cast<int>(signs) + (slot < kPatternsPerLane ? 32768 : 0) : 0;
}

// Index of the nearest of `count` codewords of DIM floats (lowest index on ties).
template <int DIM>
__device__ __forceinline__ int nearest_codeword(const float (&v)[DIM], const float *codebook, int count, int lane) {
    float cost = __builtin_inff();
    int index = 0x7fffffff;
    for (int entry = lane; entry < count; entry += 64) {
        const float *word = codebook + static_cast<size_t>(entry) * DIM;
        float candidate = 0.0f;
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            const float difference = __fsub_rn(word[d], v[d]);
            candidate = __fadd_rn(candidate, __fmul_rn(difference, difference));
        }
        if (candidate < cost) {
            cost = candidate;
            index = entry;
        }
    }
    const float smallest = wave_minimum(cost);
    if (!(smallest < __builtin_inff())) return 0;  // no cost compared below infinity (NaN inputs): the first codeword
    uint64_t lanes = __ballot(cost == smallest);
    int best = 0x7fffffff;
    do {   // one lane but for ties
        best = min(best, __builtin_amdgcn_readlane(index, __builtin_ctzll(lanes)));
        lanes &= lanes - 1;
    } while (lanes);
    return best;
}

// The workgroup's table, and its copy into LDS: the magnitude patterns of the lattice, or the whole
// codebook when STAGED says it fits.  Nothing waits here; a barrier has to follow.
template <int DIM, bool LATTICE, bool STAGED>
__device__ __forceinline__ const float *stage_table(const float *codebook, int codebook_size) {
    const float *source = LATTICE ? codebook + static_cast<size_t>(codebook_size) * 8 : codebook;
    if constexpr (LATTICE) {
#pragma unroll
        for (int i = 0; i < kPatternFloats / (4 * 64 * kWaveRows); ++i) {
            const int at = 4 * (threadIdx.x + 64 * kWaveRows * i);
            *reinterpret_cast<Quad *>(staged + at) = *reinterpret_cast<const Quad *>(source + at);
        }
    } else if constexpr (STAGED) {
        for (int i = 2 * threadIdx.x; i < codebook_size * DIM; i += 2 * 64 * kWaveRows)   // (DIM is even)
            *reinterpret_cast<Pair *>(staged + i) = *reinterpret_cast<const Pair *>(source + i);
    }
    return source;
}

struct NearestArgs {
    const float *vectors;
    const float *codebook;  // [count, dim]; lattice: the 256 magnitude patterns follow
    int32_t *codes;
    long long vectors_count;
    int count;
};

template <int DIM, bool LATTICE, bool STAGED>
__global__ void __launch_bounds__(256) vector_nearest_kernel(const NearestArgs a) {
    const float *table = stage_table<DIM, LATTICE, STAGED>(a.codebook, a.count);
    const int lane = threadIdx.x & 63;
    const long long wave = static_cast<long long>(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const long long waves = static_cast<long long>(gridDim.x) * (blockDim.x >> 6);
    LanePatterns patterns;
    if constexpr (LATTICE) load_patterns(patterns, table, lane);
    __syncthreads();
    for (long long vector = wave; vector < a.vectors_count; vector += waves) {
        int code;
        if constexpr (LATTICE) {
            float point;
            code = nearest_lattice_code(a.vectors[vector * 8 + (lane & 7)], patterns, staged, lane, point);
        } else {
            float v[DIM];
#pragma unroll
            for (int d = 0; d < DIM; ++d) v[d] = a.vectors[vector * DIM + d];
            code = nearest_codeword<DIM>(v, STAGED ? staged : a.codebook, a.count, lane);
        }
        if (lane == 0) a.codes[vector] = code;
    }
}

struct VectorTileArgs {
    const float *original, *feedback, *coeff, *scales, *codebook;
    float *output;
    float *deviation_t;   // null, or [width, rows]: original - output, for the trailing updates
    int32_t *encoded;
    int rows, width, region_start, tile_start, tile_width, group, groups_per_row, codebook_size;
    int whole_rows;   // four rows' deviations of a column are one aligned store
};

constexpr int kSpan = 128;       // columns that the wavefront's pairs cover
constexpr int kSpans = 2;        // of them in the widest tile

// Coefficient rows of the block at `local` for the lane's columns in span HALF and behind it.  Columns that are not behind
// the block (or past the tile, which is even) receive numbers too: nothing reads the corrections of a rounded column again.
template <int DIM, int SPANS, int HALF>
__device__ __forceinline__ void request_rows(float (&rows)[DIM][2 * SPANS], const VectorTileArgs &a, int local, int lane) {
    const float *first = a.coeff + static_cast<size_t>(a.tile_start + local) * a.width + a.tile_start;
#pragma unroll
    for (int h = HALF; h < SPANS; ++h) {
        const int column = min(kSpan * h + 2 * lane, a.tile_width - 2);
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            const Pair pair = *reinterpret_cast<const Pair *>(first + static_cast<size_t>(d) * a.width + column);
            rows[d][2 * h] = pair.value[0];
            rows[d][2 * h + 1] = pair.value[1];
        }
    }
}

// A row's share of a tile: its columns in registers, and what waits in LDS to be written.
template <int SPANS>
struct RowTile {
    float corrections[2 * SPANS], weights[2 * SPANS], scales[2 * SPANS];
    float *restored, *deviations;   // [tile columns]
    int *codes;                     // [tile blocks]
};

// The blocks of span HALF, one after another.
template <int DIM, bool LATTICE, bool STAGED, int SPANS, int HALF>
__device__ __forceinline__ void round_span(RowTile<SPANS> &t, const VectorTileArgs &a, const LanePatterns &patterns, const float *original, int lane) {
    const int end = min(a.tile_width, kSpan * (HALF + 1));
    const int mine = lane & (DIM - 1);
    for (int local = kSpan * HALF; local < end; local += DIM) {
        float along[DIM][2 * SPANS];
        request_rows<DIM, SPANS, HALF>(along, a, local, lane);   // on their way during the search
        const float weight = original[local + mine];
        __builtin_amdgcn_sched_barrier(0);

        const int holder = (local - kSpan * HALF) >> 1;   // the lane with the block's first pair
        const float scale = lane_value(t.scales[2 * HALF], holder);  // a block lies inside one scale group
        float quotients[2];   // every lane divides its own columns
#pragma unroll
        for (int s = 0; s < 2; ++s)
            quotients[s] = __fdiv_rn(__fadd_rn(t.weights[2 * HALF + s], t.corrections[2 * HALF + s]), t.scales[2 * HALF + s]);
        int code;
        float word;   // the lane's coordinate
        if constexpr (LATTICE) {
            const int from = 4 * (holder + (mine >> 1));
            const float low = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(from, __builtin_bit_cast(int, quotients[0])));
            const float high = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(from, __builtin_bit_cast(int, quotients[1])));
            code = nearest_lattice_code((lane & 1) ? high : low, patterns, staged, lane, word);
        } else {
            float normalized[DIM];
#pragma unroll
            for (int d = 0; d < DIM; ++d) normalized[d] = lane_value(quotients[d & 1], holder + (d >> 1));
            const float *table = STAGED ? staged : a.codebook;
            code = nearest_codeword<DIM>(normalized, table, a.codebook_size, lane);
            word = table[static_cast<size_t>(code) * DIM + mine];
        }
        const float reconstruction = __fmul_rn(word, scale), deviation = __fsub_rn(weight, reconstruction);
        t.restored[local + mine] = reconstruction;   // (lanes of one coordinate write the same)
        t.deviations[local + mine] = deviation;
        t.codes[local / DIM] = code;
        float shared[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) shared[d] = lane_value(deviation, d);
#pragma unroll
        for (int s = 2 * HALF; s < 2 * SPANS; ++s) {
            float pushed = __fmul_rn(shared[0], along[0][s]);
#pragma unroll
            for (int d = 1; d < DIM; ++d) pushed = __fadd_rn(pushed, __fmul_rn(shared[d], along[d][s]));
            t.corrections[s] = __fadd_rn(t.corrections[s], pushed);
        }
    }
}

// SPANS spans of 128 columns.  Bound by vector-ALU issue along a row's chain of blocks, with two wavefronts per SIMD at 2048
// rows.  128 columns of 2048 rows on E8P: 30 us; 48 with four columns in each of 32 lanes, coefficients in 32 loads a block,
// costs and indexes reduced together, and a winner worked out by every lane for all coordinates.
template <int DIM, bool LATTICE, bool STAGED, int SPANS>
__global__ void __launch_bounds__(64 * kWaveRows) round_vector_tile_kernel(const VectorTileArgs a) {
    __shared__ __align__(16) float restored[kWaveRows][kSpan * SPANS], deviations[kWaveRows][kSpan * SPANS];
    __shared__ int codes[kWaveRows][kSpan * SPANS / DIM];
    const float *table = stage_table<DIM, LATTICE, STAGED>(a.codebook, a.codebook_size);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int first_row = blockIdx.x * kWaveRows;
    const int row = min(first_row + wave, a.rows - 1);   // wavefronts behind the last row do its work again and write nothing
    const size_t row_base = static_cast<size_t>(row) * a.width;
    RowTile<SPANS> t;
    t.restored = restored[wave];
    t.deviations = deviations[wave];
    t.codes = codes[wave];
#pragma unroll
    for (int h = 0; h < SPANS; ++h) {
        const int column = kSpan * h + 2 * lane;   // (a tile is even: a pair lies inside or outside)
        const bool inside = column < a.tile_width;
        const size_t at = row_base + a.tile_start + (inside ? column : 0);
        const Pair feedback = *reinterpret_cast<const Pair *>(a.feedback + at), weights = *reinterpret_cast<const Pair *>(a.original + at);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            t.corrections[2 * h + s] = inside ? feedback.value[s] : 0.0f;
            t.weights[2 * h + s] = inside ? weights.value[s] : 0.0f;
            const int group = (a.tile_start + (inside ? column + s : 0) - a.region_start) / a.group;
            t.scales[2 * h + s] = a.scales[static_cast<size_t>(row) * a.groups_per_row + group];
        }
    }
    LanePatterns patterns;
    if constexpr (LATTICE) load_patterns(patterns, table, lane);
    __syncthreads();
    const float *original = a.original + row_base + a.tile_start;
    round_span<DIM, LATTICE, STAGED, SPANS, 0>(t, a, patterns, original, lane);
    if constexpr (SPANS > 1) round_span<DIM, LATTICE, STAGED, SPANS, SPANS - 1>(t, a, patterns, original, lane);

    __syncthreads();
    if (first_row + wave < a.rows) {
        for (int column = lane; column < a.tile_width; column += 64) a.output[row_base + a.tile_start + column] = restored[wave][column];
        int32_t *encoded = a.encoded + static_cast<size_t>(row) * (a.width / DIM) + a.tile_start / DIM;
        for (int block = lane; block < a.tile_width / DIM; block += 64) encoded[block] = codes[wave][block];
    }
    if (a.deviation_t) {
        for (int column = threadIdx.x; column < a.tile_width; column += 64 * kWaveRows) {
            float *target = a.deviation_t + static_cast<size_t>(a.tile_start + column) * a.rows + first_row;
            if (a.whole_rows) {
                static_assert(kWaveRows == 4, "one float4 of a column's rows");
                *reinterpret_cast<float4 *>(target) = make_float4(deviations[0][column], deviations[1][column], deviations[2][column], deviations[3][column]);
            } else {
#pragma unroll
                for (int r = 0; r < kWaveRows; ++r)
                    if (first_row + r < a.rows) target[r] = deviations[r][column];
            }
        }
    }
}

// LDS a launch needs: the pattern table, or the codebook when it is staged.
inline bool fits_in_lds(int entries, int dimension) {
    return static_cast<size_t>(entries) * dimension * sizeof(float) <= kStagedBytes;
}

}  // namespace

extern "C" int mk_vector_nearest(const float *vectors, long long count, int dimension, const float *codebook,
                                 int codebook_size, int lattice, int32_t *codes, void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MK_REQUIRE(count >= 0 && codebook_size >= 1, MK_ERR_INVALID, "mk_vector_nearest: sizes must be positive");
    MK_REQUIRE(dimension == 2 || dimension == 4 || dimension == 8 || dimension == 16, MK_ERR_UNSUPPORTED,
               "mk_vector_nearest: codewords of 2, 4, 8 or 16 coordinates (got %d)", dimension);
    MK_REQUIRE(!lattice || (dimension == 8 && codebook_size == 65536), MK_ERR_INVALID,
               "mk_vector_nearest: the lattice search needs the 65536-point table of 8 coordinates");
    if (count == 0) return MK_OK;
    MK_REQUIRE(vectors && codebook && codes, MK_ERR_INVALID, "mk_vector_nearest: null tensor pointer");
    NearestArgs a{vectors, codebook, codes, count, codebook_size};
    long long blocks = (count + 3) / 4;
    if (blocks > 256 * 16) blocks = 256 * 16;
    const dim3 grid(static_cast<unsigned>(blocks)), block(256);
    const bool staged_codebook = !lattice && fits_in_lds(codebook_size, dimension);
    const size_t lds = lattice ? kPatternFloats * sizeof(float)
                               : (staged_codebook ? static_cast<size_t>(codebook_size) * dimension * sizeof(float) : 0);
#define MK_NEAREST(DIM)                                                                                          \
    if (staged_codebook) hipLaunchKernelGGL((vector_nearest_kernel<DIM, false, true>), grid, block, lds, stream, a); \
    else hipLaunchKernelGGL((vector_nearest_kernel<DIM, false, false>), grid, block, 0, stream, a)
    if (lattice) hipLaunchKernelGGL((vector_nearest_kernel<8, true, false>), grid, block, lds, stream, a);
    else if (dimension == 2) { MK_NEAREST(2); }
    else if (dimension == 4) { MK_NEAREST(4); }
    else if (dimension == 8) { MK_NEAREST(8); }
    else { MK_NEAREST(16); }
#undef MK_NEAREST
    MK_LAUNCH_CHECK("mk_vector_nearest");
    return MK_OK;
}

// Shared with the sweep over all regions, whose scales lie `groups_per_row` apart and whose deviations are kept.
int mk_round_vector_tile(const float *original, const float *feedback, const float *coeff, const float *scales,
                         const float *codebook, float *output, float *deviation_t, int32_t *encoded, int rows, int width,
                         int region_start, int tile_start, int tile_width, int group, int groups_per_row, int dimension,
                         int codebook_size, int lattice, hipStream_t stream) {
    MK_REQUIRE(original && feedback && coeff && scales && codebook && output && encoded, MK_ERR_INVALID,
               "mk_feedback_round_vector_tile: null tensor pointer");
    MK_REQUIRE(rows >= 1 && width >= 1 && group >= 1 && codebook_size >= 1, MK_ERR_INVALID,
               "mk_feedback_round_vector_tile: sizes must be positive");
    MK_REQUIRE(dimension == 2 || dimension == 4 || dimension == 8 || dimension == 16, MK_ERR_UNSUPPORTED,
               "mk_feedback_round_vector_tile: codewords of 2, 4, 8 or 16 coordinates (got %d)", dimension);
    MK_REQUIRE(tile_start >= 0 && tile_width >= 1 && tile_start + tile_width <= width && tile_start >= region_start,
               MK_ERR_INVALID, "mk_feedback_round_vector_tile: columns [%d, %d) lie outside a row of %d", tile_start,
               tile_start + tile_width, width);
    MK_REQUIRE(tile_width <= kSpan * kSpans, MK_ERR_UNSUPPORTED,
               "mk_feedback_round_vector_tile: at most %d columns per call (got %d)", kSpan * kSpans, tile_width);
    MK_REQUIRE(width % dimension == 0 && tile_start % dimension == 0 && tile_width % dimension == 0 &&
                   group % dimension == 0,
               MK_ERR_INVALID, "mk_feedback_round_vector_tile: rows, tiles and scale groups must hold whole codewords");
    MK_REQUIRE(!lattice || (dimension == 8 && codebook_size == 65536), MK_ERR_INVALID,
               "mk_feedback_round_vector_tile: the lattice search needs the 65536-point table of 8 coordinates");
    VectorTileArgs a{original, feedback, coeff, scales, codebook, output, deviation_t, encoded, rows, width, region_start, tile_start,
                     tile_width, group, groups_per_row, codebook_size,
                     rows % kWaveRows == 0 && (reinterpret_cast<uintptr_t>(deviation_t) & 15u) == 0};
    const dim3 grid(mk_cdiv(rows, kWaveRows)), block(64 * kWaveRows);
    const bool staged_codebook = !lattice && fits_in_lds(codebook_size, dimension);
    const size_t lds = lattice ? kPatternFloats * sizeof(float)
                               : (staged_codebook ? static_cast<size_t>(codebook_size) * dimension * sizeof(float) : 0);
#define MK_TILE(...)                                                                                                   \
    if (tile_width <= kSpan) hipLaunchKernelGGL((round_vector_tile_kernel<__VA_ARGS__, 1>), grid, block, lds, stream, a); \
    else hipLaunchKernelGGL((round_vector_tile_kernel<__VA_ARGS__, kSpans>), grid, block, lds, stream, a)
#define MK_TILE_CODEBOOK(DIM)                             \
    if (staged_codebook) { MK_TILE(DIM, false, true); }   \
    else { MK_TILE(DIM, false, false); }
    if (lattice) { MK_TILE(8, true, false); }
    else if (dimension == 2) { MK_TILE_CODEBOOK(2) }
    else if (dimension == 4) { MK_TILE_CODEBOOK(4) }
    else if (dimension == 8) { MK_TILE_CODEBOOK(8) }
    else { MK_TILE_CODEBOOK(16) }
#undef MK_TILE_CODEBOOK
#undef MK_TILE
    MK_LAUNCH_CHECK("mk_feedback_round_vector_tile");
    return MK_OK;
}

extern "C" int mk_feedback_round_vector_tile(const float *original, const float *feedback, const float *coeff,
                                             const float *scales, const float *codebook, float *output,
                                             int32_t *encoded, int rows, int width, int region_start,
                                             int tile_start, int tile_width, int group, int groups_per_row,
                                             int dimension, int codebook_size, int lattice, void *stream) {
    return mk_round_vector_tile(original, feedback, coeff, scales, codebook, output, nullptr, encoded, rows, width, region_start,
                                tile_start, tile_width, group, groups_per_row, dimension, codebook_size, lattice,
                                static_cast<hipStream_t>(stream));
}
