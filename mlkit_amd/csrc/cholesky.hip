// Diagonal-block step of a blocked Cholesky factorisation on gfx950.
//
// The error-feedback coefficients are U blockdiag(U)^-1 for the damped Hessian H = U^T U
// (K up to 16384).  The library factorisation spends most of its time in its small
// unblocked panel kernel, so the blocked algorithm is driven from the host; its products are
// those of factor_products.hip, and this file supplies the rest: a workgroup factors a
// diagonal block of at most 128 x 128 in registers and, on request, carries 64 columns of the
// block's rows through the same elimination, which makes them the factor's block row (one workgroup per 64 columns; no triangular solve is needed).
//
// Replaces the `torch.linalg.cholesky_ex` call of `feedback_coefficients`
// (quantization/algorithms/error_feedback.py:37-83 in /root/reference/src/mlkit) for large
// matrices on the device; mk_hessian_reversed, mk_unit_upper_from_factor and
// mk_blocks_upper_from_factor are the tensor operations in front of it and behind it (:55-66
// index reversal and damping, :72-83 division by the diagonal or its blocks and reversal
// back), one pass over the matrix each.

#include "mk_common.h"

#include <type_traits>

namespace {

constexpr int kBlock = 128;
constexpr int kThreads = 256;

struct BlockArgs {
    float *matrix;       // the block's top-left element; row-major with `leading` floats per row
    long long leading;
    int size;            // rows = columns of the block, 1 ... 128
    int first_column;    // index of the block's first column in the whole matrix (for status)
    int *status;         // stays 0, or becomes 1 + the column whose pivot is not positive
    int row_columns;     // columns to the right of the block, in the same rows, that take the same elimination
    float *factor_out;   // where the factor goes when row_columns > 0 (128 floats per row); else in place
};

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float lane_value(float x, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

constexpr int kTile = 16;                       // rows and columns of a tile
constexpr int kTiles = kBlock / kTile;          // tile columns of the block
constexpr int kWaves = kThreads / 64;
constexpr int kCarried = kWaves * kTile;        // columns a workgroup carries beside the block
constexpr int kColumnFloats = kTile + 4;        // a tile column in LDS (16-byte aligned, banks spread)

// In: the upper triangle of a symmetric positive definite block.  Out: U with block = U^T U
// in the upper triangle, zeros below it.  A pivot that is not positive (or not finite)
// records its column and leaves the block unspecified.
//
// ROW: the workgroup also carries 64 columns to the right of the block, which take the same row
// operations and so become U_jj^-T A_jr, the block row of the factor.  Every workgroup factors the block
// itself (from the matrix, which nobody overwrites: the factor goes to `factor_out`), and the first one stores it.
//
// Right-looking over panels of 16 rows, by two sets of four wavefronts.  The second set holds the block and the carried
// columns as 16 x 16 tiles (negated) in its accumulators, wavefront w of it tile columns 3 - w, 4 + w and, beside the block, w;
// the first eliminates, its wavefront w the columns of the same tiles.  Per panel:
//   1. the tiles' owners put the panel's row of tiles into LDS by columns; barrier;
//   2. a lane of the first set takes a column of 16 values into registers, lanes 0 ... 15 of EVERY wavefront the diagonal
//      tile's, the other lanes those of the wavefront's three tiles, and all 16 elimination steps run inside the wavefront: row
//      j is scaled by 1 / sqrt(pivot), row i > j loses U[j][i] (a scalar, from lane i) times row j.  Finished rows go back to
//      LDS four at a time; barrier;
//   3. the next row of tiles loses U_r^T U_c on the matrix cores and goes out as in 1; barrier.  The other rows, and the
//      finished rows' way to memory, follow beside the next elimination.
// A 16 x 16 x 4 accumulator holds rows 4 (lane / 16) + i of a column where the operands hold k = lane / 16, so product i takes
// k = 4 (lane / 16) + i and a tile is read as an operand exactly as it is held: one 16-byte LDS read.  A panel's sixteen
// products are summed first and subtracted in one addition, so an entry is rounded at most 7 + 15 times on its way (128
// times in a running accumulator, which left the coefficients of 1024 columns 4.1e-7 from 64 bits; now 2.6e-7, 3.3e-7
// with PAIRS).
//
// PAIRS: two rows at a time -- both are finished, then an entry loses fma(u_j, u_j, u_{j+1} u_{j+1}) in one subtraction, pair by
// pair -- in the elimination as on the matrix cores, where a product of 16 x 16 x 1 in four blocks takes row j + 1 of a tile
// times the wavefront's three tiles and a second one adds row j.  The order of additions that the coefficients of vector grids
// are worked out in: a code that a last bit of a coefficient turns takes the rest of its row along when it stands for eight
// weights, and conversions stay what they were, bit for bit.
//
// What bounds the kernel is the chain of 128 pivots: a panel takes about 4000 cycles, 1550 of them elimination (up to 2700
// while the other set's products share the SIMD), 700 the products it waits for.  One copy of the code serves all panels, since
// a launch runs it once and instruction fetches would show.  A block with 768 columns beside it, called back to back: 17.9 us;
// with one set of four wavefronts doing all of it in turn 24.9 (2200 cycles a panel went into the stores alone, and as many
// into products that nobody waited for yet).  The rows' factors as row broadcasts instead of scalars, with the diagonal tile
// in all lanes: 26.8 (the broadcasts do not become part of the multiply-adds).  With PAIRS 28.6 (between others, 64 to 1920
// columns beside the block); 48.3 with 64 entries of the block in each of 256 threads and a barrier for every pair.
template <bool ROW, bool PAIRS>
__global__ void __launch_bounds__(2 * kThreads, 2) cholesky_block_kernel(const BlockArgs a) {
    __builtin_amdgcn_s_setprio(3);   // in front of a trailing update that runs beside it
    __shared__ __align__(16) float panel[2][kTiles + kWaves][kTile][kColumnFloats];   // [buffer][tile column][column][row]
    // (in the padding: 30720 bytes of LDS go beside two workgroups of a trailing update, one word more does not)
    int &failed = reinterpret_cast<int &>(panel[1][0][0][kTile]), &stopped = reinterpret_cast<int &>(panel[1][0][0][kTile + 1]);
    if (threadIdx.x == 0) failed = *a.status, stopped = 0;
    const int n = a.size;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & (kWaves - 1));
    const bool eliminating = __builtin_amdgcn_readfirstlane(threadIdx.x / kThreads) == 0;
    const int column = lane & 15, quarter = lane >> 4;
    const int left_column = kWaves - 1 - wave, right_column = wave + kWaves;
    const int carried_first = kCarried * static_cast<int>(blockIdx.x) + kTile * wave;   // of this wavefront, counted from the block's end
    // Addresses are clamped into the block instead of guarded: a branch per load would wait for each of them in turn.
    const uint32_t leading = static_cast<uint32_t>(a.leading), last = static_cast<uint32_t>(n - 1);
    const uint32_t carried_column = n + min(carried_first + column, a.row_columns - 1);
    const int panels = (n + kTile - 1) / kTile;
    float *factor = ROW ? a.factor_out : a.matrix;
    const uint32_t factor_leading = ROW ? kBlock : leading;

    if (!eliminating) {   // uniform
        // tiles of row r: tile column 3 - wave (r <= 3), tile column wave + 4, the carried ones
        f32x4 left[kWaves], right[kTiles], beside[kTiles];
        auto block_tile = [&](int r, int c) __attribute__((always_inline)) -> f32x4 {
            f32x4 tile;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t first = r * kTile + 4 * quarter + i, second = c * kTile + column;
                const uint32_t row = min(first, second), col = max(first, second);   // the upper triangle stands for both
                tile[i] = a.matrix[min(row, last) * leading + min(col, last)];
            }
            return tile;
        };
#pragma unroll
        for (int r = 0; r < kTiles; ++r) {
            if (r < kWaves) left[r] = block_tile(r, left_column);   // (tiles below the diagonal: any numbers, never used)
            right[r] = block_tile(r, right_column);
            if constexpr (ROW) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    beside[r][i] = a.matrix[min(static_cast<uint32_t>(r * kTile + 4 * quarter + i), last) * leading + carried_column];
            }
        }
#pragma unroll
        for (int r = 0; r < kTiles; ++r) {
            // Outside the block: an identity diagonal keeps every pivot of the padding at one.
            auto negated = [&](f32x4 &tile, int c) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int row = r * kTile + 4 * quarter + i, col = c * kTile + column;
                    tile[i] = max(row, col) < n ? -tile[i] : (row == col ? -1.0f : 0.0f);
                }
            };
            if (r < kWaves) negated(left[r], left_column);
            negated(right[r], right_column);
            if constexpr (ROW) {
#pragma unroll
                for (int i = 0; i < 4; ++i) beside[r][i] = r * kTile + 4 * quarter + i < n ? -beside[r][i] : 0.0f;
            }
        }
        auto publish = [&](int r) __attribute__((always_inline)) {   // row r of the wavefront's tiles, by columns
            float (*tiles)[kTile][kColumnFloats] = panel[r & 1];
            auto put = [&](int tile_column, f32x4 tile) __attribute__((always_inline)) {
                *reinterpret_cast<f32x4 *>(&tiles[tile_column][column][4 * quarter]) = -tile;
            };
            if (r < kWaves) put(left_column, left[r]);
            put(right_column, right[r]);
            if constexpr (ROW) put(wave + kTiles, beside[r]);
        };
        publish(0);
        __syncthreads();
        if (failed) return;   // an earlier block already did: do nothing
#pragma unroll 1
        for (int s = 0; s + 1 < panels; ++s) {
            __builtin_amdgcn_s_setprio(3);   // the other wavefronts wait
            __syncthreads();   // the finished rows of panel s are there
            if (stopped) return;
            float (*tiles)[kTile][kColumnFloats] = panel[s & 1];
            auto operand = [&](int tile_column) __attribute__((always_inline)) -> f32x4 {
                return *reinterpret_cast<const f32x4 *>(&tiles[tile_column][column][4 * quarter]);
            };
            // PAIRS: the panel's values of a column; lanes of quarter 0, 1 and 2 hold those of the three tiles' columns
            auto column_of = [&](float (&values)[kTile], int tile_column) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const f32x4 four = reinterpret_cast<const f32x4 *>(tiles[tile_column][column])[i];
#pragma unroll
                    for (int k = 0; k < 4; ++k) values[4 * i + k] = four[k];
                }
            };
            float columns[PAIRS ? kTile : 1];
            if constexpr (PAIRS) column_of(columns, quarter == 1 ? right_column : ROW && quarter == 2 ? wave + kTiles : left_column);
            auto pairs_from = [&](int r, f32x4 &on_left, f32x4 &on_right, f32x4 &on_beside) __attribute__((always_inline)) {
                float rows[kTile];
                column_of(rows, r);
#pragma unroll
                for (int k = 0; k < kTile; k += 2) {
                    f32x16 sum = {};   // of row k + 1, then of row k
                    sum = __builtin_amdgcn_mfma_f32_16x16x1f32(rows[k + 1], columns[k + 1], sum, 0, 0, 0);
                    sum = __builtin_amdgcn_mfma_f32_16x16x1f32(rows[k], columns[k], sum, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        on_left[i] += sum[i];
                        on_right[i] += sum[4 + i];
                        if constexpr (ROW) on_beside[i] += sum[8 + i];
                    }
                }
            };
            // what the next elimination waits for: tile row s + 1
            const f32x4 u_left = operand(left_column), u_right = operand(right_column), u_beside = operand(ROW ? wave + kTiles : wave);
            f32x4 from_left = {}, from_right = {}, from_beside = {};
            if constexpr (PAIRS) {
#pragma unroll
                for (int r = 1; r < kTiles; ++r)
                    if (r == s + 1) {   // uniform
                        if (r < kWaves) from_left = left[r];
                        from_right = right[r];
                        if constexpr (ROW) from_beside = beside[r];
                    }
                pairs_from(s + 1, from_left, from_right, from_beside);
            } else {
                const f32x4 next = operand(s + 1);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    from_left = __builtin_amdgcn_mfma_f32_16x16x4f32(next[i], u_left[i], from_left, 0, 0, 0);
                    from_right = __builtin_amdgcn_mfma_f32_16x16x4f32(next[i], u_right[i], from_right, 0, 0, 0);
                    if constexpr (ROW) from_beside = __builtin_amdgcn_mfma_f32_16x16x4f32(next[i], u_beside[i], from_beside, 0, 0, 0);
                }
            }
#pragma unroll
            for (int r = 1; r < kTiles; ++r)
                if (r == s + 1) {   // uniform
                    if (r < kWaves) left[r] = PAIRS ? from_left : left[r] + from_left;
                    right[r] = PAIRS ? from_right : right[r] + from_right;
                    if constexpr (ROW) beside[r] = PAIRS ? from_beside : beside[r] + from_beside;
                    publish(r);
                }
            __syncthreads();
            // Beside that elimination: what panel s takes from the rows behind, and its finished rows to memory.
            __builtin_amdgcn_s_setprio(2);
#pragma unroll
            for (int r = 2; r < kTiles; ++r) {
                if (r <= s + 1) continue;   // uniform, as all the conditions here
                if constexpr (PAIRS) {
                    f32x4 unused = {};
                    pairs_from(r, r < kWaves ? left[r] : unused, right[r], beside[r]);
                    continue;
                }
                const f32x4 row_operand = operand(r);
                auto products = [&](f32x4 u) __attribute__((always_inline)) -> f32x4 {
                    f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int i = 0; i < 4; ++i) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(row_operand[i], u[i], sum, 0, 0, 0);
                    return sum;
                };
                if (r < kWaves && r <= left_column) left[r] += products(u_left);   // (tiles below the diagonal are not needed)
                if (r <= right_column) right[r] += products(u_right);
                if constexpr (ROW) beside[r] += products(u_beside);
            }
            const int row = s * kTile + 4 * quarter;   // of this lane's first value
            if (blockIdx.x == 0) {   // uniform
                auto store = [&](int tile_column, f32x4 tile) __attribute__((always_inline)) {
                    const int to = tile_column * kTile + column;
                    if (tile_column == s) tile = operand(s);   // (finished behind the barrier)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (row + i < n && to < n) factor[(row + i) * factor_leading + to] = to >= row + i ? tile[i] : 0.0f;
                };
                store(left_column, u_left);
                store(right_column, u_right);
            }
            if constexpr (ROW) {
                if (carried_first + column < a.row_columns) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (row + i < n) a.matrix[(row + i) * leading + carried_column] = u_beside[i];
                }
            }
        }
        return;
    }

    __syncthreads();
    if (failed) return;
#pragma unroll 1
    for (int s = 0; s < panels; ++s) {
        float (*tiles)[kTile][kColumnFloats] = panel[s & 1];
        // a column of the panel per lane
        const int own = quarter == 1 ? left_column : wave + kWaves * (quarter - 1);   // tile column of lanes 16 ... 63
        float *source = tiles[quarter == 0 ? s : own][column];
        float value[kTile];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const f32x4 four = reinterpret_cast<const f32x4 *>(source)[i];
#pragma unroll
            for (int k = 0; k < 4; ++k) value[4 * i + k] = four[k];
        }
        auto keep = [&](int first, int stop) __attribute__((always_inline)) {   // finished rows, four at a time
#pragma unroll
            for (int i = first; i < stop; ++i)
                reinterpret_cast<f32x4 *>(source)[i] = f32x4{value[4 * i], value[4 * i + 1], value[4 * i + 2], value[4 * i + 3]};
        };
        float pivot = 1.0f;   // of this lane's column
        auto reciprocal_root = [&](int j) __attribute__((always_inline)) -> float {
            pivot = lane == j ? value[j] : pivot;
            return __builtin_amdgcn_rsqf(lane_value(value[j], j));   // accurate to an ulp; an IEEE square root and division would double the chain
        };
        if constexpr (PAIRS) {
            float reciprocal = reciprocal_root(0);
#pragma unroll
            for (int j = 0; j < kTile; j += 2) {
                value[j] *= reciprocal;
                const float link = lane_value(value[j], j + 1);
                value[j + 1] = __builtin_fmaf(-link, value[j], value[j + 1]);
                value[j + 1] *= reciprocal_root(j + 1);
                auto take = [&](int i) __attribute__((always_inline)) {   // one rounding for the pair's sum, one for the difference
                    const float first = lane_value(value[j], i), second = lane_value(value[j + 1], i);
                    value[i] -= __builtin_fmaf(first, value[j], second * value[j + 1]);
                };
                if (j + 2 < kTile) {
                    take(j + 2);
                    reciprocal = reciprocal_root(j + 2);
                }
#pragma unroll
                for (int i = j + 3; i < kTile; ++i) take(i);
                if ((j & 3) == 2 && quarter > 0 && own != s && (ROW || quarter < 3)) keep(j / 4, j / 4 + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            float reciprocal = reciprocal_root(0);
#pragma unroll
            for (int j = 0; j < kTile; ++j) {
                value[j] *= reciprocal;
                if (j + 1 < kTile) {   // the next pivot's chain first: the rest of this step hides its latency
                    value[j + 1] = __builtin_fmaf(-lane_value(value[j], j + 1), value[j], value[j + 1]);
                    reciprocal = reciprocal_root(j + 1);
                }
                float factors[kTile];
#pragma unroll
                for (int i = j + 2; i < kTile; ++i) factors[i] = lane_value(value[j], i);
#pragma unroll
                for (int i = j + 2; i < kTile; ++i) value[i] = __builtin_fmaf(-factors[i], value[j], value[i]);
                // (the diagonal tile later: another wavefront may still have to read it as it was)
                if ((j & 3) == 3 && quarter > 0 && own != s && (ROW || quarter < 3)) keep(j / 4, j / 4 + 1);
                // step by step: put off, as the compiler would have it, the updates of a row are one dependent chain
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        const uint64_t accepted = __builtin_amdgcn_ballot_w64(static_cast<uint32_t>(__float_as_int(pivot)) - 1u < 0x7f7fffffu);   // positive and finite
        const uint32_t refused = ~static_cast<uint32_t>(accepted) & 0xffffu;
        if (refused) {   // every eliminating wavefront of every workgroup comes to the same value
            if (threadIdx.x == 0) *a.status = a.first_column + s * kTile + __builtin_ctz(refused) + 1;
            stopped = 1;
            if (s + 1 < panels) __syncthreads();   // the others read it behind this barrier
            return;
        }
        if (s + 1 < panels) {
            __syncthreads();
            if (quarter == 0 && wave == 0) keep(0, 4);
            __syncthreads();   // the next panel's rows are there
            continue;
        }
        // The last panel's rows: lanes 0 ... 15 of the diagonal tile's owner, and the other tiles from their columns' lanes.
        if (blockIdx.x == 0 && (quarter == 0 ? s == left_column || s == right_column : quarter < 3 && own != s)) {
            const int to = (quarter == 0 ? s : own) * kTile + column;
            if (to < n) {
#pragma unroll
                for (int j = 0; j < kTile; ++j) {
                    const int row = s * kTile + j;   // uniform
                    if (row < n) factor[row * factor_leading + to] = to >= row ? value[j] : 0.0f;
                }
            }
        }
        if constexpr (ROW) {
            if (quarter == 3 && carried_first + column < a.row_columns) {
#pragma unroll
                for (int j = 0; j < kTile; ++j) {
                    const int row = s * kTile + j;
                    if (row < n) a.matrix[row * leading + carried_column] = value[j];
                }
            }
        }
    }
}

}  // namespace

// ---- the matrix that goes into the factorisation, and the coefficients that come out ---------

struct ReverseArgs {
    const float *source;
    float *target;
    const long long *order;  // null: index a reads row / column width - 1 - a
    const float *addend;     // one float: added to every diagonal entry (after zeros became ones)
    int width;
};

// target[a][b] = source[i(a)][i(b)]; on the diagonal a zero becomes one and *addend is added.
__global__ void __launch_bounds__(256) reversed_matrix_kernel(const ReverseArgs a) {
    const int row = blockIdx.y;
    const int column = (blockIdx.x * 256 + threadIdx.x) * 4;
    if (column >= a.width) return;
    const long long source_row = a.order ? a.order[row] : a.width - 1 - row;
    const float *from = a.source + static_cast<size_t>(source_row) * a.width;
    float values[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int b = column + i;
        const bool inside = b < a.width;
        const long long source_column = a.order ? a.order[inside ? b : 0] : a.width - 1 - (inside ? b : 0);
        float value = from[source_column];
        if (b == row) value = __fadd_rn(value == 0.0f ? 1.0f : value, *a.addend);
        values[i] = value;
    }
    float *to = a.target + static_cast<size_t>(row) * a.width + column;
    if (column + 3 < a.width && (a.width & 3) == 0) {
        *reinterpret_cast<float4 *>(to) = make_float4(values[0], values[1], values[2], values[3]);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (column + i < a.width) to[i] = values[i];
    }
}

// out[a][b] = U[w-1-b][w-1-a] / U[w-1-b][w-1-b] on and above the diagonal, zero below it: the factor transposed, every
// column divided by its diagonal entry, both index orders reversed; 32 x 32 tiles turned in LDS so that reads and writes both
// run along rows.  Tiles below the diagonal are not read.
__global__ void __launch_bounds__(256) unit_upper_kernel(const float *factor, float *out, int width) {
    __shared__ float tile[32][33];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;   // 8 rows of 32 threads
    const int r0 = blockIdx.y * 32, c0 = blockIdx.x * 32;
    if (blockIdx.x >= blockIdx.y) {   // uniform
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = r0 + ty + 8 * j, c = c0 + tx;
            const bool inside = r < width && c < width && r <= c;
            const float value = factor[static_cast<size_t>(inside ? r : 0) * width + (inside ? c : 0)];
            const float pivot = factor[static_cast<size_t>(inside ? r : 0) * (width + 1)];
            tile[ty + 8 * j][tx] = inside ? __fdiv_rn(value, pivot) : 0.0f;
        }
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) tile[ty + 8 * j][tx] = 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int c = c0 + ty + 8 * j, r = r0 + tx;   // tile[r - r0][c - c0] goes to out[w-1-c][w-1-r]
        if (r < width && c < width)
            out[static_cast<size_t>(width - 1 - c) * width + (width - 1 - r)] = tile[tx][ty + 8 * j];
    }
}

// The same for steps of STEP columns: with R[a][b] = U[w-1-b][w-1-a], every row of a block column of R times the inverse of the
// block on the diagonal, by forward substitution -- x_j = (r_j - x_0 d_0j - x_1 d_1j - ...) / d_jj, fused, in ascending order, which
// are the bits that the library's triangular solve gives.  64 x 64 tiles: a lane holds a row of a block column (whose STEP
// values lie in STEP rows of U, side by side for the lanes), the block on the diagonal is uniform, and results are turned in LDS.
// Bound by HBM.  2048 columns, steps of 8: 8.7 us, 153 as tensor operations (zeros below the diagonal, reversal, a
// gathered and turned copy, the library's solve, two copies back).
template <int STEP>
__global__ void __launch_bounds__(256) blocks_upper_kernel(const float *factor, float *out, int width) {
    __shared__ float tile[64][65];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
    if (blockIdx.x >= blockIdx.y) {   // uniform
        const int r = r0 + lane;
        for (int first = wave * STEP; first < 64; first += 4 * STEP) {
            const int column = c0 + first;
            if (column >= width) break;   // uniform; (the width holds whole blocks)
            const float *corner = factor + static_cast<size_t>(width - 1 - column) * (width + 1);   // d_kj: j rows above, k columns before
            float x[STEP];
#pragma unroll
            for (int j = 0; j < STEP; ++j) {
                const float *row = factor + static_cast<size_t>(width - 1 - column - j) * width + (width - 1);
                x[j] = row[-min(r, column + j)];
            }
#pragma unroll
            for (int j = 0; j < STEP; ++j) {
                float rest = r <= column + j ? x[j] : 0.0f;
#pragma unroll
                for (int k = 0; k < j; ++k) rest = __builtin_fmaf(-x[k], corner[-(static_cast<ptrdiff_t>(j) * width + k)], rest);
                x[j] = __fdiv_rn(rest, corner[-(static_cast<ptrdiff_t>(j) * width + j)]);
                tile[lane][first + j] = x[j];
            }
        }
    } else {
        for (int i = threadIdx.x; i < 64 * 64; i += 256) tile[i >> 6][i & 63] = 0.0f;
    }
    __syncthreads();
    for (int i = wave; i < 64; i += 4)
        if (r0 + i < width && c0 + lane < width) out[static_cast<size_t>(r0 + i) * width + c0 + lane] = tile[i][lane];
}

extern "C" int mk_hessian_reversed(const float *source, float *target, int width, const long long *order,
                                   const float *addend, void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MK_REQUIRE(source && target && addend, MK_ERR_INVALID, "mk_hessian_reversed: null pointer");
    MK_REQUIRE(width >= 1 && width <= 65535, MK_ERR_INVALID, "mk_hessian_reversed: width out of range");
    MK_REQUIRE(source != target, MK_ERR_INVALID, "mk_hessian_reversed: source and target must not alias");
    ReverseArgs a{source, target, order, addend, width};
    hipLaunchKernelGGL(reversed_matrix_kernel, dim3(mk_cdiv(width, 1024), width), dim3(256), 0, stream, a);
    MK_LAUNCH_CHECK("mk_hessian_reversed");
    return MK_OK;
}

extern "C" int mk_unit_upper_from_factor(const float *factor, float *out, int width, void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MK_REQUIRE(factor && out, MK_ERR_INVALID, "mk_unit_upper_from_factor: null pointer");
    MK_REQUIRE(width >= 1 && width <= 65535 * 32, MK_ERR_INVALID, "mk_unit_upper_from_factor: width out of range");
    MK_REQUIRE(factor != out, MK_ERR_INVALID, "mk_unit_upper_from_factor: factor and out must not alias");
    hipLaunchKernelGGL(unit_upper_kernel, dim3(mk_cdiv(width, 32), mk_cdiv(width, 32)), dim3(256), 0, stream, factor, out, width);
    MK_LAUNCH_CHECK("mk_unit_upper_from_factor");
    return MK_OK;
}

extern "C" int mk_blocks_upper_from_factor(const float *factor, float *out, int width, int step, void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MK_REQUIRE(factor && out, MK_ERR_INVALID, "mk_blocks_upper_from_factor: null pointer");
    MK_REQUIRE(step == 2 || step == 4 || step == 8 || step == 16, MK_ERR_UNSUPPORTED,
               "mk_blocks_upper_from_factor: steps of 2, 4, 8 or 16 columns (got %d)", step);
    MK_REQUIRE(width >= step && width % step == 0 && width <= 65535 * 64, MK_ERR_INVALID,
               "mk_blocks_upper_from_factor: the width must hold whole steps");
    MK_REQUIRE(factor != out, MK_ERR_INVALID, "mk_blocks_upper_from_factor: factor and out must not alias");
    const dim3 grid(mk_cdiv(width, 64), mk_cdiv(width, 64)), block(256);
    if (step == 2) hipLaunchKernelGGL(blocks_upper_kernel<2>, grid, block, 0, stream, factor, out, width);
    else if (step == 4) hipLaunchKernelGGL(blocks_upper_kernel<4>, grid, block, 0, stream, factor, out, width);
    else if (step == 8) hipLaunchKernelGGL(blocks_upper_kernel<8>, grid, block, 0, stream, factor, out, width);
    else hipLaunchKernelGGL(blocks_upper_kernel<16>, grid, block, 0, stream, factor, out, width);
    MK_LAUNCH_CHECK("mk_blocks_upper_from_factor");
    return MK_OK;
}

namespace {

int check_block(const float *matrix, long long leading, int size, int first_column, int row_columns, const float *factor_out,
                const int *status) {
    MK_REQUIRE(matrix && status, MK_ERR_INVALID, "mk_cholesky_block: null pointer");
    MK_REQUIRE(size >= 1 && size <= kBlock, MK_ERR_UNSUPPORTED, "mk_cholesky_block: blocks of 1 to %d rows (got %d)", kBlock, size);
    MK_REQUIRE(row_columns >= 0 && leading >= static_cast<long long>(size) + row_columns && first_column >= 0, MK_ERR_INVALID,
               "mk_cholesky_block: rows overlap");
    MK_REQUIRE(leading <= (1ll << 32) / kBlock, MK_ERR_INVALID, "mk_cholesky_block: a block's rows must lie within 2^32 floats");
    MK_REQUIRE(row_columns == 0 || factor_out, MK_ERR_INVALID,
               "mk_cholesky_block: a block row needs a separate place for the factor");
    return MK_OK;
}

}  // namespace

extern "C" int mk_cholesky_block(float *matrix, long long leading, int size, int first_column, int row_columns,
                                 float *factor_out, int *status, void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (int refused = check_block(matrix, leading, size, first_column, row_columns, factor_out, status)) return refused;
    BlockArgs a{matrix, leading, size, first_column, status, row_columns, factor_out};
    if (row_columns > 0)
        hipLaunchKernelGGL((cholesky_block_kernel<true, false>), dim3(mk_cdiv(row_columns, kCarried)), dim3(2 * kThreads), 0, stream, a);
    else
        hipLaunchKernelGGL((cholesky_block_kernel<false, false>), dim3(1), dim3(2 * kThreads), 0, stream, a);
    MK_LAUNCH_CHECK("mk_cholesky_block");
    return MK_OK;
}

extern "C" int mk_cholesky_block_pairs(float *matrix, long long leading, int size, int first_column, int row_columns,
                                 float *factor_out, int *status, void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (int refused = check_block(matrix, leading, size, first_column, row_columns, factor_out, status)) return refused;
    BlockArgs a{matrix, leading, size, first_column, status, row_columns, factor_out};
    if (row_columns > 0)
        hipLaunchKernelGGL((cholesky_block_kernel<true, true>), dim3(mk_cdiv(row_columns, kCarried)), dim3(2 * kThreads), 0, stream, a);
    else
        hipLaunchKernelGGL((cholesky_block_kernel<false, true>), dim3(1), dim3(2 * kThreads), 0, stream, a);
    MK_LAUNCH_CHECK("mk_cholesky_block_pairs");
    return MK_OK;
}
