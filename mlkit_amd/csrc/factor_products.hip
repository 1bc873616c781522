// Products of the blocked Cholesky factorisation H = U^T U on gfx950: rows of the matrix lose U^T U over the rows of U that
// are finished.  Two shapes: one block of rows inside a panel (`mk_factor_block_rows`, short and wide), and everything behind
// a finished panel (`mk_factor_trailing`, square).
//
// Used by `feedback_coefficients` (quantization/algorithms/error_feedback.py:37-83 of the reference, which calls
// torch.linalg.cholesky_ex).

#include "mk_common.h"

#include <type_traits>

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kBlockRows = 128;
constexpr int kThreads = 256;

struct ProductArgs {
    float *matrix;   // row-major, `width` floats per row; rows k_first ... k_stop - 1 hold the finished U
    int width;
    int k_first, k_stop;
    int row_first, row_stop;   // rows that lose the products, from column `row_first` (block rows) or their own (trailing) on
};

// An element `bytes` behind a uniform pointer: the offset in 32 bits, so that an access takes a scalar base and one register.
template <typename T>
__device__ __forceinline__ T *element_at(T *uniform, uint32_t bytes) {
    using Byte = std::conditional_t<std::is_const_v<T>, const char, char>;
    return reinterpret_cast<T *>(reinterpret_cast<Byte *>(uniform) + bytes);
}

// ---- one block of rows ------------------------------------------------------------------------
//
// A[r][c] -= sum_k U[k][r] U[k][c], at most 128 rows r, every column c from the block's first on.  The block kernel in front
// and the one behind wait for this launch, so its own chain counts: a wavefront keeps 16 R x 16 C values and takes its operands
// straight from memory in the layout of the 16 x 16 x 4 product (four rows of U, 64 adjacent bytes of each), a stage of S
// products' operands ahead; with SPLIT the four wavefronts of a workgroup take a quarter of the k each and their sums meet in
// LDS.  Without, sums are one chain over ascending k (what the library's kernels compute, bit for bit).
//
// Bound by latency where the matrix is narrow: the three products of 896 columns 4.4 us each (library products 8, and 78 and 48
// where one workgroup was chosen); 14 us with 10880 columns beside 128 k.  32 x 64 values a workgroup from 4096 columns on, where
// the operands that all workgroups read together count (32 x 32 below: twice the workgroups, half their chain).
template <int R, int C, bool SPLIT, int S>
__global__ void __launch_bounds__(kThreads, 3) block_rows_kernel(const ProductArgs a) {
    __builtin_amdgcn_s_setprio(3);   // in front of a trailing update that runs beside it
    constexpr int kRows = 16 * R, kColumns = 16 * C;
    constexpr int kAcross = SPLIT ? 1 : 4;   // wavefronts of a workgroup side by side
    constexpr int kTileFloats = kRows * kColumns;
    __shared__ __align__(16) float partial[SPLIT ? 3 * kTileFloats : 4];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int along = lane & 15, quarter = lane >> 4;
    const int row0 = a.row_first + static_cast<int>(blockIdx.y) * kRows;
    const int column0 = a.row_first + (static_cast<int>(blockIdx.x) * kAcross + (SPLIT ? 0 : wave)) * kColumns;
    if (!SPLIT && column0 >= a.width) return;   // (no barrier follows)
    const int depth = SPLIT ? (a.k_stop - a.k_first) / 4 : a.k_stop - a.k_first;   // a multiple of 32
    const float *from = a.matrix + static_cast<size_t>(a.k_first + (SPLIT ? wave * depth : 0)) * a.width;   // uniform

    uint32_t left_at[R], right_at[C];   // of k = quarter; columns beyond the matrix are read from its last one
#pragma unroll
    for (int r = 0; r < R; ++r) left_at[r] = 4u * (static_cast<uint32_t>(quarter) * a.width + min(row0 + 16 * r + along, a.width - 1));
#pragma unroll
    for (int c = 0; c < C; ++c) right_at[c] = 4u * (static_cast<uint32_t>(quarter) * a.width + min(column0 + 16 * c + along, a.width - 1));

    f32x4 sums[R][C];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < C; ++c) sums[r][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    struct Stage {
        float left[S][R], right[S][C];
    };
    auto fetch = [&](int k, Stage &stage) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const float *rows = from + static_cast<size_t>(k + 4 * s) * a.width;
#pragma unroll
            for (int r = 0; r < R; ++r) stage.left[s][r] = *element_at(rows, left_at[r]);
#pragma unroll
            for (int c = 0; c < C; ++c) stage.right[s][c] = *element_at(rows, right_at[c]);
        }
    };
    auto multiply = [&](const Stage &stage) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int c = 0; c < C; ++c)
                    sums[r][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(stage.left[s][r], stage.right[s][c], sums[r][c], 0, 0, 0);
    };
    constexpr int kStage = 4 * S;
    Stage even, odd;
    fetch(0, even);
    for (int k = 0; k < depth; k += 2 * kStage) {
        const bool second = k + kStage < depth;   // uniform
        if (second) fetch(k + kStage, odd);
        __builtin_amdgcn_sched_barrier(0);
        multiply(even);
        if (!second) break;
        if (k + 2 * kStage < depth) fetch(k + 2 * kStage, even);
        __builtin_amdgcn_sched_barrier(0);
        multiply(odd);
    }

    // value i of a lane: row 4 quarter + i, column `along` of its 16 x 16 tile
    if constexpr (SPLIT) {
        // Wavefront w adds up tiles w, w + 4, ...: its own sums stay in registers, the others' come through LDS in the
        // order of the k they cover.
        auto slot = [&](int tile, int of) __attribute__((always_inline)) -> f32x4 * {   // `of`: 0 ... 2, the wavefronts other than the tile's
            return reinterpret_cast<f32x4 *>(partial + (of * R * C + tile) * 256) + lane;
        };
#pragma unroll
        for (int tile = 0; tile < R * C; ++tile)
            if (wave != (tile & 3)) *slot(tile, wave - (wave > (tile & 3) ? 1 : 0)) = sums[tile / C][tile % C];
        __syncthreads();
#pragma unroll
        for (int tile = 0; tile < R * C; ++tile) {
            if (wave != (tile & 3)) continue;   // uniform
            f32x4 total;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const f32x4 part = w == (tile & 3) ? sums[tile / C][tile % C] : *slot(tile, w - (w > (tile & 3) ? 1 : 0));
                total = w == 0 ? part : total + part;
            }
            const int column = column0 + 16 * (tile % C) + along;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = row0 + 16 * (tile / C) + 4 * quarter + i;
                if (row < a.row_stop && column < a.width) a.matrix[static_cast<size_t>(row) * a.width + column] -= total[i];
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int column = column0 + 16 * c + along;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int row = row0 + 16 * r + 4 * quarter + i;
                    if (row < a.row_stop && column < a.width) a.matrix[static_cast<size_t>(row) * a.width + column] -= sums[r][c][i];
                }
            }
    }
}

template <int R, int C, bool SPLIT, int S>
void launch_block_rows(const ProductArgs &a, hipStream_t stream) {
    const dim3 grid(mk_cdiv(a.width - a.row_first, 16 * C * (SPLIT ? 1 : 4)), mk_cdiv(a.row_stop - a.row_first, 16 * R));
    hipLaunchKernelGGL((block_rows_kernel<R, C, SPLIT, S>), grid, dim3(kThreads), 0, stream, a);
}

// ---- everything behind a panel ----------------------------------------------------------------
//
// A[r][c] -= sum_k U[k][r] U[k][c], c >= r, one chain over ascending k, on tiles of 64 SUB x 64 SUB: four wavefronts of
// SUB x SUB products of 32 x 32 x 2, both operands straight from memory into LDS, sixteen rows of U at a time in four buffers,
// so that a transfer has three chunks' time to land.  Tiles below the diagonal are not computed.  Eight tile rows go down a
// column of tiles before the next column, and an XCD takes neighbouring tiles: the 64 tiles that it works on at a time read 16
// operand panels, not 65.  VEC: rows start on 16-byte boundaries and move in 16-byte pieces, otherwise in single floats.
constexpr int kDepth = 16, kBuffers = 4, kBand = 8;
// Tiles of 128 x 128 from here on (two rounds of two per compute unit): fewer leave the GPU idle, or a last round nearly
// empty.  360 columns behind a panel of 1024: 22 us on 64 x 64 tiles, 75 on 128 x 128.
constexpr int kLargeTiles = 1024;
// Beyond the 64 KB of its buffers: one workgroup per compute unit, beside which a workgroup of the block kernel finds room.
// Without, block kernels wait for tiles to end: 11008 columns in 6.5 ms instead of 6.2, 8184 in 3.47 instead of 3.40.  (Tiles of
// 64 x 64 take 32 KB and end soon.)
constexpr size_t kRoomBeside = 20 * 1024;

struct TrailingArgs {
    ProductArgs product;
    int row_tiles, column_tiles;   // from row_first on
    int per_xcd;                   // tiles (those below the diagonal included) of an XCD
};

__device__ __forceinline__ void piece_to_lds(const float *source, float *target, std::true_type) {
    __builtin_amdgcn_global_load_lds(source, target, 16, 0, 0);   // lane l's 16 bytes at 16 l from the uniform LDS address
}
__device__ __forceinline__ void piece_to_lds(const float *source, float *target, std::false_type) {
    __builtin_amdgcn_global_load_lds(source, target, 4, 0, 0);
}

template <int SUB, bool VEC>
__global__ void __launch_bounds__(kThreads, 3) trailing_kernel(const TrailingArgs t) {
    constexpr int kTile = 64 * SUB;
    // Each buffer a variable of its own: the compiler then sees that a transfer into one cannot touch another that is read.
    // (The left operand's rows, then the right one's: with more than four variables it loses sight of some.)
    __shared__ __align__(16) float buffer0[2][kDepth][kTile], buffer1[2][kDepth][kTile], buffer2[2][kDepth][kTile], buffer3[2][kDepth][kTile];
    const ProductArgs &a = t.product;
    int index = static_cast<int>(blockIdx.x & 7) * t.per_xcd + static_cast<int>(blockIdx.x >> 3);
    int band = 0, tall = 0;
    for (;; ++band) {   // uniform; a band of tile rows starts at its own first column
        tall = min(kBand, t.row_tiles - band * kBand);
        if (tall <= 0) return;
        const int count = tall * (t.column_tiles - band * kBand);
        if (index < count) break;
        index -= count;
    }
    const int tile_column = band * kBand + index / tall, tile_row = band * kBand + index % tall;
    if (tile_column < tile_row) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = a.row_first + tile_row * kTile, column0 = a.row_first + tile_column * kTile;
    const int wave_row = (wave >> 1) * 32 * SUB, wave_column = (wave & 1) * 32 * SUB;

    // A wavefront moves rows 4 wave ... 4 wave + 3 of a chunk, a few per instruction or part of one.
    using Vec = std::bool_constant<VEC>;
    constexpr int kPiece = VEC ? 4 : 1, kLanes = VEC ? kTile / 4 : 64, kParts = VEC ? 1 : SUB, kRowsAtOnce = 64 / kLanes;
    constexpr int kTransfers = 4 / kRowsAtOnce * kParts * 2;   // a wavefront's per chunk
    uint32_t left_lane[kParts], right_lane[kParts];
#pragma unroll
    for (int part = 0; part < kParts; ++part) {
        const int along = part * 64 + (lane & (kLanes - 1)) * kPiece;
        const uint32_t down = static_cast<uint32_t>(lane / kLanes) * a.width;
        left_lane[part] = 4u * (down + min(row0 + along, a.width - kPiece));   // (beyond the matrix: its last values, not used)
        right_lane[part] = 4u * (down + min(column0 + along, a.width - kPiece));
    }
    const float *panel = a.matrix + static_cast<size_t>(a.k_first + 4 * wave) * a.width;
    auto fetch = [&](int chunk, float (&buffer)[2][kDepth][kTile]) __attribute__((always_inline)) {
        const float *rows = panel + static_cast<size_t>(chunk) * kDepth * a.width;
#pragma unroll
        for (int one = 0; one < 4; one += kRowsAtOnce)
#pragma unroll
            for (int part = 0; part < kParts; ++part) {
                piece_to_lds(element_at(rows + static_cast<size_t>(one) * a.width, left_lane[part]), &buffer[0][4 * wave + one][64 * part], Vec{});
                piece_to_lds(element_at(rows + static_cast<size_t>(one) * a.width, right_lane[part]), &buffer[1][4 * wave + one][64 * part], Vec{});
            }
    };
    f32x16 sums[SUB][SUB];
#pragma unroll
    for (int i = 0; i < SUB; ++i)
#pragma unroll
        for (int j = 0; j < SUB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) sums[i][j][r] = 0.0f;
    // Product i takes rows SUB l + i of the wavefront's, l = lane % 32: a lane's operands lie side by side.
    struct alignas(4 * SUB) Operands {
        float of[SUB];
    };
    const uint32_t left_read = (lane >> 5) * kTile + wave_row + SUB * (lane & 31), right_read = (lane >> 5) * kTile + wave_column + SUB * (lane & 31);
    const int chunks = (a.k_stop - a.k_first) / kDepth;   // a multiple of four
    // `behind`: chunks that follow, three or more as three.  The transfers of two of them may still be under way.
    auto advance = [&](int chunk, auto behind, const float (&buffer)[2][kDepth][kTile], float (&last_read)[2][kDepth][kTile]) __attribute__((always_inline)) {
        constexpr int kUnderWay = (behind.value < 2 ? behind.value : 2) * kTransfers;
        static_assert(kUnderWay < 64, "the counter's range");
        __builtin_amdgcn_s_waitcnt(0x0f70 | (kUnderWay & 15) | ((kUnderWay >> 4) << 14));   // vmcnt (bits 0 ... 3 and 14 ... 15) alone
        // landed for every wavefront, and the buffer written next has been read by all (their products took the operands).
        // The bare instruction: __syncthreads would wait for the transfers under way.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if constexpr (behind.value == 3) fetch(chunk + 3, last_read);
        const float *left_rows = &buffer[0][0][0] + left_read, *right_rows = &buffer[1][0][0] + right_read;
        auto operands = [](const float *at) __attribute__((always_inline)) { return *reinterpret_cast<const Operands *>(at); };
        Operands left = operands(left_rows), right = operands(right_rows);
#pragma unroll
        for (int k = 0; k < kDepth; k += 2) {   // the next operands are requested in front of the products
            const int next = k + 2 < kDepth ? k + 2 : k;
            const Operands next_left = operands(left_rows + next * kTile), next_right = operands(right_rows + next * kTile);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < SUB; ++i)
#pragma unroll
                for (int j = 0; j < SUB; ++j) sums[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(left.of[i], right.of[j], sums[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            left = next_left, right = next_right;
        }
    };
    fetch(0, buffer0);
    fetch(1, buffer1);
    fetch(2, buffer2);
    using More = std::integral_constant<int, 3>;
    int chunk = 0;
    for (; chunk + 4 < chunks; chunk += 4) {
        advance(chunk, More{}, buffer0, buffer3);
        advance(chunk + 1, More{}, buffer1, buffer0);
        advance(chunk + 2, More{}, buffer2, buffer1);
        advance(chunk + 3, More{}, buffer3, buffer2);
    }
    advance(chunk, More{}, buffer0, buffer3);
    advance(chunk + 1, std::integral_constant<int, 2>{}, buffer1, buffer0);
    advance(chunk + 2, std::integral_constant<int, 1>{}, buffer2, buffer1);
    advance(chunk + 3, std::integral_constant<int, 0>{}, buffer3, buffer2);

    // Value r of product (i, j): row SUB (8 (r / 4) + 4 (lane / 32) + r % 4) + i, column SUB (lane % 32) + j.
    float *corner = a.matrix + static_cast<size_t>(row0 + wave_row) * a.width + column0 + wave_column;
    const uint32_t cell = 4u * SUB * (static_cast<uint32_t>((lane >> 5) * 4) * a.width + (lane & 31));
    const int rows_left = a.row_stop - row0 - wave_row - SUB * (lane >> 5) * 4, columns_left = a.width - column0 - wave_column - SUB * (lane & 31);
    const auto finish = [&](auto whole) __attribute__((always_inline)) {
        // a row's SUB adjacent values together where they are all there and lie on their alignment
        constexpr int kTogether = whole.value && VEC ? SUB : 1;
        struct alignas(4 * kTogether) Values {
            float of[kTogether];
        };
#pragma unroll
        for (int i = 0; i < SUB; ++i)
#pragma unroll
            for (int first = 0; first < 16; first += 8) {
                Values held[8][SUB / kTogether];
                auto at = [&](int r, int j) __attribute__((always_inline)) -> Values * {
                    return reinterpret_cast<Values *>(element_at(corner + static_cast<size_t>(SUB * ((r >> 2) * 8 + (r & 3)) + i) * a.width + j, cell));
                };
                auto present = [&](int r, int j) __attribute__((always_inline)) -> bool {
                    return whole.value || (SUB * ((r >> 2) * 8 + (r & 3)) + i < rows_left && j < columns_left);
                };
#pragma unroll
                for (int r = 0; r < 8; ++r)
#pragma unroll
                    for (int j = 0; j < SUB; j += kTogether)
                        if (present(first + r, j)) held[r][j / kTogether] = *at(first + r, j);
#pragma unroll
                for (int r = 0; r < 8; ++r)
#pragma unroll
                    for (int j = 0; j < SUB; j += kTogether)
                        if (present(first + r, j)) {
                            Values &now = held[r][j / kTogether];
#pragma unroll
                            for (int of = 0; of < kTogether; ++of) now.of[of] -= sums[i][j + of][first + r];
                            *at(first + r, j) = now;
                        }
            }
    };
    if (row0 + kTile <= a.row_stop && column0 + kTile <= a.width) finish(std::true_type{});   // uniform
    else finish(std::false_type{});
}

// `lds`: bytes that a workgroup asks for beyond its buffers.
template <int SUB>
void launch_trailing(const ProductArgs &a, size_t lds, hipStream_t stream) {
    constexpr int kTile = 64 * SUB;
    TrailingArgs t{a, mk_cdiv(a.row_stop - a.row_first, kTile), mk_cdiv(a.width - a.row_first, kTile), 0};
    int tiles = 0;
    for (int band = 0; band * kBand < t.row_tiles; ++band)
        tiles += (t.row_tiles - band * kBand < kBand ? t.row_tiles - band * kBand : kBand) * (t.column_tiles - band * kBand);
    t.per_xcd = mk_cdiv(tiles, 8);
    const bool pieces = a.width % 4 == 0 && a.row_first % 4 == 0 && (reinterpret_cast<uintptr_t>(a.matrix) & 15u) == 0;
    if (pieces) hipLaunchKernelGGL((trailing_kernel<SUB, true>), dim3(8 * t.per_xcd), dim3(kThreads), lds, stream, t);
    else hipLaunchKernelGGL((trailing_kernel<SUB, false>), dim3(8 * t.per_xcd), dim3(kThreads), lds, stream, t);
}

int check_product(const char *name, const float *matrix, int width, int k_first, int k_stop, int row_first, int row_stop, int depth_unit) {
    MK_REQUIRE(matrix, MK_ERR_INVALID, "%s: null pointer", name);
    MK_REQUIRE(k_first >= 0 && k_first < k_stop && k_stop <= row_first && row_first < row_stop && row_stop <= width, MK_ERR_INVALID,
               "%s: rows [%d, %d) must lie behind rows [%d, %d) of %d", name, row_first, row_stop, k_first, k_stop, width);
    MK_REQUIRE((k_stop - k_first) % depth_unit == 0, MK_ERR_UNSUPPORTED, "%s: products over multiples of %d rows (got %d)", name, depth_unit,
               k_stop - k_first);
    MK_REQUIRE(width <= (1 << 24), MK_ERR_UNSUPPORTED, "%s: at most 2^24 columns", name);
    return MK_OK;
}

}  // namespace

extern "C" int mk_factor_block_rows(float *matrix, int width, int k_first, int k_stop, int row_first, int row_stop, int one_chain,
                                    void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (int refused = check_product("mk_factor_block_rows", matrix, width, k_first, k_stop, row_first, row_stop, kBlockRows)) return refused;
    MK_REQUIRE(row_stop - row_first <= kBlockRows, MK_ERR_UNSUPPORTED, "mk_factor_block_rows: at most %d rows", kBlockRows);
    const ProductArgs a{matrix, width, k_first, k_stop, row_first, row_stop};
    if (one_chain) launch_block_rows<1, 1, false, 8>(a, stream);
    else if (width - row_first <= 4096) launch_block_rows<2, 2, true, 4>(a, stream);
    else launch_block_rows<2, 4, true, 2>(a, stream);
    MK_LAUNCH_CHECK("mk_factor_block_rows");
    return MK_OK;
}

extern "C" int mk_factor_trailing(float *matrix, int width, int k_first, int k_stop, int row_first, int row_stop, int leave_room,
                                  void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (int refused = check_product("mk_factor_trailing", matrix, width, k_first, k_stop, row_first, row_stop, kBuffers * kDepth)) return refused;
    const long long row_tiles = (row_stop - row_first + 127) / 128, column_tiles = (width - row_first + 127) / 128;
    MK_REQUIRE(row_tiles * column_tiles < (1ll << 26), MK_ERR_UNSUPPORTED, "mk_factor_trailing: too many tiles");
    const ProductArgs a{matrix, width, k_first, k_stop, row_first, row_stop};
    if (row_tiles * (2 * column_tiles - row_tiles + 1) / 2 < kLargeTiles) launch_trailing<1>(a, 0, stream);
    else launch_trailing<2>(a, leave_room ? kRoomBeside : 0, stream);
    MK_LAUNCH_CHECK("mk_factor_trailing");
    return MK_OK;
}
