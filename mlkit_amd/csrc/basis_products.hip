// The dense half of the blocked transform on gfx950, for bases that do not fit a wavefront's registers: every row of `order`
// blocks of `power` values is multiplied, block by block, by a dense [order, order] basis.
//
// Covers the basis product of structured_transform (quantization/operations/orthogonal_transforms.py:101-109 of the
// reference) for bases of more than 32 rows, through mk_basis_mix (hadamard.hip) up to 256.

#include "mk_common.h"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

struct ProductArgs {
    const float *source;
    float *target;
    const float *basis;   // [order, order] row-major
    const float *signs_after;
    long long rows;
    int order, log_power, transpose;
    int row_tiles;        // tiles of the basis' rows
    long long column_tiles;
};

constexpr int kThreads = 256;
constexpr int kMaxOrder = 8192;
constexpr int kChainOrder = 256;         // bases up to here keep one chain of multiply-adds (the bits of a thread per column)
constexpr long long kShortLaunch = 256;  // workgroups of 128 x 128 values

// target[r, f', p] = sum_f mix[f', f] source[r, f, p] as a matrix product: f' down, f along the sum, the pairs (r, p) across.
// A workgroup of four wavefronts (SUB x SUB products of 32 x 32 x 2 each, DOWN of the wavefronts one below the other) owns 64 x 64,
// 64 x 256 or 128 x 128 of them; DEPTH f at a time go through LDS, the next ones on their way in registers.  A chunk's blocks of one r lie side by side in memory,
// whatever the power, and threads take them in that order.  Sums run over ascending f from zero, the fused multiply-add chain
// of the kernels for smaller bases bit for bit.  PARTIAL: 64 f at a time, their sums added up behind that, for bases of more than
// kChainOrder rows, whose rounding would otherwise grow with the chain (380 rows: 3.5e-7 from 64 bits, the library's product 1.8e-7
// to 3.5e-7; so 1.5e-7).
//
// The tiles of one pair of columns go to one XCD, whose L2 then has the source for all but the first of them.  Bound by memory
// for bases of up to about 100 rows, by the fp32 matrix cores beyond.  5120 rows as 44 blocks of 64: 44 us (114 with the basis
// in registers, 22 at copy rate); 3840 rows as 104 blocks of 8: 21 us and 4608 as 204 of 32: 190 us (64 TFLOP/s), against 620 us
// and 7.6 ms with a thread per column of blocks; 2048 rows as 1040 blocks of 8: 590 us (470 as one
// chain).
template <int SUB, int DOWN, int DEPTH, bool PARTIAL>
__global__ void __launch_bounds__(kThreads, 2) basis_product_kernel(const ProductArgs a) {
    constexpr int kRows = 32 * SUB * DOWN, kColumns = 32 * SUB * (4 / DOWN);
    constexpr int kLogDepth = DEPTH == 16 ? 4 : 5;
    static_assert(DEPTH == 1 << kLogDepth, "");
    constexpr int kLeftStride = kRows + 4, kRightStride = kColumns + 4;
    constexpr int kLeftLoads = DEPTH * kRows / kThreads, kRightLoads = DEPTH * kColumns / 4 / kThreads;
    __shared__ __align__(16) float left[2][DEPTH][kLeftStride], right[2][DEPTH][kRightStride];   // [f][f'], [f][(r, p)]
    const long long turn = blockIdx.x >> 3;
    const long long column_tile = turn / a.row_tiles * 8 + (blockIdx.x & 7);
    const int row_tile = static_cast<int>(turn % a.row_tiles);
    if (column_tile >= a.column_tiles) return;   // whole workgroups
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int out0 = row_tile * kRows;
    const long long column0 = column_tile * kColumns;
    const int wave_row = (wave % DOWN) * 32 * SUB, wave_column = (wave / DOWN) * 32 * SUB;
    const int log_piece = min(a.log_power, 31 - __builtin_clz(kColumns));   // values of a block inside the tile
    const long long row_size = static_cast<long long>(a.order) << a.log_power;

    // This thread's quads of a chunk: value 4 * quad of block f of row r.
    const float *right_source[kRightLoads];
    int right_block[kRightLoads], right_slot[kRightLoads];
#pragma unroll
    for (int i = 0; i < kRightLoads; ++i) {
        const int q = i * kThreads + static_cast<int>(threadIdx.x);
        const int local_row = q >> (log_piece - 2 + kLogDepth), block = (q >> (log_piece - 2)) & (DEPTH - 1), quad = q & ((1 << (log_piece - 2)) - 1);
        const int across = (local_row << log_piece) + 4 * quad;
        const long long column = column0 + across;
        long long row = column >> a.log_power;
        if (row >= a.rows) row = a.rows - 1;   // past the end: numbers that nobody writes out
        right_source[i] = a.source + row * row_size + (column & ((1ll << a.log_power) - 1)) + (static_cast<long long>(block) << a.log_power);
        right_block[i] = block;
        right_slot[i] = block * kRightStride + across;
    }
    float left_held[kLeftLoads];
    float4 right_held[kRightLoads];
    auto left_at = [&](int i, int &f, int &out) __attribute__((always_inline)) {   // threads along the basis' rows as they lie
        const int flat = i * kThreads + static_cast<int>(threadIdx.x);
        f = a.transpose ? flat / kRows : flat % DEPTH;
        out = a.transpose ? flat % kRows : flat / DEPTH;
    };
    auto fetch = [&](int first) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kRightLoads; ++i) {
            const bool inside = first + right_block[i] < a.order;
            right_held[i] = *reinterpret_cast<const float4 *>(right_source[i] + (static_cast<long long>(inside ? first : -right_block[i]) << a.log_power));
            if (!inside) right_held[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);   // (block 0 read instead)
        }
#pragma unroll
        for (int i = 0; i < kLeftLoads; ++i) {
            int f, out;
            left_at(i, f, out);
            const bool inside = first + f < a.order && out0 + out < a.order;
            const int at = a.transpose ? (first + f) * a.order + out0 + out : (out0 + out) * a.order + first + f;
            const float held = a.basis[inside ? at : 0];
            left_held[i] = inside ? held : 0.0f;
        }
    };
    auto keep = [&](int buffer) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kRightLoads; ++i) *reinterpret_cast<float4 *>(&right[buffer][0][0] + right_slot[i]) = right_held[i];
#pragma unroll
        for (int i = 0; i < kLeftLoads; ++i) {
            int f, out;
            left_at(i, f, out);
            left[buffer][f][out] = left_held[i];
        }
    };
    f32x16 sums[SUB][SUB], totals[PARTIAL ? SUB : 1][SUB];
    auto clear = [](auto &tiles) __attribute__((always_inline)) {
        for (auto &row : tiles)
            for (f32x16 &tile : row) tile = f32x16{};
    };
    clear(sums);
    clear(totals);
    fetch(0);
    keep(0);
    __syncthreads();
    // Product i takes rows SUB l + i of the wavefront's, l = lane % 32: a lane's operands lie side by side.
    struct alignas(4 * SUB) Values {
        float of[SUB];
    };
    const int left_read = (lane >> 5) * kLeftStride + wave_row + SUB * (lane & 31), right_read = (lane >> 5) * kRightStride + wave_column + SUB * (lane & 31);
    for (int first = 0, buffer = 0; first < a.order; first += DEPTH, buffer ^= 1) {
        const bool more = first + DEPTH < a.order;   // uniform
        if (more) fetch(first + DEPTH);
        const float *left_rows = &left[buffer][0][0] + left_read, *right_rows = &right[buffer][0][0] + right_read;
#pragma unroll
        for (int k = 0; k < DEPTH; k += 2) {
            const Values l = *reinterpret_cast<const Values *>(left_rows + k * kLeftStride), r = *reinterpret_cast<const Values *>(right_rows + k * kRightStride);
#pragma unroll
            for (int i = 0; i < SUB; ++i)
#pragma unroll
                for (int j = 0; j < SUB; ++j) sums[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(l.of[i], r.of[j], sums[i][j], 0, 0, 0);
        }
        if constexpr (PARTIAL) {
            if (((first + DEPTH) & 63) == 0 || !more) {   // uniform
#pragma unroll
                for (int i = 0; i < SUB; ++i)
#pragma unroll
                    for (int j = 0; j < SUB; ++j) totals[i][j] += sums[i][j];
                clear(sums);
            }
        }
        if (more) keep(buffer ^ 1);
        __syncthreads();
    }
    // Value r of product (i, j): row SUB (8 (r / 4) + 4 (lane / 32) + r % 4) + i, column SUB (lane % 32) + j.
    const long long column = column0 + wave_column + SUB * (lane & 31);
    const long long row = column >> a.log_power;
    if (row >= a.rows) return;
    const int p = static_cast<int>(column & ((1ll << a.log_power) - 1));   // a multiple of SUB, as the power is
    float *target = a.target + row * row_size + p;
#pragma unroll
    for (int i = 0; i < SUB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int out = out0 + wave_row + SUB * ((r >> 2) * 8 + (lane >> 5) * 4 + (r & 3)) + i;
            if (out >= a.order) continue;
            Values value;
#pragma unroll
            for (int j = 0; j < SUB; ++j) value.of[j] = PARTIAL ? totals[PARTIAL ? i : 0][j][r] : sums[i][j][r];
            if (a.signs_after) {   // uniform
                const Values sign = *reinterpret_cast<const Values *>(a.signs_after + (static_cast<long long>(out) << a.log_power) + p);
#pragma unroll
                for (int j = 0; j < SUB; ++j) value.of[j] *= sign.of[j];
            }
            *reinterpret_cast<Values *>(target + (static_cast<long long>(out) << a.log_power)) = value;
        }
}

template <int SUB, int DOWN, int DEPTH>
int launch(ProductArgs a, hipStream_t stream) {
    constexpr int kRows = 32 * SUB * DOWN, kColumns = 32 * SUB * (4 / DOWN);
    a.row_tiles = mk_cdiv(a.order, kRows);
    a.column_tiles = ((a.rows << a.log_power) + kColumns - 1) / kColumns;
    const long long groups = (a.column_tiles + 7) / 8 * 8 * a.row_tiles;
    MK_REQUIRE(groups < (1ll << 31), MK_ERR_UNSUPPORTED, "mk_basis_mix: too many rows");
    if (a.order > kChainOrder)
        hipLaunchKernelGGL((basis_product_kernel<SUB, DOWN, DEPTH, true>), dim3(static_cast<unsigned>(groups)), dim3(kThreads), 0, stream, a);
    else
        hipLaunchKernelGGL((basis_product_kernel<SUB, DOWN, DEPTH, false>), dim3(static_cast<unsigned>(groups)), dim3(kThreads), 0, stream, a);
    return MK_OK;
}

}  // namespace

int mk_basis_product_launch(const float *source, float *target, const float *basis, long long rows, int order, int log_power, int transpose,
                            const float *signs_after, hipStream_t stream) {
    const ProductArgs a{source, target, basis, signs_after, rows, order, log_power, transpose, 0, 0};
    // A launch that leaves most of the GPU idle waits for memory once per chunk: small tiles, deep chunks (19 rows as 380 blocks
    // of 16: 24 us, 50 on the large tiles; 512 as 108 of 16: 11 and 21; from 256 large tiles on both take as long).
    if (((rows << log_power) + 127) / 128 * mk_cdiv(order, 128) <= kShortLaunch) return launch<1, 2, 32>(a, stream);
    if (order <= 64) return launch<2, 1, 16>(a, stream);
    return launch<2, 2, 16>(a, stream);
}

extern "C" int mk_basis_product(const float *source, float *target, const float *basis, long long rows, int order, int power,
                                int transpose, const float *signs_after, void *stream_) {
    MK_REQUIRE(rows >= 0 && order >= 1 && power >= 1, MK_ERR_INVALID, "mk_basis_product: sizes must be positive");
    MK_REQUIRE(order <= kMaxOrder, MK_ERR_UNSUPPORTED, "mk_basis_product: basis order %d exceeds %d", order, kMaxOrder);
    MK_REQUIRE(power >= 4 && (power & (power - 1)) == 0, MK_ERR_UNSUPPORTED, "mk_basis_product: blocks of a power of two of at least 4 values");
    if (rows == 0) return MK_OK;
    MK_REQUIRE(source && target && basis, MK_ERR_INVALID, "mk_basis_product: null tensor pointer");
    MK_REQUIRE(source != target, MK_ERR_INVALID, "mk_basis_product: source and target must not alias");
    MK_REQUIRE(((reinterpret_cast<uintptr_t>(source) | reinterpret_cast<uintptr_t>(target) | reinterpret_cast<uintptr_t>(signs_after)) & 15u) == 0,
               MK_ERR_UNSUPPORTED, "mk_basis_product: tensors must be 16-byte aligned");
    int log_power = 0;
    while ((1 << log_power) < power) ++log_power;
    if (int status = mk_basis_product_launch(source, target, basis, rows, order, log_power, transpose, signs_after, static_cast<hipStream_t>(stream_)))
        return status;
    MK_LAUNCH_CHECK("mk_basis_product");
    return MK_OK;
}
