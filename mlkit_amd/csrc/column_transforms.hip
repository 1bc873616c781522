// Transforms down the columns of a weight, and what goes with them: the Walsh-Hadamard transform of every column without
// turning the matrix, turning a matrix (and converting it to FP32 on the way), and the signs of a seeded rotation.
//
// Covers quantization/algorithms/incoherence.py:56-98 and formats/composition.py:14-47 of the reference, which
// rotate the output side of a weight as `rotate(w.T.contiguous()).T`.

#include "mk_common.h"

namespace {

// ---- columns --------------------------------------------------------------------------------

struct ColumnArgs {
    const void *source;
    float *target;
    const float *signs_before, *signs_after;   // of the rows, or null
    int columns, groups, groups_per_xcd;
    float scale;
};

template <int COLUMNS, int GROUPS, int VALUES>
constexpr int kExchangeFloats = (VALUES * (GROUPS / 2) + GROUPS) * COLUMNS;   // half of a workgroup's values, padded

// The transform of GROUPS * VALUES rows.  Thread (c, g) first holds rows VALUES g + k of column c, k = 0 ... VALUES - 1, and
// does the stages over k in registers; through LDS it comes to hold VALUES / GROUPS of the k with all g, whose stages
// follow: ascending strides, as in the transform of rows, so that both give the same bits.  A matrix is read once and
// written once.  The exchange takes two turns so that a workgroup's values fit LDS and
// a thread its registers: in turn p a thread in half h of the groups puts half h ^ p of its k there and takes
// what it needs of the groups' half h ^ p, into the registers that came free.
//
// Up to 2048 rows bound by HBM.  Neighbouring workgroups share 128-byte lines, so they are given to one XCD, whose L2 has
// the line: workgroup b takes column group (b % 8) * groups_per_xcd + b / 8.
//
// 14336 columns of 1024 / 2048 / 4096 fp32 values, signs before or behind: 20 / 39 / 122 us (from bf16 17 / 33 / 108), against
// 63 + 63 us for torch's strided copies around the row transform at 1024, 119 + 119 at 2048 and 255 + 255 at 4096.  At 4096
// rows 16 columns a workgroup of 1024 threads, in 103 registers; 8 columns take 145 (each line of 128 bytes is then fetched by
// four workgroups), and 180 with two workgroups on a compute unit (their lines leave the L2 before the neighbours come).
// 41 KB of LDS at least keep a fourth workgroup away at 1024 rows for the same reason (22 us with it).  Signs before, read by
// every thread for itself instead of through LDS: 44 at 2048 rows, 127 at 4096.
//
// OFFSET: the type of a thread's byte offset, 32 bits wherever the matrix has fewer bytes.
template <int COLUMNS, int GROUPS, int VALUES, int SOURCE, typename OFFSET>
__global__ void __launch_bounds__(COLUMNS * GROUPS, 4) fwht_columns_kernel(const ColumnArgs a) {
    constexpr int kHeld = VALUES / GROUPS;         // the k of a thread behind the exchange
    constexpr int kHalf = VALUES / 2, kHalfGroups = GROUPS / 2;
    constexpr int kSignStride = GROUPS + 4;        // signs of one k, its groups side by side
    extern __shared__ __align__(16) float exchange[];
    constexpr int kElement = SOURCE == MK_F32 ? 4 : 2;
    constexpr int kSigns = VALUES / COLUMNS;       // a thread's share of the signs
    static_assert(VALUES * kSignStride <= kExchangeFloats<COLUMNS, GROUPS, VALUES> && GROUPS * (VALUES + 4) <= kExchangeFloats<COLUMNS, GROUPS, VALUES>,
                  "the signs take the exchange's place");
    const int group = static_cast<int>(blockIdx.x & 7) * a.groups_per_xcd + static_cast<int>(blockIdx.x >> 3);
    if (group >= a.groups) return;   // whole workgroups
    const int local = threadIdx.x & (COLUMNS - 1), g = threadIdx.x / COLUMNS;
    const int half = __builtin_amdgcn_readfirstlane(g / kHalfGroups);   // a wavefront's groups lie in one half
    const int column = group * COLUMNS + local;
    const bool inside = column < a.columns;
    const char *source = static_cast<const char *>(a.source);
    const OFFSET from = (static_cast<OFFSET>(g * VALUES) * a.columns + (inside ? column : a.columns - 1)) * kElement;
    float sign[kSigns];
    if (a.signs_before) {   // uniform
#pragma unroll
        for (int i = 0; i < kSigns; ++i) sign[i] = a.signs_before[threadIdx.x + i * COLUMNS * GROUPS];
    }
    float value[2][kHalf];   // [k / kHalf][k % kHalf]
#pragma unroll
    for (int k = 0; k < VALUES; ++k, source += static_cast<size_t>(a.columns) * kElement)   // (a uniform row and the thread's
        value[k / kHalf][k % kHalf] = mk_load_as_float(source + from, 0, SOURCE);           // offset: one address register)
    if (a.signs_before) {   // (through LDS: read by each thread for itself they are as many loads again)
#pragma unroll
        for (int i = 0; i < kSigns; ++i) {
            const int row = threadIdx.x + i * COLUMNS * GROUPS;
            exchange[row / VALUES * (VALUES + 4) + row % VALUES] = sign[i];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < VALUES; k += 4) {
            const float4 four = *reinterpret_cast<const float4 *>(exchange + g * (VALUES + 4) + k);
            const float along[4] = {four.x, four.y, four.z, four.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) value[(k + j) / kHalf][(k + j) % kHalf] *= along[j];
        }
        __syncthreads();   // the exchange takes their place
    }
    auto butterfly = [](float &first, float &second) __attribute__((always_inline)) {
        const float low = first, high = second;
        first = low + high;
        second = low - high;
    };
    auto turned_halves = [&]() __attribute__((always_inline)) {
        if (half)
#pragma unroll
            for (int i = 0; i < kHalf; ++i) {
                const float first = value[0][i];
                value[0][i] = value[1][i];
                value[1][i] = first;
            }
    };
#pragma unroll
    for (int stride = 1; stride < VALUES; stride *= 2)
#pragma unroll
        for (int k = 0; k < VALUES; ++k)
            if ((k & stride) == 0) butterfly(value[k / kHalf][k % kHalf], value[(k + stride) / kHalf][(k + stride) % kHalf]);
    // (a pad of a group's floats behind the k of one reader keeps the readers of a wavefront on different banks)
    auto slot = [&](int k, int in_half) __attribute__((always_inline)) -> int {
        return (k * kHalfGroups + k / kHeld + in_half) * COLUMNS + local;
    };
    turned_halves();
#pragma unroll
    for (int turn = 0; turn < 2; ++turn) {
        if (turn) __syncthreads();   // the turn before has been read
#pragma unroll
        for (int i = 0; i < kHalf; ++i) exchange[slot((half ^ turn) * kHalf + i, g & (kHalfGroups - 1))] = value[turn][i];
        __syncthreads();
#pragma unroll
        for (int m = 0; m < kHeld; ++m)
#pragma unroll
            for (int j = 0; j < kHalfGroups; ++j) value[turn][m * kHalfGroups + j] = exchange[slot(g * kHeld + m, j)];
    }
    turned_halves();
    // now [half of the groups][which of the thread's k, group within the half]
#pragma unroll
    for (int stride = 1; stride < kHalfGroups; stride *= 2)
#pragma unroll
        for (int i = 0; i < kHalf; ++i)
            if ((i & stride) == 0) {
                butterfly(value[0][i], value[0][i + stride]);
                butterfly(value[1][i], value[1][i + stride]);
            }
#pragma unroll
    for (int i = 0; i < kHalf; ++i) butterfly(value[0][i], value[1][i]);
#pragma unroll
    for (int i = 0; i < VALUES; ++i) value[i / kHalf][i % kHalf] *= a.scale;
    if (a.signs_after) {   // uniform; a thread's rows lie VALUES apart, their signs are turned to lie side by side
        __syncthreads();   // the exchange has been read
#pragma unroll
        for (int i = 0; i < kSigns; ++i) {
            const int row = threadIdx.x + i * COLUMNS * GROUPS;
            exchange[(row % VALUES) * kSignStride + row / VALUES] = a.signs_after[row];
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < kHalf; i += 4) {   // four groups of one k
                const float4 sign = *reinterpret_cast<const float4 *>(exchange + (g * kHeld + i / kHalfGroups) * kSignStride + h * kHalfGroups + i % kHalfGroups);
                const float along[4] = {sign.x, sign.y, sign.z, sign.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) value[h][i + j] *= along[j];
            }
    }
    if (!inside) return;
    const OFFSET to = (static_cast<OFFSET>(g * kHeld) * a.columns + column) * 4;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < kHeld; ++m) {
            char *target = reinterpret_cast<char *>(a.target) + (static_cast<size_t>(h * kHalfGroups) * VALUES + m) * a.columns * 4;
#pragma unroll
            for (int of = 0; of < kHalfGroups; ++of, target += static_cast<size_t>(VALUES) * a.columns * 4)
                *reinterpret_cast<float *>(target + to) = value[h][m * kHalfGroups + of];
        }
}

template <int COLUMNS, int GROUPS, int VALUES, int SOURCE, typename OFFSET>
void launch_columns_of(const ColumnArgs &a, hipStream_t stream) {
    constexpr size_t needed = kExchangeFloats<COLUMNS, GROUPS, VALUES> * sizeof(float), lds = needed < 41 * 1024 ? 41 * 1024 : needed;
    static const hipError_t allowed = hipFuncSetAttribute(reinterpret_cast<const void *>(&fwht_columns_kernel<COLUMNS, GROUPS, VALUES, SOURCE, OFFSET>),
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    static_cast<void>(allowed);   // a refusal shows in the launch
    hipLaunchKernelGGL((fwht_columns_kernel<COLUMNS, GROUPS, VALUES, SOURCE, OFFSET>), dim3(8 * a.groups_per_xcd), dim3(COLUMNS * GROUPS), lds, stream, a);
}

template <int COLUMNS, int GROUPS, int VALUES, int SOURCE>
void launch_columns(ColumnArgs a, hipStream_t stream) {
    a.groups = mk_cdiv(a.columns, COLUMNS);
    a.groups_per_xcd = mk_cdiv(a.groups, 8);
    if (4ull * GROUPS * VALUES * a.columns < (1ull << 32)) launch_columns_of<COLUMNS, GROUPS, VALUES, SOURCE, uint32_t>(a, stream);
    else launch_columns_of<COLUMNS, GROUPS, VALUES, SOURCE, uint64_t>(a, stream);
}

template <int SOURCE>
void launch_rows(const ColumnArgs &a, int rows, hipStream_t stream) {
    // 4096 rows: 16 columns a workgroup where half the compute units get one (3072 columns 22 us, 30 with 8; 1000: 18 and 14)
    if (rows == 1024) launch_columns<16, 32, 32, SOURCE>(a, stream);
    else if (rows == 2048) launch_columns<16, 32, 64, SOURCE>(a, stream);
    else if (a.columns >= 2048) launch_columns<16, 64, 64, SOURCE>(a, stream);
    else launch_columns<8, 64, 64, SOURCE>(a, stream);
}

// ---- turning a matrix -----------------------------------------------------------------------

struct TransposeArgs {
    const void *source;
    float *target;
    int rows, columns, tiles_across;
};

// 64 x 64 tiles through LDS, fp32 4096 x 14336 in 100 us (4.7 TB/s; torch's strided copy 255), from bf16 in 77 (320 with its
// conversion); reads and writes both move whole 16-byte pieces along rows where the sizes allow it (VEC).
template <int SOURCE, bool VEC>
__global__ void __launch_bounds__(256) transpose_kernel(const TransposeArgs a) {
    __shared__ float tile[64][65];
    const int tx = (threadIdx.x & 15) * 4, ty = threadIdx.x >> 4;
    const int row_tile = blockIdx.x / a.tiles_across, row0 = row_tile * 64, column0 = (blockIdx.x - row_tile * a.tiles_across) * 64;   // uniform
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int local = ty + 16 * j, row = min(row0 + local, a.rows - 1);
        const size_t base = static_cast<size_t>(row) * a.columns;
        if constexpr (VEC) {
            const size_t at = base + min(column0 + tx, a.columns - 4);   // past the edge: numbers that nobody writes out
            if constexpr (SOURCE == MK_F32) {
                const float4 four = *reinterpret_cast<const float4 *>(static_cast<const float *>(a.source) + at);
                tile[local][tx] = four.x; tile[local][tx + 1] = four.y; tile[local][tx + 2] = four.z; tile[local][tx + 3] = four.w;
            } else {
                const uint2 four = *reinterpret_cast<const uint2 *>(static_cast<const uint16_t *>(a.source) + at);
                const uint32_t word[2] = {four.x, four.y};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint16_t raw = static_cast<uint16_t>(word[i / 2] >> (16 * (i & 1)));
                    tile[local][tx + i] = SOURCE == MK_F16 ? static_cast<float>(__builtin_bit_cast(_Float16, raw)) : mk_bf16_to_float(raw);
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) tile[local][tx + i] = mk_load_as_float(a.source, base + min(column0 + tx + i, a.columns - 1), SOURCE);
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int local = ty + 16 * j, column = column0 + local, row = row0 + tx;
        if (column >= a.columns) continue;
        float *to = a.target + static_cast<size_t>(column) * a.rows + row;
        if constexpr (VEC) {
            if (row < a.rows) *reinterpret_cast<float4 *>(to) = make_float4(tile[tx][local], tile[tx + 1][local], tile[tx + 2][local], tile[tx + 3][local]);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (row + i < a.rows) to[i] = tile[tx + i][local];
        }
    }
}

template <int SOURCE>
void launch_transpose(const TransposeArgs &a, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>(a.tiles_across) * mk_cdiv(a.rows, 64));
    const bool whole = a.rows % 4 == 0 && a.columns % 4 == 0
                       && ((reinterpret_cast<uintptr_t>(a.source) | reinterpret_cast<uintptr_t>(a.target)) & 15u) == 0;
    if (whole) hipLaunchKernelGGL((transpose_kernel<SOURCE, true>), grid, dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((transpose_kernel<SOURCE, false>), grid, dim3(256), 0, stream, a);
}

// ---- signs ------------------------------------------------------------------------------------

// The hash works on 32 bits: every step is masked to them.
__global__ void __launch_bounds__(256) hash_signs_kernel(float *out, int width, uint32_t seed) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= width) return;
    uint32_t v = static_cast<uint32_t>(i) + seed;
    v = (v ^ (v >> 16)) * 0x45D9F3Bu;
    v = (v ^ (v >> 16)) * 0x45D9F3Bu;
    v ^= v >> 16;
    out[i] = v & 1u ? 1.0f : -1.0f;
}

}  // namespace

extern "C" int mk_fwht_columns(const void *source, int source_dtype, float *target, int rows, int columns,
                               const float *signs_before, const float *signs_after, float scale, void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MK_REQUIRE(rows == 1024 || rows == 2048 || rows == 4096, MK_ERR_UNSUPPORTED,
               "mk_fwht_columns: columns of 1024, 2048 or 4096 values, not %d", rows);
    MK_REQUIRE(columns >= 1, MK_ERR_INVALID, "mk_fwht_columns: sizes must be positive");
    MK_REQUIRE(source && target, MK_ERR_INVALID, "mk_fwht_columns: null tensor pointer");
    MK_REQUIRE(source != target, MK_ERR_INVALID, "mk_fwht_columns: source and target must not alias");
    MK_REQUIRE(mk_dtype_valid(source_dtype), MK_ERR_INVALID, "mk_fwht_columns: unknown dtype code");
    ColumnArgs a{source, target, signs_before, signs_after, columns, 0, 0, scale};
    if (source_dtype == MK_F32) launch_rows<MK_F32>(a, rows, stream);
    else if (source_dtype == MK_F16) launch_rows<MK_F16>(a, rows, stream);
    else launch_rows<MK_BF16>(a, rows, stream);
    MK_LAUNCH_CHECK("mk_fwht_columns");
    return MK_OK;
}

extern "C" int mk_transpose(const void *source, int source_dtype, float *target, int rows, int columns, void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MK_REQUIRE(rows >= 1 && columns >= 1, MK_ERR_INVALID, "mk_transpose: sizes must be positive");
    MK_REQUIRE((rows + 63ll) / 64 * ((columns + 63ll) / 64) < (1ll << 24), MK_ERR_UNSUPPORTED, "mk_transpose: too many tiles");
    MK_REQUIRE(source && target, MK_ERR_INVALID, "mk_transpose: null tensor pointer");
    MK_REQUIRE(source != target, MK_ERR_INVALID, "mk_transpose: source and target must not alias");
    MK_REQUIRE(mk_dtype_valid(source_dtype), MK_ERR_INVALID, "mk_transpose: unknown dtype code");
    TransposeArgs a{source, target, rows, columns, mk_cdiv(columns, 64)};
    if (source_dtype == MK_F32) launch_transpose<MK_F32>(a, stream);
    else if (source_dtype == MK_F16) launch_transpose<MK_F16>(a, stream);
    else launch_transpose<MK_BF16>(a, stream);
    MK_LAUNCH_CHECK("mk_transpose");
    return MK_OK;
}

extern "C" int mk_hash_signs(float *out, int width, unsigned int seed, void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MK_REQUIRE(out && width >= 1, MK_ERR_INVALID, "mk_hash_signs: a buffer of at least one value is required");
    hipLaunchKernelGGL(hash_signs_kernel, dim3(mk_cdiv(width, 256)), dim3(256), 0, stream, out, width, seed);
    MK_LAUNCH_CHECK("mk_hash_signs");
    return MK_OK;
}
