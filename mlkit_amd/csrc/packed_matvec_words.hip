// Packed matrix-vector products that the streaming and table kernels do not take: rows that are not whole chunks of 32 codes,
// and the last rows of a matrix that do not fill a tile.

#include "packed_matvec_impl.h"

namespace {

using mk_matvec::load_piece;
using mk_matvec::piece_code;
using mk_matvec::transposed_value_of_lane;
using mk_matvec::transposed_wave_sum;
using mk_matvec::WordArgs;
using mk_matvec::Words4;

constexpr int kRows = 4, kPiece = mk_matvec::kPieceCodes, kMaxWaves = 8;   // rows and codes of a lane's turn; wavefronts of a workgroup

template <int XT>
__device__ __forceinline__ void load_values(float (&value)[kPiece], const void *x, size_t index) {
    if constexpr (XT == MK_F32) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const Words4 four = reinterpret_cast<const Words4 *>(static_cast<const float *>(x) + index)[q];
#pragma unroll
            for (int i = 0; i < 4; ++i) value[4 * q + i] = __uint_as_float(four[i]);
        }
    } else {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const Words4 four = reinterpret_cast<const Words4 *>(static_cast<const uint16_t *>(x) + index)[q];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint16_t raw = static_cast<uint16_t>(four[i / 2] >> (16 * (i & 1)));
                value[8 * q + i] = XT == MK_F16 ? static_cast<float>(__builtin_bit_cast(_Float16, raw)) : mk_bf16_to_float(raw);
            }
        }
    }
}

// y[m, n] = sum_k (value of code[n, k] * scale (+ zero)) * x[m, k] (+ bias[n]), every weight worked out in fp32 and multiplied
// in fp32.  A team of `waves` wavefronts takes four rows; its lanes go along them in pieces of sixteen codes, which are whole bytes
// for every width and lie inside one scale group; a last piece that is not whole goes code by code.
//
// Bound by the work per code (four rows share the activations a lane converts).  One to three rows left over of a layer of 6656
// columns, which every second layer of this kind has (k and v projections of an odd number of rows): 67 us with a wavefront per
// row that read byte by byte and code by code.
template <int BITS, int XT, int M>
__global__ void __launch_bounds__(64 * kMaxWaves) words_kernel(const WordArgs a) {
    constexpr int kSums = kRows * M;
    __shared__ float table[256];
    __shared__ float partial[kMaxWaves][kSums];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int team = wave / a.waves, place = wave - team * a.waves;   // uniform
    const int teams = (blockDim.x >> 6) / a.waves;
    const int row0 = a.first_row + (static_cast<int>(blockIdx.x) * teams + team) * kRows;
    const int sample0 = blockIdx.y * M;
    if (!a.uniform) {
        for (int i = threadIdx.x; i < (1 << BITS); i += blockDim.x) table[i] = i < a.n_values ? a.values[i] : 0.0f;
        __syncthreads();
    }
    const uint8_t *row_codes[kRows];
    size_t row_scales[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        const size_t row = min(row0 + r, a.rows - 1);   // past the last row: a repeat that is not stored
        row_codes[r] = a.packed + row * a.row_bytes;
        row_scales[r] = row * a.groups;
    }
    size_t x_row[M];
#pragma unroll
    for (int m = 0; m < M; ++m) x_row[m] = static_cast<size_t>(min(sample0 + m, a.samples - 1)) * a.width;

    float sums[kSums];
#pragma unroll
    for (int i = 0; i < kSums; ++i) sums[i] = 0.0f;
    const int pieces = a.width / kPiece, stride = 64 * a.waves;
    for (int piece = 64 * place + lane; piece < pieces; piece += stride) {
        uint32_t words[kRows][mk_matvec::kPieceWords<BITS>];
        float scale[kRows], zero[kRows], weight[kRows][kPiece];
        const uint32_t group = a.pieces_per_group > 0 ? static_cast<uint32_t>(piece) / static_cast<uint32_t>(a.pieces_per_group) : 0;
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            load_piece<BITS>(words[r], row_codes[r] + static_cast<size_t>(piece) * (2 * BITS));
            scale[r] = mk_load_as_float(a.scales, row_scales[r] + group, a.scale_dtype);
            zero[r] = a.zeros ? mk_load_as_float(a.zeros, row_scales[r] + group, a.scale_dtype) : 0.0f;
        }
#pragma unroll
        for (int r = 0; r < kRows; ++r)
#pragma unroll
            for (int k = 0; k < kPiece; ++k) {
                const uint32_t code = piece_code<BITS>(words[r], k);
                const float value = a.uniform ? a.grid_min + static_cast<float>(code) * a.grid_step : table[code];   // uniform
                weight[r][k] = a.zeros ? value * scale[r] + zero[r] : value * scale[r];
            }
#pragma unroll
        for (int m = 0; m < M; ++m) {
            float value[kPiece];
            load_values<XT>(value, a.x, x_row[m] + static_cast<size_t>(piece) * kPiece);
#pragma unroll
            for (int k = 0; k < kPiece; ++k)
#pragma unroll
                for (int r = 0; r < kRows; ++r) sums[r * M + m] = __builtin_fmaf(weight[r][k], value[k], sums[r * M + m]);
        }
    }
    if (place == 0 && lane < a.width - pieces * kPiece) {   // the last piece, a code per lane
        const int k = pieces * kPiece + lane, bit = k * BITS;
        const size_t group = a.pieces_per_group > 0 ? pieces / a.pieces_per_group : 0;
        float value[M];
#pragma unroll
        for (int m = 0; m < M; ++m) value[m] = mk_load_as_float(a.x, x_row[m] + k, XT);
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            const uint8_t *from = row_codes[r] + (bit >> 3);
            uint32_t word = from[0];
            if ((bit & 7) + BITS > 8) word |= static_cast<uint32_t>(from[1]) << 8;
            const uint32_t code = (word >> (bit & 7)) & ((1u << BITS) - 1u);
            float weight = a.uniform ? a.grid_min + static_cast<float>(code) * a.grid_step : table[code];
            weight *= mk_load_as_float(a.scales, row_scales[r] + group, a.scale_dtype);
            if (a.zeros) weight += mk_load_as_float(a.zeros, row_scales[r] + group, a.scale_dtype);
#pragma unroll
            for (int m = 0; m < M; ++m) sums[r * M + m] = __builtin_fmaf(weight, value[m], sums[r * M + m]);
        }
    }
    transposed_wave_sum<kSums>(sums, lane);
    float total = sums[0];
    const int index = transposed_value_of_lane<kSums>(lane);   // lanes below kSums: every value once
    if (a.waves > 1) {   // uniform
        if (lane < kSums) partial[wave][index] = total;
        __syncthreads();
        if (place != 0) return;
        total = 0.0f;
        for (int w = 0; w < a.waves; ++w) total += partial[wave + w][index];
    }
    const int row = row0 + index / M, sample = sample0 + index % M;
    if (lane >= kSums || row >= a.rows || sample >= a.samples) return;
    if (a.bias) total += mk_load_as_float(a.bias, row, a.bias_dtype);
    mk_store_from_float(a.y, static_cast<size_t>(sample) * a.rows + row, XT, total);
}

template <int BITS, int XT, int M>
void launch(const WordArgs &args, hipStream_t stream) {
    WordArgs a = args;
    const int pieces = a.width / kPiece, quads = mk_cdiv(a.rows - a.first_row, kRows);
    // As many wavefronts to four rows as the pieces keep busy; eight only where a compute unit has no other rows to work on.
    a.waves = pieces <= 64 ? 1 : pieces <= 128 ? 2 : 4;
    if (pieces > 256 && static_cast<long long>(quads) * mk_cdiv(a.samples, M) <= 512) a.waves = kMaxWaves;
    const int waves = a.waves > 4 ? a.waves : quads * a.waves < 4 ? quads * a.waves : 4;
    const dim3 grid(mk_cdiv(quads, waves / a.waves), mk_cdiv(a.samples, M));
    hipLaunchKernelGGL((words_kernel<BITS, XT, M>), grid, dim3(64 * waves), 0, stream, a);
}

template <int BITS, int XT>
void with_samples(const WordArgs &a, hipStream_t stream) {
    if (a.samples == 1) launch<BITS, XT, 1>(a, stream);
    else if (a.samples == 2) launch<BITS, XT, 2>(a, stream);
    else if (a.samples <= 4) launch<BITS, XT, 4>(a, stream);
    else launch<BITS, XT, 8>(a, stream);
}

template <int BITS>
void with_type(const WordArgs &a, hipStream_t stream) {
    if (a.x_dtype == MK_F32) with_samples<BITS, MK_F32>(a, stream);
    else if (a.x_dtype == MK_F16) with_samples<BITS, MK_F16>(a, stream);
    else with_samples<BITS, MK_BF16>(a, stream);
}

}  // namespace

void mk_matvec::words_launch(const WordArgs &a, int bits, hipStream_t stream) {
    switch (bits) {
        case 1: with_type<1>(a, stream); break;
        case 2: with_type<2>(a, stream); break;
        case 3: with_type<3>(a, stream); break;
        case 4: with_type<4>(a, stream); break;
        case 5: with_type<5>(a, stream); break;
        case 6: with_type<6>(a, stream); break;
        case 7: with_type<7>(a, stream); break;
        default: with_type<8>(a, stream); break;
    }
}
