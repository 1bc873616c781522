// Packed scalar-codec matrix-vector product: planning and the C entry points.
//
// Replaces the reference's `matrix_vector` wrapper and direct launch
// (kernels/packed_linear.py:181-226, inference/packed_linear.py:181-245 in
// /root/reference/src/mlkit).

#include <cstdlib>

#include "packed_matvec_impl.h"

#define MK_DECLARE_WIDTH(n)                                                                  \
    bool mk_matvec_launch_b##n(const mk_matvec::MatvecArgs &, const mk_matvec::Plan &, int, \
                               bool, hipStream_t);
MK_DECLARE_WIDTH(2) MK_DECLARE_WIDTH(3) MK_DECLARE_WIDTH(4) MK_DECLARE_WIDTH(5)
MK_DECLARE_WIDTH(6) MK_DECLARE_WIDTH(7) MK_DECLARE_WIDTH(8)
#undef MK_DECLARE_WIDTH

namespace {

using mk_matvec::kChunkCodes;
using mk_matvec::kMaxTableEntries;
using mk_matvec::MatvecArgs;
using mk_matvec::Plan;
using mk_matvec::WordArgs;

int next_pow2(int v) {
    int p = 1;
    while (p < v) p <<= 1;
    return p;
}

// Dynamic LDS of one workgroup: value table, fp32 scale (and zero) tile, per-wave row sums.
size_t lds_bytes_for(const Plan &p, int groups, bool uniform, bool has_zero) {
    (void)has_zero;
    const size_t tile_rows = static_cast<size_t>(p.rows_parallel) * p.rows_per_thread;
    size_t tile_slots = tile_rows * groups;
    if (tile_slots < 4u * p.threads) tile_slots = 4u * p.threads;  // kStaged * threads
    size_t floats = (uniform ? 0 : kMaxTableEntries) + 2 * tile_slots;
    floats += tile_rows > static_cast<size_t>(p.threads) ? tile_rows : p.threads;  // bias tile
    const int group_rows = p.sample_tile >= 8 ? 1 : (p.sample_tile == 4 ? 2 : 4);
    floats += 2 * static_cast<size_t>(group_rows) * p.sample_tile * p.threads;  // per-lane sums, two buffers
    return floats * sizeof(float);
}

// Development switches, read from the environment once per process (not per launch).
struct Tuning {
    int no_stream4, no_pairs, workgroups, rows_parallel;  // rows_parallel 0: planned
};
const Tuning &tuning() {
    static const Tuning values = [] {
        auto read = [](const char *name, int fallback) {
            const char *text = std::getenv(name);
            return text && *text ? std::atoi(text) : fallback;
        };
        return Tuning{read("MK_MATVEC_NO_STREAM4", 0), read("MK_MATVEC_NO_PAIRS", 0), read("MK_MATVEC_WORKGROUPS", 512),
                      read("MK_MATVEC_ROWS_PARALLEL", 0)};
    }();
    return values;
}

// Whether the chunked kernel beats the word kernel, whose workgroups cost less to start and whose rows share the activations: on
// larger layers of few samples.  us here against us there, codes that mostly no cache holds:
// * one sample beyond 2^24 weights -- INT8 with fp32 x 4096 x 4096 10.2 / 10.1, 4096 x 6144 12.0 / 15.6, 8192 x 4096 13.9 / 17.5, 22016 x
//   8192 43 / 72; fp32 scales under fp16 x: INT8 10.4 / 9.9, 12.0 / 15.4, 14.8 / 17.0, 3-bit codebook 13.3 / 10.3, 13.3 / 15.8, 15.0 /
//   17.5 -- but beyond 2^25 for tables of two and four bits, which the word kernel unpacks in the fewest steps (NF4 with fp32 x
//   13.1 / 8.5, 13.8 / 12.9, 15.2 / 14.3, 46 / 56);
// * two samples from 2^24 likewise with bf16 x (NF4 4096 x 6144 16.7 / 22.3, 8192 x 4096 19.1 / 21.2), with fp16 x unless on such a
//   table (2-bit grid 13.1 / 15.0, 17.0 / 16.7; NF4 16.4 / 14.4, 19.0 / 16.6), and with fp32 x on even grids in rows of more than 4096
//   codes (INT8 15.5 / 16.7, 3 bits 4096 x 8192 14.2 / 16.0, but 8192 x 4096 17.5 / 16.4);
// * two otherwise, three and four from 2^25 (NF4 with fp32 x, two: 4096 x 6144 17.2 / 15.1, 4096 x 11008 18.5 / 21.7; INT8, four: 8192 x
//   4096 27.7 / 21.7, 4096 x 11008 23.9 / 30.0, 11008 x 4096 30.4 / 28.2);
// * more only in rows of at least 8192 codes on even grids: fp32 x and up to seven bits from 3 * 2^24 weights (3 bits, eight samples:
//   4096 x 11008 40 / 39, 8192 x 8192 48 / 53, 22016 x 8192 116 / 132; INT8 53 / 54 and 132 / 133), fp16 x and four bits from 2^25
//   (4096 x 11008 26 / 28, 4096 x 14336 28 / 35); eight samples of 16 bits take 4 to 11 times as long otherwise;
// * rows of more than 16384 codes, where a thread holds two chunks, on even grids with one and two samples from 3 * 2^24, with
//   bf16 x from 2^25 (INT8 with fp32 x, one: 2048 x 18432 21.4 / 20.1, 4096 x 18432 22.9 / 32.7; 3 bits with bf16 x, one and two: 2048 x
//   18432 18.9 / 19.8 and 21.6 / 28.8; NF4 62 / 18 and 75 / 28, INT8 with four samples 65 / 45).
bool chunked_is_faster(int samples, int rows, int width, int bits, int x_dtype, bool uniform) {
    const long long weights = static_cast<long long>(rows) * width, unit = 1ll << 24;
    if (width > 16384) return uniform && samples <= 2 && weights > (x_dtype == MK_BF16 ? 2 : 3) * unit;
    if (samples <= 2) {
        const bool quick_table = !uniform && (bits == 2 || bits == 4);
        const bool early = samples == 1 ? !quick_table : x_dtype == MK_BF16 || (x_dtype == MK_F16 ? !quick_table : uniform && width > 4096);
        return weights > (early ? 1 : 2) * unit;
    }
    if (samples <= 4) return weights > 2 * unit;
    if (!uniform || width < 8192) return false;
    return x_dtype == MK_F32 ? bits < 8 && weights > 3 * unit : x_dtype == MK_F16 && bits == 4 && weights > 2 * unit;
}

// Chooses the lane/row decomposition of the chunked kernel; returns false when the
// layer needs the word kernel (widths or groups that are not multiples of 32 codes,
// or a scale tile that does not fit in LDS) or is faster there.
//
// A row's chunks are spread over `seg` lanes (a power of two up to 64, or whole
// wavefronts), one chunk per lane, two when a row has more than 512 chunks.  Every
// thread owns 2U rows, so a workgroup multiplies a tile of rows_parallel * 2U adjacent
// rows; rows_parallel grows (up to 256 threads) only while the grid keeps at least two
// workgroups per compute unit.
bool plan_chunked(int samples, int rows, int width, int group, int groups, int bits, int x_dtype,
                  bool uniform, bool has_zero, Plan &p) {
    if (bits < 2 || width % kChunkCodes != 0) return false;
    if (!chunked_is_faster(samples, rows, width, bits, x_dtype, uniform)) return false;
    if (group % kChunkCodes != 0 && group < width) return false;
    const int chunks_per_row = width / kChunkCodes;
    int c = chunks_per_row > 512 ? 2 : 1;
    if (chunks_per_row > 1024) return false;
    const int max_tile = (x_dtype == MK_F32 ? 4 : 8) / c;
    int mt = 1;
    while (mt < samples && mt < max_tile) mt <<= 1;
    const int lanes = mk_cdiv(chunks_per_row, c);
    const int seg = lanes <= 64 ? next_pow2(lanes) : 64 * mk_cdiv(lanes, 64);
    const int rows_per_thread = mk_matvec::kThreadRows;
    int rows_parallel = seg < 64 ? 64 / seg : 1;
    const int wanted_workgroups = tuning().workgroups;
    while (seg * rows_parallel * 2 <= 256 &&
           rows / (rows_parallel * 2 * rows_per_thread) >= wanted_workgroups)
        rows_parallel *= 2;
    if (tuning().rows_parallel > 0) rows_parallel = tuning().rows_parallel;
    const int threads = seg * rows_parallel;
    if (threads % 64 != 0 || threads > 512) return false;
    p.sample_tile = mt;
    p.chunks = c;
    p.seg_lanes = seg;
    p.rows_parallel = rows_parallel;
    p.threads = threads;
    p.rows_per_thread = rows_per_thread;
    p.lds_bytes = lds_bytes_for(p, groups, uniform, has_zero);
    if (p.lds_bytes > 60 * 1024) return false;
    p.grid_x = 0;
    return true;
}

// Rows [first_row, output_width) through the word kernel.
int launch_words(const void *x, int x_dtype, const uint8_t *packed, const void *scales, int scale_dtype,
                 const float *values, int n_values, const void *zeros, const void *bias, int bias_dtype, void *y, int samples,
                 int output_width, int input_width, int group, int bits, int uniform, float grid_min,
                 float grid_step, int first_row, hipStream_t stream) {
    WordArgs w{};
    w.x = x; w.packed = packed; w.scales = scales; w.zeros = zeros; w.values = values; w.n_values = n_values; w.bias = bias;
    w.y = y; w.samples = samples; w.rows = output_width; w.width = input_width;
    w.groups = mk_cdiv(input_width, group); w.first_row = first_row;
    w.pieces_per_group = group >= input_width ? 0 : group / 16;   // (groups shorter than a row are multiples of sixteen codes)
    w.row_bytes = static_cast<size_t>(input_width) * bits / 8;
    w.x_dtype = x_dtype; w.scale_dtype = scale_dtype; w.bias_dtype = bias_dtype; w.uniform = uniform;
    w.grid_min = grid_min; w.grid_step = grid_step;
    mk_matvec::words_launch(w, bits, stream);
    MK_LAUNCH_CHECK("mk_packed_matvec");
    return MK_OK;
}

}  // namespace

extern "C" int mk_packed_layout_supported(int bits, int input_width, int group) {
    if (bits < 1 || bits > 8 || input_width < 1 || group < 1) return 0;
    const int divisor = mk_gcd(bits, 8);
    const int codes_per_word = 8 / divisor;
    if (input_width % codes_per_word || group % codes_per_word) return 0;
    const int group_words = group / codes_per_word;
    int tile_words = group_words & -group_words;
    if (tile_words > 128 / codes_per_word) tile_words = 128 / codes_per_word;
    return tile_words * codes_per_word >= 16 ? 1 : 0;
}

extern "C" int mk_packed_matvec(const void *x, int x_dtype, const uint8_t *packed, const void *scales,
                                int scale_dtype, const float *values, int n_values, const void *zeros,
                                const void *bias, int bias_dtype, void *y, int samples,
                                int output_width, int input_width, int group, int bits, int uniform,
                                float grid_min, float grid_step, void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MK_REQUIRE(x && packed && scales && y, MK_ERR_INVALID, "mk_packed_matvec: null tensor pointer");
    MK_REQUIRE(mk_dtype_valid(x_dtype) && mk_dtype_valid(scale_dtype), MK_ERR_INVALID,
               "mk_packed_matvec: unknown dtype code");
    MK_REQUIRE(!bias || mk_dtype_valid(bias_dtype), MK_ERR_INVALID, "mk_packed_matvec: unknown bias dtype");
    MK_REQUIRE(samples >= 1 && output_width >= 1 && input_width >= 1 && group >= 1, MK_ERR_INVALID,
               "mk_packed_matvec: sizes must be positive");
    MK_REQUIRE(bits >= 1 && bits <= 8, MK_ERR_INVALID, "mk_packed_matvec: code width must be 1..8 bits");
    MK_REQUIRE(uniform || (values && n_values >= 1 && n_values <= (1 << bits)), MK_ERR_INVALID,
               "mk_packed_matvec: a value table of at most 2^bits entries is required");
    MK_REQUIRE(mk_packed_layout_supported(bits, input_width, group), MK_ERR_UNSUPPORTED,
               "mk_packed_matvec: rows or scale groups split a packing word (bits=%d width=%d group=%d)",
               bits, input_width, group);
    const int groups = mk_cdiv(input_width, group);
    const bool aligned = (reinterpret_cast<uintptr_t>(packed) & 3u) == 0 &&
                         (reinterpret_cast<uintptr_t>(scales) & 3u) == 0 &&
                         (reinterpret_cast<uintptr_t>(zeros) & 3u) == 0 &&
                         (reinterpret_cast<uintptr_t>(bias) & 3u) == 0 &&
                         (reinterpret_cast<uintptr_t>(x) & 15u) == 0 &&
                         (static_cast<size_t>(input_width) * mk_dtype_bytes(x_dtype)) % 16 == 0;
    int done_rows = 0;  // rows [0, done_rows) are covered by a chunked kernel
    Plan plan;
    if (aligned && !tuning().no_stream4 &&
        mk_matvec::long_accepts(samples, output_width, input_width, group, bits, x_dtype, scale_dtype, uniform != 0) &&
        (reinterpret_cast<uintptr_t>(scales) & 1u) == 0) {
        mk_matvec::Stream4Args s4;
        s4.x = x; s4.packed = packed; s4.scales = scales; s4.zeros = zeros; s4.bias = bias; s4.y = y;
        s4.samples = samples; s4.rows = output_width; s4.width = input_width; s4.group = group;
        s4.groups = groups; s4.bias_dtype = bias_dtype; s4.grid_min = grid_min; s4.grid_step = grid_step;
        s4.values = values; s4.n_values = n_values; s4.uniform = uniform; s4.bits = bits;
        s4.x_dtype = x_dtype; s4.scale_dtype = scale_dtype;
        done_rows = mk_matvec::long_launch(s4, stream);
        MK_REQUIRE(done_rows >= 0, MK_ERR_HIP, "mk_packed_matvec: the runtime refused the kernel's launch");
        if (input_width <= 16384 && output_width - done_rows >= 4) {   // (the grouped launch leaves the same rows % 4 to the word kernel)
            const int more = mk_matvec::stream4_launch_remainder(s4, done_rows, stream);
            MK_REQUIRE(more >= 0, MK_ERR_HIP, "mk_packed_matvec: the runtime refused the kernel's LDS size");
            done_rows += more;
        }
        if (done_rows > 0) MK_LAUNCH_CHECK("mk_packed_matvec");
    } else if (aligned && !tuning().no_stream4 &&
               mk_matvec::stream4_accepts(samples, input_width, group, bits, x_dtype, scale_dtype, uniform != 0) &&
        (reinterpret_cast<uintptr_t>(scales) & 1u) == 0) {
        mk_matvec::Stream4Args s4;
        s4.x = x; s4.packed = packed; s4.scales = scales; s4.zeros = zeros; s4.bias = bias; s4.y = y;
        s4.samples = samples; s4.rows = output_width; s4.width = input_width; s4.group = group;
        s4.groups = groups; s4.bias_dtype = bias_dtype; s4.grid_min = grid_min; s4.grid_step = grid_step;
        s4.values = values; s4.n_values = n_values; s4.uniform = uniform; s4.bits = bits;
        s4.x_dtype = x_dtype; s4.scale_dtype = scale_dtype;
        done_rows = mk_matvec::stream4_launch(s4, stream);
        MK_REQUIRE(done_rows >= 0, MK_ERR_HIP, "mk_packed_matvec: the runtime refused the kernel's LDS size");
        if (output_width - done_rows >= 4) {
            const int more = mk_matvec::stream4_launch_remainder(s4, done_rows, stream);
            MK_REQUIRE(more >= 0, MK_ERR_HIP, "mk_packed_matvec: the runtime refused the kernel's LDS size");
            done_rows += more;
        }
        if (done_rows > 0) MK_LAUNCH_CHECK("mk_packed_matvec");
    } else if (aligned && !tuning().no_pairs &&
               mk_matvec::pairs_accepts(input_width, group, bits, x_dtype, scale_dtype) &&
               (reinterpret_cast<uintptr_t>(scales) & 1u) == 0) {
        mk_matvec::Stream4Args s4;
        s4.x = x; s4.packed = packed; s4.scales = scales; s4.zeros = zeros; s4.bias = bias; s4.y = y;
        s4.samples = samples; s4.rows = output_width; s4.width = input_width; s4.group = group;
        s4.groups = groups; s4.bias_dtype = bias_dtype; s4.grid_min = grid_min; s4.grid_step = grid_step;
        s4.values = values; s4.n_values = n_values; s4.uniform = uniform; s4.bits = bits;
        s4.x_dtype = x_dtype; s4.scale_dtype = scale_dtype;
        done_rows = mk_matvec::pairs_launch(s4, stream);
        if (done_rows > 0) MK_LAUNCH_CHECK("mk_packed_matvec");
    } else if (aligned && plan_chunked(samples, output_width, input_width, group, groups, bits, x_dtype,
                                uniform != 0, zeros != nullptr, plan)) {
        const int tile_rows = plan.rows_parallel * plan.rows_per_thread;
        const int tiles = output_width / tile_rows;
        if (tiles > 0) {
            MatvecArgs a;
            a.x = x; a.packed = packed; a.scales = scales; a.zeros = zeros; a.values = values;
            a.bias = bias; a.y = y;
            a.scale_row_offset = 0;
            a.samples = samples; a.rows = output_width; a.width = input_width; a.group = group;
            a.groups = groups; a.n_values = n_values; a.scale_dtype = scale_dtype; a.bias_dtype = bias_dtype;
            a.seg_lanes = plan.seg_lanes; a.rows_parallel = plan.rows_parallel;
            a.chunks_per_row = input_width / kChunkCodes;
            a.grid_min = grid_min; a.grid_step = grid_step;
            plan.grid_x = tiles;
            bool launched = false;
            switch (bits) {
                case 2: launched = mk_matvec_launch_b2(a, plan, x_dtype, uniform != 0, stream); break;
                case 3: launched = mk_matvec_launch_b3(a, plan, x_dtype, uniform != 0, stream); break;
                case 4: launched = mk_matvec_launch_b4(a, plan, x_dtype, uniform != 0, stream); break;
                case 5: launched = mk_matvec_launch_b5(a, plan, x_dtype, uniform != 0, stream); break;
                case 6: launched = mk_matvec_launch_b6(a, plan, x_dtype, uniform != 0, stream); break;
                case 7: launched = mk_matvec_launch_b7(a, plan, x_dtype, uniform != 0, stream); break;
                case 8: launched = mk_matvec_launch_b8(a, plan, x_dtype, uniform != 0, stream); break;
            }
            if (launched) {
                MK_LAUNCH_CHECK("mk_packed_matvec");
                done_rows = tiles * tile_rows;
            }
        }
    }
    if (done_rows < output_width)
        return launch_words(x, x_dtype, packed, scales, scale_dtype, values, n_values, zeros, bias, bias_dtype, y, samples,
                            output_width, input_width, group, bits, uniform, grid_min, grid_step, done_rows, stream);
    return MK_OK;
}

extern "C" int mk_packed_matvec_group(const void *const *x, int x_dtype, int count, const uint8_t *const *packed,
                                      const void *const *scales, int scale_dtype, const float *values, int n_values,
                                      const void *const *zeros, const void *const *bias, int bias_dtype,
                                      void *const *y, const int *output_widths, int samples, int input_width,
                                      int group, int bits, int uniform, float grid_min, float grid_step,
                                      void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MK_REQUIRE(count >= 1 && count <= mk_matvec::kMaxGroupMembers, MK_ERR_INVALID,
               "mk_packed_matvec_group: 1 to %d matrices per call", mk_matvec::kMaxGroupMembers);
    MK_REQUIRE(x && packed && scales && y && output_widths, MK_ERR_INVALID, "mk_packed_matvec_group: null argument");
    MK_REQUIRE(samples >= 1 && input_width >= 1 && group >= 1, MK_ERR_INVALID,
               "mk_packed_matvec_group: sizes must be positive");
    bool with_zeros = zeros && zeros[0];
    const bool dtypes_valid = mk_dtype_valid(x_dtype) && mk_dtype_valid(scale_dtype) && (!bias || mk_dtype_valid(bias_dtype)) &&
                              bits >= 1 && bits <= 8;
    // The kernels that take a group: the INT4 streaming kernels, else the table kernels.
    const bool streaming = dtypes_valid && !tuning().no_stream4 &&
                           mk_matvec::stream4_accepts(samples, input_width, group, bits, x_dtype, scale_dtype, uniform != 0);
    const bool tables = dtypes_valid && !streaming && !tuning().no_pairs && (uniform || (values && n_values >= 1 && n_values <= (1 << bits))) &&
                        mk_packed_layout_supported(bits, input_width, group) &&
                        input_width <= 16384 &&   // (longer rows: one launch per matrix)
                        mk_matvec::pairs_accepts(input_width, group, bits, x_dtype, scale_dtype);
    bool one_launch = (streaming || tables) && (static_cast<size_t>(input_width) * mk_dtype_bytes(x_dtype)) % 16 == 0;
    for (int i = 0; i < count; ++i) {
        MK_REQUIRE(x[i] && packed[i] && scales[i] && y[i] && output_widths[i] >= 1, MK_ERR_INVALID,
                   "mk_packed_matvec_group: matrix %d has a null pointer or no rows", i);
        MK_REQUIRE(((zeros && zeros[i]) != 0) == with_zeros, MK_ERR_INVALID,
                   "mk_packed_matvec_group: either every matrix has offsets or none has");
        const void *bias_i = bias ? bias[i] : nullptr;
        one_launch = one_launch && (reinterpret_cast<uintptr_t>(x[i]) & 15u) == 0 &&
                     (reinterpret_cast<uintptr_t>(packed[i]) & 3u) == 0 &&
                     (reinterpret_cast<uintptr_t>(scales[i]) & 3u) == 0 &&
                     (reinterpret_cast<uintptr_t>(with_zeros ? zeros[i] : nullptr) & 3u) == 0 &&
                     (reinterpret_cast<uintptr_t>(bias_i) & 3u) == 0;
    }
    if (!one_launch) {  // the same results, one launch per matrix
        for (int i = 0; i < count; ++i)
            if (int status = mk_packed_matvec(x[i], x_dtype, packed[i], scales[i], scale_dtype, values, n_values,
                                              with_zeros ? zeros[i] : nullptr, bias ? bias[i] : nullptr, bias_dtype,
                                              y[i], samples, output_widths[i], input_width, group, bits, uniform,
                                              grid_min, grid_step, stream_))
                return status;
        return MK_OK;
    }
    mk_matvec::Stream4Args shared{};
    shared.x = x[0]; shared.samples = samples; shared.width = input_width; shared.group = group;
    shared.groups = mk_cdiv(input_width, group); shared.bias_dtype = bias_dtype; shared.grid_min = grid_min;
    shared.grid_step = grid_step; shared.values = values; shared.n_values = n_values; shared.uniform = uniform;
    shared.bits = bits; shared.x_dtype = x_dtype; shared.scale_dtype = scale_dtype;
    mk_matvec::Stream4Group members{};
    members.count = count;
    for (int i = 0; i < count; ++i) {
        members.member[i].x = x[i];
        members.member[i].packed = packed[i];
        members.member[i].scales = scales[i];
        members.member[i].zeros = with_zeros ? zeros[i] : nullptr;
        members.member[i].bias = bias ? bias[i] : nullptr;
        members.member[i].y = y[i];
    }
    int rows_per_tile = 0;
    if (streaming)
        MK_REQUIRE(mk_matvec::stream4_launch_group(shared, members, output_widths, &rows_per_tile, stream) == 0, MK_ERR_HIP,
                   "mk_packed_matvec_group: the runtime refused the kernel's LDS size");
    else
        mk_matvec::pairs_launch_group(shared, members, output_widths, &rows_per_tile, stream);
    MK_LAUNCH_CHECK("mk_packed_matvec_group");
    for (int i = 0; i < count; ++i) {  // rows past a member's last whole tile
        int covered = output_widths[i] / rows_per_tile * rows_per_tile;
        if (streaming && output_widths[i] - covered >= 4) {   // their whole four-row tiles, as in the single call
            mk_matvec::Stream4Args own = shared;
            own.x = x[i]; own.packed = packed[i]; own.scales = scales[i]; own.zeros = members.member[i].zeros;
            own.bias = members.member[i].bias; own.y = y[i]; own.rows = output_widths[i];
            const int more = mk_matvec::stream4_launch_remainder(own, covered, stream);
            MK_REQUIRE(more >= 0, MK_ERR_HIP, "mk_packed_matvec_group: the runtime refused the kernel's LDS size");
            MK_LAUNCH_CHECK("mk_packed_matvec_group");
            covered += more;
        }
        if (covered < output_widths[i])
            if (int status = launch_words(x[i], x_dtype, packed[i], scales[i], scale_dtype, values, n_values, members.member[i].zeros,
                                          members.member[i].bias, bias_dtype, y[i], samples, output_widths[i],
                                          input_width, group, bits, uniform, grid_min, grid_step, covered, stream))
                return status;
    }
    return MK_OK;
}

extern "C" int mk_packed_layer_matvec(const mk_packed_layer *layer, const void *x, int x_dtype, void *y, int samples, void *stream) {
    MK_REQUIRE(layer, MK_ERR_INVALID, "mk_packed_layer_matvec: null layer");
    const mk_packed_layer &l = *layer;
    return mk_packed_matvec(x, x_dtype, l.packed, l.scales, l.scale_dtype, l.values, l.n_values, l.zeros, l.bias, l.bias_dtype, y, samples,
                            l.output_width, l.input_width, l.group, l.bits, l.uniform, l.grid_min, l.grid_step, stream);
}
