// Packed weight x nine and more rows of activations: planning and the C entry point (kernels: packed_matmul_impl.h).
//
// Covers the inputs for which inference/packed_linear.py:110-154 of /root/reference/src/mlkit decodes the whole weight
// and calls a dense product.

#include "packed_matmul_impl.h"

#include <cmath>

using mk_matmul::MatmulArgs;
using mk_matmul::MatmulPlan;

int mk_matmul_launch_0(const MatmulArgs &, const MatmulPlan &, int, hipStream_t);
int mk_matmul_launch_1(const MatmulArgs &, const MatmulPlan &, int, hipStream_t);
int mk_matmul_launch_2(const MatmulArgs &, const MatmulPlan &, int, hipStream_t);
int mk_matmul_launch_3(const MatmulArgs &, const MatmulPlan &, int, hipStream_t);
int mk_matmul_launch_4(const MatmulArgs &, const MatmulPlan &, int, hipStream_t);

namespace {

// Tiles of a launch.  A workgroup's fixed cost (arguments, scales, the first trip through its code, the sum over
// wavefronts) is 2 to 3 us, so the smallest tiles win that give at most one workgroup to each of the 256 compute units:
// 4096 x 4096, 16 / 32 / 64 / 128 rows of x: 6.8 / 8.2 / 9.9 / 13.0 us with 1 x 1, 2 x 1, 2 x 2, 4 x 2 tiles of 16 (RT x MT;
// one size down: 10.0 us at 32 rows, 12.4 at 64, 17.8 at 128; one up 8.1, 9.9, 12.9).  Layers with more tiles than that: two
// workgroups of four wavefronts on a compute unit, 64 rows of x each (14336 x 4096, 128 rows: 44 us; 51 with one
// workgroup of eight).
MatmulPlan plan_for(int samples, int rows) {
    static constexpr int kTiles[][2] = {{1, 1}, {2, 1}, {2, 2}, {4, 1}, {4, 2}};
    MatmulPlan plan{};
    for (const auto &tile : kTiles) {
        plan.row_tiles = tile[0];
        plan.sample_tiles = tile[1];
        plan.waves = mk_matmul::kMaxWaves;
        if (static_cast<long long>(mk_cdiv(rows, 16 * tile[0])) * mk_cdiv(samples, 16 * tile[1]) <= 256) return plan;
    }
    if (samples <= 16) {
        plan.sample_tiles = 1;
    } else if (samples > 32) {
        plan.row_tiles = 2;
        plan.sample_tiles = 4;
        plan.waves = 4;
    }
    return plan;
}

// The next smaller tiles, where the scales of a plan's rows do not fit LDS (8192 x 28672 INT4 with offsets, 64 rows of x: 114 us
// with 2 x 2 tiles, 209 straight to 1 x 1).  Where they fit but keep a second workgroup of 2 x 4 tiles off the compute unit
// smaller tiles lose all the same (14336 x 4096 in groups of 64, 64 rows: 34 us, 48 with 2 x 2).
void step_down(MatmulPlan &plan, int steps) {
    if (plan.sample_tiles == 4) {
        plan.sample_tiles = 2;
        plan.waves = steps < mk_matmul::kMaxWaves ? steps : mk_matmul::kMaxWaves;
    } else if (plan.row_tiles == 4 || plan.sample_tiles == 1) {
        plan.row_tiles /= 2;
    } else {
        plan.sample_tiles = 1;
    }
}

// Whether fp16 and bf16 hold every value of a grid, in the range the kernel brings them to.
bool grid_held(float minimum, float step, int codes) {
    float largest = 0.0f;
    for (int code = 0; code < codes; ++code) largest = std::fmax(largest, std::fabs(std::fmaf(static_cast<float>(code), step, minimum)));
    if (!(largest > 0.0f) || !std::isfinite(largest)) return false;
    int exponent;
    std::frexp(largest, &exponent);
    for (int code = 0; code < codes; ++code) {
        const float units = std::ldexp(std::fmaf(static_cast<float>(code), step, minimum), 8 - exponent);   // 2^7 ... 2^8 and below
        if (units != std::rint(units)) return false;   // eight bits from the largest value's first on: both types have them
    }
    return true;
}

int matmul(const void *x, int x_dtype, const uint8_t *packed, const void *scales, int scale_dtype, const float *values, int n_values,
           const void *zeros, const void *bias, int bias_dtype, void *y, int samples, int output_width, int input_width, int group,
           int bits, int uniform, float grid_min, float grid_step, int values_held, void *stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    MK_REQUIRE(x && packed && scales && y, MK_ERR_INVALID, "mk_packed_matmul: null tensor pointer");
    MK_REQUIRE(samples >= 1 && output_width >= 1 && input_width >= 1 && group >= 1, MK_ERR_INVALID,
               "mk_packed_matmul: sizes must be positive");
    MK_REQUIRE(x_dtype == MK_F16 || x_dtype == MK_BF16, MK_ERR_UNSUPPORTED, "mk_packed_matmul: fp16 or bf16 activations");
    MK_REQUIRE(scale_dtype == MK_F16 || scale_dtype == MK_BF16, MK_ERR_UNSUPPORTED, "mk_packed_matmul: fp16 or bf16 scales");
    MK_REQUIRE(!bias || mk_dtype_valid(bias_dtype), MK_ERR_INVALID, "mk_packed_matmul: unknown bias dtype");
    MK_REQUIRE(input_width % 32 == 0, MK_ERR_UNSUPPORTED, "mk_packed_matmul: rows of a multiple of 32 codes");
    MK_REQUIRE(bits == 2 || bits == 3 || bits == 4 || (bits == 8 && uniform), MK_ERR_UNSUPPORTED,
               "mk_packed_matmul: codes of 2, 3 or 4 bits, or of 8 on a uniform grid");
    MK_REQUIRE(uniform || (values && n_values >= 1 && n_values <= (1 << bits)), MK_ERR_INVALID,
               "mk_packed_matmul: a value table of at most 2^bits entries is required");
    const bool whole_row = group >= input_width;
    MK_REQUIRE(whole_row || group % 128 == 0 || group == 64, MK_ERR_UNSUPPORTED,
               "mk_packed_matmul: scale groups of 64 columns, of a multiple of 128, or of the whole row");
    MK_REQUIRE(((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(packed)) & 15u) == 0, MK_ERR_UNSUPPORTED,
               "mk_packed_matmul: activations and codes must be 16-byte aligned");
    MK_REQUIRE(static_cast<long long>(samples) * input_width < (1ll << 31), MK_ERR_UNSUPPORTED, "mk_packed_matmul: too many activations");

    MatmulArgs a{};
    a.x = x; a.packed = packed; a.scales = static_cast<const uint16_t *>(scales); a.zeros = static_cast<const uint16_t *>(zeros);
    a.values = values; a.bias = bias; a.y = y;
    a.samples = samples; a.rows = output_width; a.width = input_width; a.groups = mk_cdiv(input_width, group); a.group = group;
    a.steps = mk_cdiv(input_width, mk_matmul::kStep);
    a.n_values = n_values; a.uniform = uniform; a.scale_bf16 = scale_dtype == MK_BF16; a.bias_dtype = bias_dtype;
    a.grid_min = grid_min; a.grid_step = grid_step;

    const int format = bits == 8 ? mk_matmul::kUniform8 : bits == 4 && uniform ? mk_matmul::kUniform4
                       : bits == 4 ? mk_matmul::kTable4 : bits == 3 ? mk_matmul::kTable3 : mk_matmul::kTable2;
    a.need_sums = zeros != nullptr || format == mk_matmul::kUniform4 || format == mk_matmul::kUniform8;

    MatmulPlan plan = plan_for(samples, output_width);
    plan.split = bits != 8 && format != mk_matmul::kUniform4 && !(uniform ? grid_held(grid_min, grid_step, 1 << bits) : values_held != 0);
    plan.sub = whole_row || group % 128 == 0 ? 1 : 2;
    a.steps_per_group = whole_row ? a.steps : group / 128 > 0 ? group / 128 : 1;
    if (a.steps_per_group > 1) {   // exact for the steps of any row: below 2^31
        int log = 0;
        while ((1 << log) < a.steps_per_group) ++log;
        a.group_shift = log - 1;
        a.group_multiplier = static_cast<uint32_t>(((1ull << (31 + log)) + a.steps_per_group - 1) / a.steps_per_group);
    }
    a.whole_quads = output_width % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 7u) == 0;
    if (plan.waves > a.steps) plan.waves = a.steps;
    const size_t table = (bits == 2 ? 2048 : bits == 3 ? 256 : format == mk_matmul::kTable4 ? 1024 : 0) * (plan.split ? 2 : 1);
    auto lds = [&] {
        const size_t stage = static_cast<size_t>(plan.waves) * plan.sample_tiles * 4096;
        const size_t sums = static_cast<size_t>(plan.waves) * plan.row_tiles * plan.sample_tiles * 1024;
        return (stage > sums ? stage : sums) + table + (64 + static_cast<size_t>(a.groups) * 64 * (a.need_sums ? 2 : 1)) * plan.row_tiles;
    };
    while (lds() > 160 * 1024 && plan.row_tiles > 1) step_down(plan, a.steps);
    while (lds() > 160 * 1024 && plan.waves > 1) plan.waves /= 2;
    MK_REQUIRE(lds() <= 160 * 1024, MK_ERR_UNSUPPORTED, "mk_packed_matmul: the scales of 16 rows do not fit a compute unit");
    int status;
    switch (format) {
        case mk_matmul::kUniform4: status = mk_matmul_launch_0(a, plan, x_dtype, stream); break;
        case mk_matmul::kTable4: status = mk_matmul_launch_1(a, plan, x_dtype, stream); break;
        case mk_matmul::kTable3: status = mk_matmul_launch_2(a, plan, x_dtype, stream); break;
        case mk_matmul::kTable2: status = mk_matmul_launch_3(a, plan, x_dtype, stream); break;
        default: status = mk_matmul_launch_4(a, plan, x_dtype, stream); break;
    }
    if (status != MK_OK) return status;
    MK_LAUNCH_CHECK("mk_packed_matmul");
    return MK_OK;
}

}  // namespace

extern "C" int mk_packed_matmul(const void *x, int x_dtype, const uint8_t *packed, const void *scales, int scale_dtype,
                                const float *values, int n_values, const void *zeros, const void *bias, int bias_dtype,
                                void *y, int samples, int output_width, int input_width, int group, int bits,
                                int uniform, float grid_min, float grid_step, void *stream) {
    return matmul(x, x_dtype, packed, scales, scale_dtype, values, n_values, zeros, bias, bias_dtype, y, samples, output_width,
                  input_width, group, bits, uniform, grid_min, grid_step, 0, stream);
}

extern "C" int mk_packed_layer_matmul(const mk_packed_layer *layer, const void *x, int x_dtype, void *y, int samples, void *stream) {
    MK_REQUIRE(layer, MK_ERR_INVALID, "mk_packed_layer_matmul: null layer");
    const mk_packed_layer &l = *layer;
    return matmul(x, x_dtype, l.packed, l.scales, l.scale_dtype, l.values, l.n_values, l.zeros, l.bias, l.bias_dtype, y, samples,
                  l.output_width, l.input_width, l.group, l.bits, l.uniform, l.grid_min, l.grid_step, l.values_held, stream);
}
