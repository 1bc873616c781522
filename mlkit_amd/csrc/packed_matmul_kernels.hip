// One format's kernels of packed_matmul_impl.h; compiled once per MK_MATMUL_FORMAT.
#include "packed_matmul_impl.h"

using namespace mk_matmul;

namespace {

template <int FORMAT, int XT, int RT, int MT, int SUB, bool SUMS, bool SPLIT>
int launch(const MatmulArgs &a, const MatmulPlan &plan, hipStream_t stream) {
    const size_t lds = lds_bytes<FORMAT, RT, MT, SPLIT>(plan.waves, a.groups, SUMS);
    auto *kernel = &packed_matmul_kernel<FORMAT, XT, RT, MT, SUB, SUMS, SPLIT>;
    static std::atomic<size_t> allowed{64 * 1024};   // raised once per kernel when a launch needs more
    if (lds > allowed.load(std::memory_order_relaxed)) {
        const hipError_t status = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (status != hipSuccess)
            return mk_fail(MK_ERR_HIP, "mk_packed_matmul: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(status));
        allowed.store(160 * 1024, std::memory_order_relaxed);
    }
    const dim3 grid(mk_cdiv(a.rows, 16 * RT), mk_cdiv(a.samples, 16 * MT));
    hipLaunchKernelGGL(kernel, grid, dim3(64 * plan.waves), lds, stream, a);
    return MK_OK;
}

template <int FORMAT, int XT, int SUB, bool SUMS, bool SPLIT>
int with_tiles(const MatmulArgs &a, const MatmulPlan &plan, hipStream_t stream) {
    switch (plan.sample_tiles * 8 + plan.row_tiles) {
        case 1 * 8 + 1: return launch<FORMAT, XT, 1, 1, SUB, SUMS, SPLIT>(a, plan, stream);
        case 1 * 8 + 2: return launch<FORMAT, XT, 2, 1, SUB, SUMS, SPLIT>(a, plan, stream);
        case 1 * 8 + 4: return launch<FORMAT, XT, 4, 1, SUB, SUMS, SPLIT>(a, plan, stream);
        case 2 * 8 + 2: return launch<FORMAT, XT, 2, 2, SUB, SUMS, SPLIT>(a, plan, stream);
        case 2 * 8 + 4: return launch<FORMAT, XT, 4, 2, SUB, SUMS, SPLIT>(a, plan, stream);
        default: return launch<FORMAT, XT, 2, 4, SUB, SUMS, SPLIT>(a, plan, stream);
    }
}

template <int FORMAT, int XT, bool SPLIT>
int with_groups(const MatmulArgs &a, const MatmulPlan &plan, hipStream_t stream) {
    if constexpr (FORMAT != kUniform4 && FORMAT != kUniform8) {   // (those two are compiled with sums only)
        if (!a.need_sums) {
            if (plan.sub == 2) return with_tiles<FORMAT, XT, 2, false, SPLIT>(a, plan, stream);
            return with_tiles<FORMAT, XT, 1, false, SPLIT>(a, plan, stream);
        }
    }
    if (plan.sub == 2) return with_tiles<FORMAT, XT, 2, true, SPLIT>(a, plan, stream);
    return with_tiles<FORMAT, XT, 1, true, SPLIT>(a, plan, stream);
}

template <int FORMAT, int XT>
int with_operands(const MatmulArgs &a, const MatmulPlan &plan, hipStream_t stream) {
    if constexpr (FORMAT != kUniform4 && FORMAT != kUniform8) {   // (their operands are exact)
        if (plan.split) return with_groups<FORMAT, XT, true>(a, plan, stream);
    }
    return with_groups<FORMAT, XT, false>(a, plan, stream);
}

}  // namespace

#define MK_PASTE_(a, b) a##b
#define MK_PASTE(a, b) MK_PASTE_(a, b)
int MK_PASTE(mk_matmul_launch_, MK_MATMUL_FORMAT)(const MatmulArgs &a, const MatmulPlan &plan, int x_dtype, hipStream_t stream) {
    if (x_dtype == MK_F16) return with_operands<MK_MATMUL_FORMAT, MK_F16>(a, plan, stream);
    return with_operands<MK_MATMUL_FORMAT, MK_BF16>(a, plan, stream);
}
