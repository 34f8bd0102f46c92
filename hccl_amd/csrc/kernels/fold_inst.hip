// One data type's instantiations of the fold kernel.  Built once per type with
//   -DHCCLX_DT=<HcclDataType enumerator> -DHCCLX_NAME=<suffix> -DHCCLX_ORDERED=<0|1>
// HCCLX_ORDERED=1 (floating types) also builds the self-first and tree modes; for integers every fold
// order gives the same bits, so the launcher maps those modes onto the chain kernel.
// The trees of one operation are a unit of their own, -DHCCLX_TREE_OP=<HcclReduceOp enumerator>: the compiler takes two to five
// minutes for those of fp16, and units are compiled side by side.
// With -DHCCLX_COPY the unit holds the byte copy kernel instead (one source, many destinations).
#include "fold.h"

#include <algorithm>
#include <atomic>

namespace hcclx {

// More than 64 KiB of dynamic LDS a kernel gets only when HIP has been asked for it: once per device, when a launch is built, so
// that launching (a plan, inside a capture) is nothing but the launch.  `done`: the devices that have been asked.
constexpr size_t kLdsUnasked = 64 * 1024;
static hipError_t ask_for_lds(const void *kernel, size_t lds, int device, std::atomic<uint64_t> &done)
{
    const uint64_t bit = 1ull << (device & 63);
    if (lds <= kLdsUnasked || (done.load(std::memory_order_acquire) & bit) != 0) return hipSuccess;
    const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);
    if (e == hipSuccess) done.fetch_or(bit, std::memory_order_release);
    return e;
}

template <int DT, int OP, int MAXN, int MODE>
static hipError_t launch_one(const FoldLaunch &l)
{
    const size_t lds = std::max<size_t>(l.nseg * sizeof(uint64_t), lds_for(l.per_cu));
    HCCLX_LAUNCH((k_fold<DT, OP, MAXN, MODE>), dim3(l.grid), dim3(kFoldThreads), lds, l.stream,
                       l.tile_end, static_cast<const SegDev *>(l.segs), l.nseg, l.total_tiles, l.store_policy, l.uniform_tiles);
    return hipGetLastError();
}

template <int DT, int OP, int MODE, int NFIX>
static hipError_t launch_waves_n(const FoldLaunch &l)
{
    const bool direct = l.nseg <= kFoldDirectSegs || l.uniform_tiles != 0;
    const size_t lds = waves_lds_bytes(static_cast<int>(l.waves)) + (direct ? 0 : l.nseg * sizeof(uint64_t));
    HCCLX_LAUNCH((k_fold_waves<DT, OP, MODE, NFIX>), dim3(static_cast<uint32_t>(l.total_tiles)), dim3(l.waves * kWaveLanes), lds,
                 l.stream, l.tile_end, static_cast<const SegDev *>(l.segs), l.nseg, l.pieces, l.store_policy, l.uniform_tiles);
    return hipGetLastError();
}

// The self-first orders get an instance per rank count up to sixteen; mixed launches and chains run on instances that read
// the count per segment.
template <int DT, int OP, int MODE>
static hipError_t launch_waves(const FoldLaunch &l)
{
    if constexpr (MODE == kFoldSelfFirst) {
        switch (l.waves_fixed) {
            case 2: return launch_waves_n<DT, OP, MODE, 2>(l);
            case 3: return launch_waves_n<DT, OP, MODE, 3>(l);
            case 4: return launch_waves_n<DT, OP, MODE, 4>(l);
            case 5: return launch_waves_n<DT, OP, MODE, 5>(l);
            case 6: return launch_waves_n<DT, OP, MODE, 6>(l);
            case 7: return launch_waves_n<DT, OP, MODE, 7>(l);
            case 8: return launch_waves_n<DT, OP, MODE, 8>(l);
            case 9: return launch_waves_n<DT, OP, MODE, 9>(l);
            case 10: return launch_waves_n<DT, OP, MODE, 10>(l);
            case 11: return launch_waves_n<DT, OP, MODE, 11>(l);
            case 12: return launch_waves_n<DT, OP, MODE, 12>(l);
            case 13: return launch_waves_n<DT, OP, MODE, 13>(l);
            case 14: return launch_waves_n<DT, OP, MODE, 14>(l);
            case 15: return launch_waves_n<DT, OP, MODE, 15>(l);
            case 16: return launch_waves_n<DT, OP, MODE, 16>(l);
            default: return launch_waves_n<DT, OP, MODE, 0>(l);
        }
    } else if constexpr (MODE == kFoldChain) {
        // from four wavefronts on they share the fold; large launches among two and three ranks do too (waves_team)
        return l.waves_team ? launch_waves_n<DT, OP, MODE, kWavesTeam>(l) : launch_waves_n<DT, OP, MODE, 0>(l);
    } else {
        return hipErrorInvalidValue;
    }
}

template <int DT, int OP, int MODE, int SHAPE>
static hipError_t launch_wide_shape(const FoldLaunch &l)
{
    constexpr int kThreads = wide_kernel_threads(MODE, SHAPE, DTypeOf<DT>::kHalfFloat);
    const size_t lds = std::max<size_t>(l.nseg * sizeof(uint64_t), lds_for(l.per_cu));
    if (l.ready_only) {
        static std::atomic<uint64_t> done{0};
        return ask_for_lds(reinterpret_cast<const void *>(&k_fold_wide<DT, OP, MODE, SHAPE>), lds, l.device, done);
    }
    HCCLX_LAUNCH((k_fold_wide<DT, OP, MODE, SHAPE>), dim3(l.grid), dim3(kThreads), lds, l.stream,
                       l.tile_end, static_cast<const SegWide *>(l.segs), l.nseg, l.total_tiles, l.xcd_remap, l.store_policy, l.uniform_tiles);
    return hipGetLastError();
}

// l.waves: sources of the widest segment
template <int DT, int OP, int R>
static hipError_t launch_wide_waves(const FoldLaunch &l)
{
    const bool direct = l.nseg <= kFoldDirectSegs || l.uniform_tiles != 0;
    const size_t lds = static_cast<size_t>(l.waves) * kWaveLanes * 16 + (direct ? 0 : l.nseg * sizeof(uint64_t));
    if (l.ready_only) {   // (64 sources and a staged prefix)
        static std::atomic<uint64_t> done{0};
        return ask_for_lds(reinterpret_cast<const void *>(&k_fold_wide_waves<DT, OP, R>), lds, l.device, done);
    }
    HCCLX_LAUNCH((k_fold_wide_waves<DT, OP, R>), dim3(static_cast<uint32_t>(l.total_tiles)), dim3(kWideWaves * kWaveLanes), lds, l.stream,
                 l.tile_end, static_cast<const SegWide *>(l.segs), l.nseg, l.waves, l.pieces, l.uniform_tiles);
    return hipGetLastError();
}

template <int DT, int OP, int MODE>
static hipError_t launch_wide(const FoldLaunch &l)
{
    if constexpr (MODE == kFoldChain) {
        switch (l.wide_shape) {
            case kWideSmall: return launch_wide_shape<DT, OP, MODE, kWideSmall>(l);
            case kWideThree: return launch_wide_shape<DT, OP, MODE, kWideThree>(l);
            case kWideFour: return launch_wide_shape<DT, OP, MODE, kWideFour>(l);
            case kWideLarge: return launch_wide_shape<DT, OP, MODE, kWideLarge>(l);
            default: return launch_wide_shape<DT, OP, MODE, kWideMany>(l);
        }
    } else if constexpr (MODE == kFoldTree) {
        return l.wide_shape == kTreeLarge ? launch_wide_shape<DT, OP, MODE, kTreeLarge>(l) : launch_wide_shape<DT, OP, MODE, kTreePlain>(l);
    } else {
        switch ((l.waves + kWideWaves - 1) / kWideWaves) {
            case 1: return launch_wide_waves<DT, OP, 1>(l);
            case 2: return launch_wide_waves<DT, OP, 2>(l);
            case 3: return launch_wide_waves<DT, OP, 3>(l);
            case 4: return launch_wide_waves<DT, OP, 4>(l);
            default: return hipErrorInvalidValue;
        }
    }
}

#ifdef HCCLX_COPY

hipError_t fold_dispatch_copy(const FoldLaunch &l)
{
    return launch_one<HCCL_DATA_TYPE_INT8, HCCL_REDUCE_SUM, 1, kFoldChain>(l);
}

#else

template <int OP, int MODE>
static hipError_t by_fan(int maxn, const FoldLaunch &l)
{
    if (l.waves != 0 && maxn <= kMaxFan) return launch_waves<HCCLX_DT, OP, MODE>(l);
    switch (maxn) {
        case 2: return launch_one<HCCLX_DT, OP, 2, MODE>(l);
        case 4: return launch_one<HCCLX_DT, OP, 4, MODE>(l);
        case 8: return launch_one<HCCLX_DT, OP, 8, MODE>(l);
        case 16: return launch_one<HCCLX_DT, OP, 16, MODE>(l);
        case kMaxWideFan: return launch_wide<HCCLX_DT, OP, MODE>(l);
        default: return hipErrorInvalidValue;
    }
}

#ifdef HCCLX_TREE_OP

template <int DT, int OP>
hipError_t fold_tree(int maxn, const FoldLaunch &l)
{
    static_assert(DT == HCCLX_DT, "the type of the unit");
    return by_fan<OP, kFoldTree>(maxn, l);
}
template hipError_t fold_tree<HCCLX_DT, HCCLX_TREE_OP>(int maxn, const FoldLaunch &l);

#else

template <int MODE>
static hipError_t by_op(int op, int maxn, const FoldLaunch &l)
{
    switch (op) {
        case HCCL_REDUCE_SUM: return by_fan<HCCL_REDUCE_SUM, MODE>(maxn, l);
        case HCCL_REDUCE_PROD: return by_fan<HCCL_REDUCE_PROD, MODE>(maxn, l);
        case HCCL_REDUCE_MAX: return by_fan<HCCL_REDUCE_MAX, MODE>(maxn, l);
        case HCCL_REDUCE_MIN: return by_fan<HCCL_REDUCE_MIN, MODE>(maxn, l);
        default: return hipErrorInvalidValue;
    }
}

#define HCCLX_CAT_(a, b) a##b
#define HCCLX_CAT(a, b) HCCLX_CAT_(a, b)

hipError_t HCCLX_CAT(fold_dispatch_, HCCLX_NAME)(int op, int maxn, int mode, const FoldLaunch &l)
{
    if (mode == kFoldChain) {
        return by_op<kFoldChain>(op, maxn, l);
    }
#if HCCLX_ORDERED
    if (mode == kFoldSelfFirst) {
        return by_op<kFoldSelfFirst>(op, maxn, l);
    }
    if (mode == kFoldTree) {
        switch (op) {
            case HCCL_REDUCE_SUM: return fold_tree<HCCLX_DT, HCCL_REDUCE_SUM>(maxn, l);
            case HCCL_REDUCE_PROD: return fold_tree<HCCLX_DT, HCCL_REDUCE_PROD>(maxn, l);
            case HCCL_REDUCE_MAX: return fold_tree<HCCLX_DT, HCCL_REDUCE_MAX>(maxn, l);
            case HCCL_REDUCE_MIN: return fold_tree<HCCLX_DT, HCCL_REDUCE_MIN>(maxn, l);
            default: return hipErrorInvalidValue;
        }
    }
#endif
    return hipErrorInvalidValue;
}

#endif
#endif

}  // namespace hcclx
