// Host-side helpers shared by the C-ABI translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string>
#include <vector>
#include "hccl_types.h"
#include "hcclx.h"
#include "kernels/launch.h"
#include "kernels/vops.h"

namespace hcclx {

// Thread-local text of the last failure; returned by hcclx_last_error().
void set_error(const std::string &msg);
int fail(int code, const std::string &msg);  // records msg, returns code
int fail_hip(hipError_t e, const char *what);

#define HCCLX_HIP(expr)                                          \
    do {                                                         \
        hipError_t e_ = (expr);                                  \
        if (e_ != hipSuccess) return ::hcclx::fail_hip(e_, #expr); \
    } while (0)

// Per-device launch resources.
struct DeviceCtx {
    int device = -1;
    int num_cus = 0;
    // Fold launches use one workgroup per tile (measured faster than a persistent grid on MI355X: the
    // hardware staggers workgroups, a grid-stride loop runs them in lock step).  A non-zero value caps
    // the grid at blocks_per_cu x CUs instead.
    uint32_t blocks_per_cu = 0;
    // Chain folds whose largest fan-in reaches this go to the wide chain kernel (HCCLX_WIDE_CHAIN_FROM); with 9 to
    // 16 sources it measured 2 to 8 % faster than the kernel that holds all sources in registers, with 8 the same.
    uint32_t wide_chain_from = 9;
    // The same for chains with a single destination (HCCLX_WIDE_CHAIN_FROM_ONE_DST): there the wide kernel has
    // shapes of its own (wide_shape_for), and an 8-source ReduceScatter measured 5 to 10 % faster on it.
    uint32_t wide_chain_from_one_dst = 5;
    // Wide launches whose segments have this many destinations give each XCD a contiguous eighth of the tiles
    // (HCCLX_WIDE_XCD_REMAP_FROM).
    uint32_t wide_xcd_remap_from = 16;
    // A single-destination chain launch that would have fewer four-vector tiles than this takes two vectors per
    // thread and eight sources at a time, to spread a small job over more CUs (HCCLX_WIDE_MIN_TILES; set from the CU count).
    uint32_t wide_min_tiles = 0;
    bool a2av_direct = true;           // HCCLX_A2AV_DIRECT: AlltoAllV tables of up to 15 ranks in the kernel arguments (0 = off)
    // V kernels whose tables live on the device cannot know their tile count on the host and run as a
    // persistent grid of this many workgroups per CU.
    uint32_t v_blocks_per_cu = 2;
    // With host tables the V kernels launch one workgroup per run of this many consecutive tiles.
    uint32_t v_tiles_per_block = 1;
    // Writing n outputs at once runs HBM a third slower than writing them one after the other (the banks see n
    // streams of row misses).  A fold whose result goes to several places therefore stores it once and a second
    // launch copies it to the other places, one place at a time in batches of fanout_run bytes (HCCLX_FANOUT_RUN)
    // whose re-reads the L2 serves: 8 x 64 MiB fp32 AllReduce 204 -> 175 us.  It pays from about 320 MiB read
    // and written by such folds in one launch (HCCLX_FANOUT_FROM, 0 = never).  Buffers that are not in the Infinity Cache
    // (256 MiB), one pass : split: 8 x 16 MiB bf16 52.4 : 48.5 us, 8 x 25 78.3 : 70.8, 8 x 32 99.4 : 88.3, 12 x 12
    // 61.5 : 52.7, 32 x 6 80.9 : 71.7, 12 x 8 43.3 : 36.8, 6 x 24 55.9 : 53.9, 8 x 8 27.1 : 28.2.  The same buffers over and
    // over, of which the cache holds what fits: 8 x 16 43.5 : 48.3, 8 x 25 65.7 : 71.0, 8 x 32 86.9 : 87.8, 12 x 12
    // 51.1 : 52.9, 12 x 16 70.2 : 68.7.
    // A batch of 16 MiB is 2 MiB in each of the eight L2s (4 MiB each) while its copies are written: 8 x 64 MiB fp16
    // AllGather with batches of 4 / 8 / 12 / 16 / 20 / 24 MiB 801 / 761 / 753 / 740 / 744 / 732 us, and with 16 the
    // fan-out of a 12 x 1 GiB AllReduce 1930 us.
    uint64_t fanout_from = 320ull << 20;
    uint64_t fanout_run = 16ull << 20;
    // AllGather(V) with host tables: from this many bytes of payload on (HCCLX_AGV_PHASED_FROM, 0 = never) the outputs
    // of a run of a source are written one after the other, each workgroup writing one output.
    uint64_t agv_phased_from = 4ull << 20;
    // The n orders of a self-first fold among up to waves_max_fan ranks (HCCLX_WAVES_MAX_FAN) take the kernel with one
    // store per wavefront when the launch writes waves_from bytes or more (HCCLX_WAVES_FROM, 0 = never); waves_chains
    // (HCCLX_WAVES_CHAINS): also chains whose value goes to several places; waves_pieces (HCCLX_WAVES_PIECES): 1 KiB
    // pieces per source and workgroup, 0 = chosen per launch (2, 4 or 8).
    uint64_t waves_from = 1;
    uint32_t waves_max_fan = 16;
    bool waves_chains = false;
    uint32_t waves_pieces = 0;
    uint32_t moe_scatter_rows = 0;          // MoE dispatch of long rows: entries of a token per wavefront, 1 or 2; 0 = chosen per launch (HCCLX_MOE_SCATTER_ROWS)
    uint64_t store_through_upto = 320ull << 20;   // fold launches with several destinations that write no more than this store through the L2 (HCCLX_STORE_THROUGH_UPTO)
    // Folds to one place that hold the workgroups of a CU few by LDS that they do not use (the largest chains and trees):
    // HCCLX_FOLD_LDS_HOLD, 0 = they ask for none, and the largest chains take the shape of the next smaller ones.
    bool fold_lds_hold = true;
    // Descriptor ring: tables of one-shot launches are written to pinned host memory and copied to the
    // device ring on the launch stream just before the kernel.
    char *h_ring = nullptr;
    char *d_ring = nullptr;
    size_t ring_bytes = 0;
    // Device address, on this GPU, of the library's fixed launch-table array (hcclx_fold_static): looked up once
    // when the context is made.
    char *static_table = nullptr;
};

// Returns the context of the current device, creating it on first use (nullptr + error set on failure).
DeviceCtx *device_ctx();

// The shape of a chain launch with one destination; *per_cu: non-zero where LDS holds more workgroups than this off a CU.
WideShape wide_shape_for(const DeviceCtx *ctx, const hcclx_wide_seg_t *segs, uint32_t nseg, int esz, uint32_t *per_cu);

// Reserves `bytes` (multiple of 256) in the descriptor ring.  Blocks the host only when the ring wraps
// onto a slice whose earlier launches have not finished.
int ring_reserve(DeviceCtx *ctx, size_t bytes, hipStream_t stream, char **h, char **d);

uint32_t grid_for(const DeviceCtx *ctx, uint64_t total_tiles);

// Whether one launch of the wavefront kernel takes this many 1 KiB pieces per source, `per_tile` of them and `waves` wavefronts
// of 64 to a workgroup: HIP allows fewer than 2^32 work-items along x.  (The register kernels' workgroups move more each.)
inline bool waves_fit(uint64_t pieces, uint32_t per_tile, uint32_t waves)
{
    return pieces / per_tile + 1 <= 0xffffffffull / (64ull * waves);
}


// One launch of the copy kernel that writes one output at a time (kernels/vops.h).
struct PhasedLaunch {
    std::vector<PhasedSource> sources;   // place = number of destinations
    std::vector<char *> dsts;            // sources.size() * grid.nd pointers, source s's at [s * nd, s * nd + ndst)
    std::vector<uint32_t> ranges;
    uint32_t shift = 0;
    uint64_t tiles = 0;
    PhasedGrid grid{};
    size_t bytes() const;       // the three arrays as they lie in the launch table
    void fill(char *h) const;
    PhasedTable table(const char *d) const;   // the arrays of a launch table at d
};
// A contiguous source that goes to several places whole.
struct PhasedStream {
    const char *src;
    uint64_t bytes;
    std::vector<char *> dst;
};
// Turns streams into launches of at most max_groups groups of kPhasedGroupTiles tiles: streams that continue each other (source
// and every destination) are joined; batches of up to batch_bytes are written to one place after the other.
void build_phased(std::vector<PhasedStream> &streams, uint64_t batch_bytes, uint32_t max_groups, std::vector<PhasedLaunch> *out);
// The non-empty blocks of an AlltoAllV with host tables (row-major n x n, elements of esz bytes), their tiles numbered
// through; returns the number of tiles.
uint64_t list_alltoallv_blocks(const void *const *send, void *const *recv, const uint64_t *send_counts, const uint64_t *sdispls,
                               const uint64_t *rdispls, uint32_t n, uint32_t esz, std::vector<CopyBlock> *blocks);
// The start table of blocks whose first tiles are begin[0 .. n): the block that holds tile g << *shift for every group g of
// the `tiles` tiles, and behind them the block of the last tile.  The smallest groups of which there are at most max_groups.
void index_tiles(const uint64_t *begin, size_t n, uint64_t tiles, uint32_t max_groups, std::vector<uint32_t> *starts, uint32_t *shift);
// A launch's tables in device memory: blocks, start table.
struct BlockLaunch {
    std::vector<CopyBlock> blocks;
    std::vector<uint32_t> starts;
    uint32_t shift = 0;
    uint64_t tiles = 0;
    void index();           // once the blocks are listed
    size_t bytes() const;
    void fill(char *h) const;
    BlockTable table(const char *d) const;   // the arrays of a launch table at d
};

// Queues the copy of a launch table from the pinned ring to its place in device memory.
int upload_table(char *d, const char *h, size_t bytes, hipStream_t stream);

}  // namespace hcclx
