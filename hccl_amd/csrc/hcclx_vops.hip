// C-ABI entry points of the V collectives (see include/hcclx.h).
#include "hcclx.h"
#include "hcclx_internal.h"
#include "kernels/elem.h"
#include "kernels/vops.h"

#include <cstring>
#include <vector>

using namespace hcclx;

namespace {

// Host tables are staged through the descriptor ring; device tables are used where they are.
int stage_tables(DeviceCtx *ctx, const uint64_t *const *tabs, int ntabs, size_t entries, int on_device,
                 hipStream_t st, const uint64_t **out)
{
    if (on_device) {
        for (int i = 0; i < ntabs; ++i) out[i] = tabs[i];
        return HCCL_SUCCESS;
    }
    const size_t one = (entries * sizeof(uint64_t) + 255) & ~static_cast<size_t>(255);
    char *h = nullptr;
    char *d = nullptr;
    int rc = ring_reserve(ctx, one * ntabs, st, &h, &d);
    if (rc != HCCL_SUCCESS) return rc;
    for (int i = 0; i < ntabs; ++i) {
        std::memcpy(h + one * i, tabs[i], entries * sizeof(uint64_t));
        out[i] = reinterpret_cast<const uint64_t *>(d + one * i);
    }
    HCCLX_HIP(hipMemcpyAsync(d, h, one * ntabs, hipMemcpyHostToDevice, st));
    return HCCL_SUCCESS;
}

int fill_ptrs(const void *const *send, void *const *recv, uint32_t n, VRankPtrs *p)
{
    if (send == nullptr || recv == nullptr) return fail(HCCL_E_PTR, "send/recv pointer array is null");
    if (n == 0 || n > kMaxVRanks) return fail(HCCL_E_PARA, "rank count outside 1.." + std::to_string(kMaxVRanks));
    std::memset(p, 0, sizeof(*p));
    for (uint32_t i = 0; i < n; ++i) {
        p->send[i] = static_cast<const char *>(send[i]);
        p->recv[i] = static_cast<char *>(recv[i]);
    }
    return HCCL_SUCCESS;
}

}  // namespace

namespace hcclx {

uint64_t list_alltoallv_blocks(const void *const *send, void *const *recv, const uint64_t *send_counts, const uint64_t *sdispls,
                               const uint64_t *rdispls, uint32_t n, uint32_t esz, std::vector<CopyBlock> *blocks)
{
    blocks->clear();
    blocks->reserve(static_cast<size_t>(n) * n);
    uint64_t tiles = 0;
    for (uint32_t i = 0; i < n; ++i) {
        for (uint32_t j = 0; j < n; ++j) {
            const uint64_t bytes = send_counts[i * n + j] * esz;
            if (bytes == 0) continue;
            char *dst = static_cast<char *>(recv[j]) + rdispls[j * n + i] * esz;
            blocks->push_back({static_cast<const char *>(send[i]) + sdispls[i * n + j] * esz, dst, bytes, tiles});
            tiles += v_tiles_of(bytes, reinterpret_cast<uint64_t>(dst), 1);
        }
    }
    return tiles;
}

void index_tiles(const uint64_t *begin, size_t n, uint64_t tiles, uint32_t max_groups, std::vector<uint32_t> *starts, uint32_t *shift)
{
    *shift = 0;
    while ((tiles - 1) >> *shift >= max_groups) ++*shift;
    starts->clear();
    starts->reserve(((tiles - 1) >> *shift) + 2);
    uint32_t b = 0;
    for (uint64_t first = 0; first < tiles + (1ull << *shift); first += 1ull << *shift) {
        const uint64_t tile = first < tiles ? first : tiles - 1;
        while (b + 1 < n && begin[b + 1] <= tile) ++b;
        starts->push_back(b);
    }
}

void BlockLaunch::index()
{
    std::vector<uint64_t> begin(blocks.size());
    for (size_t b = 0; b < blocks.size(); ++b) begin[b] = blocks[b].begin;
    // four groups to a block, so that a small table stays small: what lies in front of the kernel is its upload
    const uint64_t groups = 4 * static_cast<uint64_t>(blocks.size());
    index_tiles(begin.data(), begin.size(), tiles, groups < kBlockTableGroups ? static_cast<uint32_t>(groups) : kBlockTableGroups, &starts,
                &shift);
}

namespace {
size_t list_bytes(size_t blocks) { return (blocks * sizeof(CopyBlock) + 255) & ~static_cast<size_t>(255); }
}  // namespace

size_t BlockLaunch::bytes() const { return list_bytes(blocks.size()) + starts.size() * sizeof(uint32_t); }

void BlockLaunch::fill(char *h) const
{
    std::memcpy(h, blocks.data(), blocks.size() * sizeof(CopyBlock));
    std::memcpy(h + list_bytes(blocks.size()), starts.data(), starts.size() * sizeof(uint32_t));
}

BlockTable BlockLaunch::table(const char *d) const
{
    return {reinterpret_cast<const CopyBlock *>(d), reinterpret_cast<const uint32_t *>(d + list_bytes(blocks.size())), shift};
}

}  // namespace hcclx

namespace {

// Tables on the host that describe equal blocks, back to back in rank order: what HcclAlltoAll passes.
bool equal_blocks(const uint64_t *send_counts, const uint64_t *sdispls, const uint64_t *rdispls, uint32_t n)
{
    const uint64_t count = send_counts[0];
    uint64_t differ = 0;
    for (uint32_t i = 0; i < n; ++i) {
        const size_t row = static_cast<size_t>(i) * n;
        uint64_t at = 0;
        for (uint32_t j = 0; j < n; ++j) {
            differ |= (send_counts[row + j] ^ count) | (sdispls[row + j] ^ at) | (rdispls[row + j] ^ at);
            at += count;
        }
        if (differ != 0) return false;
    }
    return true;
}

bool is_capturing(hipStream_t stream)
{
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &st) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return st != hipStreamCaptureStatusNone;
}

}  // namespace

namespace hcclx {

// An exchange of equal blocks of `count` elements needs no table.  *launched: false where it goes by the tables after all (a
// captured launch, so that what can be captured stays as it is; a grid has at most 2^32 work-items along x).
int alltoall_equal(const void *const *send, void *const *recv, uint64_t count, uint32_t n, int dtype, void *stream, bool *launched)
{
    *launched = false;
    if (!device_ctx()) return HCCL_E_RUNTIME;
    const uint64_t block_bytes = count * dtype_size(dtype);
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (block_bytes == 0 || block_bytes >= (1ull << 35) || is_capturing(st)) return HCCL_SUCCESS;
    VRankPtrs ptrs;
    const int rc = fill_ptrs(send, recv, n, &ptrs);
    if (rc != HCCL_SUCCESS) return rc;
    EqualBlocks tab;
    std::memcpy(tab.send, ptrs.send, sizeof(tab.send));
    std::memcpy(tab.recv, ptrs.recv, sizeof(tab.recv));
    tab.bytes = block_bytes;
    const hipError_t e = launch_equal_blocks(tab, n, st);
    if (e != hipSuccess) return fail_hip(e, "alltoall kernel launch");
    *launched = true;
    return HCCL_SUCCESS;
}

}  // namespace hcclx

extern "C" {

int hcclx_alltoallv(const void *const *send, void *const *recv, const uint64_t *send_counts,
                    const uint64_t *sdispls, const uint64_t *rdispls, uint32_t n, int dtype,
                    int tables_on_device, void *stream)
{
    DeviceCtx *ctx = device_ctx();
    if (!ctx) return HCCL_E_RUNTIME;
    const int esz = dtype_size(dtype);
    if (esz == 0) return fail(HCCL_E_NOT_SUPPORT, "unknown data type " + std::to_string(dtype));
    if (!send_counts || !sdispls || !rdispls) return fail(HCCL_E_PTR, "count/displacement table is null");
    VRankPtrs ptrs;
    int rc = fill_ptrs(send, recv, n, &ptrs);
    if (rc != HCCL_SUCCESS) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (!tables_on_device) {
        if (equal_blocks(send_counts, sdispls, rdispls, n)) {
            bool launched = false;
            rc = alltoall_equal(send, recv, send_counts[0], n, dtype, stream, &launched);
            if (rc != HCCL_SUCCESS || launched) return rc;
        }
        bool small = n <= kA2avInlineRanks && ctx->a2av_direct;
        for (size_t k = 0; k < static_cast<size_t>(n) * n && small; ++k) {
            small = send_counts[k] <= 0xffffffffull && sdispls[k] <= 0xffffffffull && rdispls[k] <= 0xffffffffull;
        }
        if (small) {
            // small host tables ride in the kernel arguments: nothing is copied in front of the kernel
            A2avInline tab;
            tab.n = n;
            tab.inv_n = 65536u / n + 1u;
            tab.esz = static_cast<uint32_t>(esz);
            uint64_t begin[kA2avInlineBlocks];
            uint64_t tiles = 0;
            for (uint32_t i = 0; i < n; ++i) {
                tab.send[i] = ptrs.send[i];
                tab.recv[i] = ptrs.recv[i];
                for (uint32_t j = 0; j < n; ++j) {
                    const uint32_t k = i * n + j;
                    tab.counts[k] = static_cast<uint32_t>(send_counts[k]);
                    tab.sdispls[k] = static_cast<uint32_t>(sdispls[k]);
                    tab.rdispls[k] = static_cast<uint32_t>(rdispls[j * n + i]);
                    begin[k] = tiles;
                    tab.begin[k] = static_cast<uint32_t>(tiles);
                    tiles += v_tiles_of(send_counts[k] * esz, reinterpret_cast<uint64_t>(ptrs.recv[j]) + rdispls[j * n + i] * esz, 1);
                }
            }
            if (tiles == 0) return HCCL_SUCCESS;
            if (tiles <= 0x7fffffffull) {
                std::vector<uint32_t> starts;
                index_tiles(begin, static_cast<size_t>(n) * n, tiles, kA2avInlineGroups, &starts, &tab.shift);
                std::memset(tab.starts, 0, sizeof(tab.starts));
                for (size_t g = 0; g < starts.size(); ++g) tab.starts[g >> 2] |= starts[g] << (g & 3) * 8;
                const hipError_t e = launch_alltoallv_inline(tab, tiles, st);
                if (e != hipSuccess) return fail_hip(e, "alltoallv kernel launch");
                return HCCL_SUCCESS;
            }
        }
        // any other host table: the non-empty blocks and their start table in device memory
        BlockLaunch l;
        l.tiles = list_alltoallv_blocks(send, recv, send_counts, sdispls, rdispls, n, static_cast<uint32_t>(esz), &l.blocks);
        if (l.tiles == 0) return HCCL_SUCCESS;
        if (l.tiles > 0x7fffffffull) return fail(HCCL_E_PARA, "too much data for one launch");
        l.index();
        char *h = nullptr;
        char *d = nullptr;
        rc = ring_reserve(ctx, l.bytes(), st, &h, &d);
        if (rc != HCCL_SUCCESS) return rc;
        l.fill(h);
        rc = upload_table(d, h, l.bytes(), st);
        if (rc != HCCL_SUCCESS) return rc;
        const hipError_t e = launch_copy_blocks(l.table(d), l.blocks.size(), l.tiles, st);
        if (e != hipSuccess) return fail_hip(e, "alltoallv kernel launch");
        return HCCL_SUCCESS;
    }
    // tables on the device: the tile count is not known here, so a persistent grid derives its own tile map
    const uint64_t grid = static_cast<uint64_t>(ctx->num_cus) * ctx->v_blocks_per_cu;
    const uint64_t *tabs[3] = {send_counts, sdispls, rdispls};
    const uint64_t *dev[3];
    rc = stage_tables(ctx, tabs, 3, static_cast<size_t>(n) * n, tables_on_device, st, dev);
    if (rc != HCCL_SUCCESS) return rc;
    hipError_t e = launch_alltoallv(ptrs, dev[0], dev[1], dev[2], n, static_cast<uint32_t>(esz),
                                    static_cast<uint32_t>(grid), 1u, st);
    if (e != hipSuccess) return fail_hip(e, "alltoallv kernel launch");
    return HCCL_SUCCESS;
}

int hcclx_allgatherv(const void *const *send, void *const *recv, const uint64_t *counts,
                     const uint64_t *displs, uint32_t n, int dtype, int tables_on_device, void *stream)
{
    DeviceCtx *ctx = device_ctx();
    if (!ctx) return HCCL_E_RUNTIME;
    const int esz = dtype_size(dtype);
    if (esz == 0) return fail(HCCL_E_NOT_SUPPORT, "unknown data type " + std::to_string(dtype));
    if (!counts || !displs) return fail(HCCL_E_PTR, "count/displacement table is null");
    VRankPtrs ptrs;
    int rc = fill_ptrs(send, recv, n, &ptrs);
    if (rc != HCCL_SUCCESS) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    uint64_t grid = static_cast<uint64_t>(ctx->num_cus) * ctx->v_blocks_per_cu;
    if (!tables_on_device) {
        uint64_t payload = 0;
        for (uint32_t i = 0; i < n; ++i) payload += counts[i] * esz;
        // Large: the outputs of a batch of tiles are written one after the other.  A source's places are one offset into
        // every receive buffer and the tables fit the kernel arguments: nothing is copied in front of the kernel.
        if (n > 1 && ctx->agv_phased_from != 0 && payload >= ctx->agv_phased_from) {
            std::vector<PhasedStream> streams;
            streams.reserve(n);
            for (uint32_t i = 0; i < n; ++i) {
                if (counts[i] != 0) streams.push_back({ptrs.send[i], counts[i] * esz, {ptrs.recv[0] + displs[i] * esz}});
            }
            std::vector<PhasedLaunch> launches;
            build_phased(streams, ctx->fanout_run, kPhasedInlineGroups, &launches);
            for (PhasedLaunch &l : launches) {
                PhasedInline tab;
                for (uint32_t d = 0; d < n; ++d) tab.base[d] = ptrs.recv[d];
                for (size_t k = 0; k < l.sources.size(); ++k) {
                    tab.sources[k] = l.sources[k];
                    tab.sources[k].place = static_cast<uint64_t>(l.dsts[k] - ptrs.recv[0]);
                }
                std::memset(tab.ranges, 0, sizeof(tab.ranges));
                for (size_t g = 0; g < l.ranges.size(); ++g) tab.ranges[g >> 1] |= (l.ranges[g] & 255u) << (g & 1) * 16 | (l.ranges[g] >> 16) << ((g & 1) * 16 + 8);
                tab.shift = l.shift;
                tab.tiles = static_cast<uint32_t>(l.tiles);
                l.grid.nd = n;
                hipError_t e = launch_phased_copy_inline(tab, l.grid, st);
                if (e != hipSuccess) return fail_hip(e, "allgatherv kernel launch");
            }
            return HCCL_SUCCESS;
        }
        uint64_t total = 0;
        for (uint32_t i = 0; i < n; ++i) {
            total += v_tiles_of(counts[i] * esz, reinterpret_cast<uint64_t>(ptrs.recv[0]) + displs[i] * esz, kAgvUnroll);
        }
        if (total == 0) return HCCL_SUCCESS;
        grid = (total + ctx->v_tiles_per_block - 1) / ctx->v_tiles_per_block;
        if (grid > 0x7fffffffull) grid = 0x7fffffffull;
        AgvTablesInline tabs;   // host tables of up to 64 ranks always fit the kernel arguments
        std::memset(&tabs, 0, sizeof(tabs));
        for (uint32_t i = 0; i < n; ++i) {
            tabs.counts[i] = counts[i];
            tabs.displs[i] = displs[i];
        }
        hipError_t e = launch_allgatherv_inline(ptrs, tabs, n, static_cast<uint32_t>(esz), static_cast<uint32_t>(grid),
                                                ctx->v_tiles_per_block, st);
        if (e != hipSuccess) return fail_hip(e, "allgatherv kernel launch");
        return HCCL_SUCCESS;
    }
    const uint64_t *dev[2] = {counts, displs};
    hipError_t e = launch_allgatherv(ptrs, dev[0], dev[1], n, static_cast<uint32_t>(esz), static_cast<uint32_t>(grid), tables_on_device ? 1u : ctx->v_tiles_per_block, st);
    if (e != hipSuccess) return fail_hip(e, "allgatherv kernel launch");
    return HCCL_SUCCESS;
}

int hcclx_displs_from_counts(const uint64_t *counts, uint32_t rows, uint32_t n, uint64_t *displs, uint64_t *totals,
                             void *stream)
{
    if (!device_ctx()) return HCCL_E_RUNTIME;
    if (!counts || !displs) return fail(HCCL_E_PTR, "counts or displs is null");
    if (n == 0 || n > kMaxVRanks) return fail(HCCL_E_PARA, "rank count outside 1.." + std::to_string(kMaxVRanks));
    if (rows == 0) return HCCL_SUCCESS;
    if (rows > 0x7fffffffu) return fail(HCCL_E_PARA, "too many rows");
    hipError_t e = launch_displs_from_counts(counts, rows, n, displs, totals, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return fail_hip(e, "displacement kernel launch");
    return HCCL_SUCCESS;
}

}  // extern "C"
