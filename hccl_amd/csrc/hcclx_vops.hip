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

void list_alltoallv_blocks(const void *const *send, void *const *recv, const uint64_t *send_counts, const uint64_t *sdispls,
                           const uint64_t *rdispls, uint32_t n, uint32_t esz, std::vector<CopyBlock> *blocks)
{
    blocks->clear();
    blocks->reserve(static_cast<size_t>(n) * n);
    for (uint32_t i = 0; i < n; ++i) {
        for (uint32_t j = 0; j < n; ++j) {
            const uint64_t bytes = send_counts[i * n + j] * esz;
            if (bytes == 0) continue;
            blocks->push_back({static_cast<const char *>(send[i]) + sdispls[i * n + j] * esz,
                               static_cast<char *>(recv[j]) + rdispls[j * n + i] * esz, bytes});
        }
    }
}

bool cut_slabs(const std::vector<CopyBlock> &blocks, size_t max_slabs, uint32_t max_at, std::vector<CopySlab> *slabs, uint32_t *shift)
{
    std::vector<uint64_t> tiles(blocks.size());
    uint64_t most = 0;
    for (size_t b = 0; b < blocks.size(); ++b) {
        tiles[b] = v_tiles_of(blocks[b].bytes, reinterpret_cast<uint64_t>(blocks[b].dst), 1);
        most = tiles[b] > most ? tiles[b] : most;
    }
    if (max_slabs < blocks.size()) max_slabs = blocks.size();
    uint64_t n = 0;
    for (*shift = 0;; ++*shift) {
        const uint64_t last = (1ull << *shift) - 1;
        n = 0;
        for (uint64_t t : tiles) n += (t + last) >> *shift;
        if (n <= max_slabs && ((most + last) >> *shift) <= max_at) break;
    }
    if (n << *shift > 0x7fffffffull) return false;
    slabs->clear();
    slabs->reserve(n);
    for (size_t b = 0; b < blocks.size(); ++b) {
        for (uint64_t k = 0; k << *shift < tiles[b]; ++k) slabs->push_back({static_cast<uint32_t>(b), static_cast<uint32_t>(k)});
    }
    return true;
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
        // Equal blocks need no table.  (A captured launch keeps to the tables, so that what can be captured stays as it
        // is; and a grid has at most 2^32 work-items along x.)
        const uint64_t block_bytes = send_counts[0] * esz;
        if (block_bytes != 0 && block_bytes < (1ull << 35) && equal_blocks(send_counts, sdispls, rdispls, n) && !is_capturing(st)) {
            EqualBlocks tab;
            std::memcpy(tab.send, ptrs.send, sizeof(tab.send));
            std::memcpy(tab.recv, ptrs.recv, sizeof(tab.recv));
            tab.bytes = block_bytes;
            const hipError_t e = launch_equal_blocks(tab, n, st);
            if (e != hipSuccess) return fail_hip(e, "alltoall kernel launch");
            return HCCL_SUCCESS;
        }
        std::vector<CopyBlock> blocks;
        list_alltoallv_blocks(send, recv, send_counts, sdispls, rdispls, n, static_cast<uint32_t>(esz), &blocks);
        if (blocks.empty()) return HCCL_SUCCESS;
        std::vector<CopySlab> slabs;
        uint32_t shift = 0;
        bool small = n <= kA2avInlineRanks && ctx->a2av_direct;
        for (size_t k = 0; k < static_cast<size_t>(n) * n && small; ++k) {
            small = send_counts[k] <= 0xffffffffull && sdispls[k] <= 0xffffffffull && rdispls[k] <= 0xffffffffull;
        }
        if (small) {
            // small host tables and their slabs ride in the kernel arguments: nothing is copied in front of the kernel
            if (!cut_slabs(blocks, kA2avInlineSlabs, 256, &slabs, &shift)) return fail(HCCL_E_PARA, "too much data for one launch");
            A2avInline tab;
            tab.n = n;
            tab.inv_n = 65536u / n + 1u;
            tab.esz = static_cast<uint32_t>(esz);
            uint8_t number[kA2avInlineBlocks];   // of the non-empty blocks in the n x n tables
            uint32_t live = 0;
            for (uint32_t i = 0; i < n; ++i) {
                tab.send[i] = ptrs.send[i];
                tab.recv[i] = ptrs.recv[i];
                for (uint32_t j = 0; j < n; ++j) {
                    const uint32_t k = i * n + j;
                    if (send_counts[k] != 0) number[live++] = static_cast<uint8_t>(k);
                    tab.counts[k] = static_cast<uint32_t>(send_counts[k]);
                    tab.sdispls[k] = static_cast<uint32_t>(sdispls[k]);
                    tab.rdispls[k] = static_cast<uint32_t>(rdispls[j * n + i]);
                }
            }
            for (size_t k = 0; k < slabs.size(); ++k) {
                const uint32_t one = number[slabs[k].source] | slabs[k].at << 8;
                tab.slabs[k >> 1] = (k & 1) ? (tab.slabs[k >> 1] | one << 16) : one;
            }
            hipError_t e = launch_alltoallv_inline(tab, static_cast<uint32_t>(slabs.size()), shift, st);
            if (e != hipSuccess) return fail_hip(e, "alltoallv kernel launch");
            return HCCL_SUCCESS;
        }
        // any other host table: the non-empty blocks and their slabs in device memory
        if (!cut_slabs(blocks, kBlockTableSlabs, ~0u, &slabs, &shift)) return fail(HCCL_E_PARA, "too much data for one launch");
        const size_t list_bytes = (blocks.size() * sizeof(CopyBlock) + 255) & ~static_cast<size_t>(255);
        const size_t bytes = list_bytes + slabs.size() * sizeof(CopySlab);
        char *h = nullptr;
        char *d = nullptr;
        rc = ring_reserve(ctx, bytes, st, &h, &d);
        if (rc != HCCL_SUCCESS) return rc;
        std::memcpy(h, blocks.data(), blocks.size() * sizeof(CopyBlock));
        std::memcpy(h + list_bytes, slabs.data(), slabs.size() * sizeof(CopySlab));
        rc = upload_table(d, h, bytes, st);
        if (rc != HCCL_SUCCESS) return rc;
        const BlockTable tab{reinterpret_cast<const CopyBlock *>(d), reinterpret_cast<const CopySlab *>(d + list_bytes)};
        hipError_t e = launch_copy_blocks(tab, static_cast<uint32_t>(slabs.size()), shift, st);
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
        // Large: the outputs of a batch of slabs are written one after the other.  A source's places are one offset into
        // every receive buffer and the tables fit the kernel arguments: nothing is copied in front of the kernel.
        if (n > 1 && ctx->agv_phased_from != 0 && payload >= ctx->agv_phased_from) {
            std::vector<PhasedStream> streams;
            streams.reserve(n);
            for (uint32_t i = 0; i < n; ++i) {
                if (counts[i] != 0) streams.push_back({ptrs.send[i], counts[i] * esz, {ptrs.recv[0] + displs[i] * esz}});
            }
            std::vector<PhasedLaunch> launches;
            build_phased(streams, ctx->fanout_run, kPhasedInlineSlabs, &launches);
            for (PhasedLaunch &l : launches) {
                PhasedInline tab;
                for (uint32_t d = 0; d < n; ++d) tab.base[d] = ptrs.recv[d];
                for (size_t k = 0; k < l.sources.size(); ++k) {
                    tab.sources[k] = l.sources[k];
                    tab.sources[k].place = static_cast<uint64_t>(l.dsts[k] - ptrs.recv[0]);
                }
                for (size_t k = 0; k < l.slabs.size(); ++k) tab.slabs[k] = l.slabs[k].source | l.slabs[k].at << 6;
                tab.nslabs = static_cast<uint32_t>(l.slabs.size());
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
