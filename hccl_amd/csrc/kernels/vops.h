// Launch interface of the V-collective kernels (vops.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "launch.h"
#include "segtab.h"

namespace hcclx {

constexpr uint32_t kMaxVRanks = 64;

// Tile geometry of the V kernels: 256 threads x `unroll` vectors of 16 bytes per tile.
// 16-byte vectors each thread moves per tile.  AlltoAllV stages and scans an n x n table per workgroup, so its
// tiles are large (32 KiB); AllGatherV's set-up is n entries, and small tiles (4 KiB: every workgroup sweeps
// a compact range and retires quickly) measured faster for its write-heavy traffic.
#ifndef HCCLX_A2AV_UNROLL
#define HCCLX_A2AV_UNROLL 8
#endif
#ifndef HCCLX_AGV_UNROLL
#define HCCLX_AGV_UNROLL 1
#endif
constexpr int kA2avUnroll = HCCLX_A2AV_UNROLL;
constexpr int kAgvUnroll = HCCLX_AGV_UNROLL;
// The copies that write one output at a time (large AllGatherV, fan-out of a fold's result): 4 KiB tiles, one vector
// per thread.  A wavefront that issues one store and ends writes HBM faster than one that issues two or four (fills of
// 1 GiB: 7.0 against 6.0 TB/s), and the same holds for these copies (8 x 64 MiB AllGather: 755 against 824 us).
constexpr int kPhasedUnroll = 1;
constexpr uint64_t kPhasedTile = 256ull * 16 * kPhasedUnroll;

// Tiles of a block of `bytes` bytes whose first destination byte sits at address `dst`.  Stores are
// aligned: the bytes before the first 16-byte boundary of dst (head) and after the last whole vector
// (tail) are moved one byte per thread by the block's last tile.  Used by the kernels and, when the
// tables are on the host, by the launcher to size the grid exactly.
// The tile grid of a block is shifted by v_shift_of() vectors so that every wavefront's 64 x 16 bytes start
// on a 1 KiB boundary of dst: whole cache lines are stored.  The first tile is then partial.
__host__ __device__ inline uint64_t v_head_of(uint64_t bytes, uint64_t dst)
{
    const uint64_t head = (16 - (dst & 15)) & 15;
    return head > bytes ? bytes : head;
}
__host__ __device__ inline uint32_t v_shift_of(uint64_t head, uint64_t dst)
{
    return static_cast<uint32_t>(((dst + head) & 1023) / 16);
}
__host__ __device__ inline uint64_t v_last_tile_of(uint64_t bytes, uint64_t dst, int unroll)   // of a block that is not empty
{
    const uint64_t kTileVecs = 256ull * unroll;
    const uint64_t head = v_head_of(bytes, dst);
    return ((bytes - head) / 16 + v_shift_of(head, dst)) / kTileVecs;
}
__host__ __device__ inline uint64_t v_tiles_of(uint64_t bytes, uint64_t dst, int unroll)
{
    return bytes == 0 ? 0 : v_last_tile_of(bytes, dst, unroll) + 1;
}

// Base pointers of every virtual rank's send and receive buffer, passed by value as a kernel argument.
struct VRankPtrs {
    const char *send[kMaxVRanks];
    char *recv[kMaxVRanks];
};

// Count / displacement tables as the kernels read them.  Host tables of up to 15 ranks travel inside the kernel
// arguments (no host-to-device copy is queued in front of the kernel); larger host tables become a list of
// blocks in device memory; tables that already live on the device are read through pointers.
struct A2avTablesPtr {
    const uint64_t *send_counts;
    const uint64_t *sdispls;
    const uint64_t *rdispls;
    __device__ uint64_t count(uint32_t p) const { return send_counts[p]; }
    __device__ uint64_t sdispl(uint32_t p) const { return sdispls[p]; }
    __device__ uint64_t rdispl(uint32_t p) const { return rdispls[p]; }
};
// Host tables.  The 4 KiB tiles of all blocks of the exchange (source i to destination j) are numbered through, and a
// workgroup moves one: there are as many workgroups as tiles, whatever the blocks' lengths.  Tiles come in groups of
// 1 << shift, and starts[g] is the block that holds the first tile of group g: the block of a tile lies between starts[g] and
// starts[g + 1].  With several groups to a block these are mostly one and the same, and two dependent scalar loads find
// it, where a search in the whole prefix of the blocks' tiles takes 2 + log2(n * n).
struct CopyBlock {
    const char *src;
    char *dst;
    uint64_t bytes;
    uint64_t begin;   // number of its first tile
};
// A launch's tables in device memory, for host tables of any size.
struct BlockTable {
    const CopyBlock *blocks;
    const uint32_t *starts;
    uint32_t shift;
};
constexpr uint32_t kBlockTableGroups = 4096;   // at most
// The same in the kernel arguments, for up to 15 ranks and 32-bit counts: nothing is copied in front of the kernel.
// Block b is source b / n, destination b % n, the empty ones among them (an empty block begins where the next one does).
constexpr uint32_t kA2avInlineRanks = 15;
constexpr uint32_t kA2avInlineBlocks = kA2avInlineRanks * kA2avInlineRanks;
constexpr uint32_t kA2avInlineGroups = 128;
struct A2avInline {
    const char *send[kA2avInlineRanks];
    char *recv[kA2avInlineRanks];
    uint32_t counts[kA2avInlineBlocks];
    uint32_t sdispls[kA2avInlineBlocks];
    uint32_t rdispls[kA2avInlineBlocks];
    uint32_t begin[kA2avInlineBlocks];
    uint32_t starts[kA2avInlineGroups / 4 + 1];   // a byte each
    uint32_t shift;
    uint32_t n;
    uint32_t inv_n;   // 65536 / n + 1: b * inv_n >> 16 is b / n for every block number
    uint32_t esz;
};
// An exchange of equal blocks: block j of rank i's send buffer becomes block i of rank j's receive buffer.
struct EqualBlocks {
    const char *send[kMaxVRanks];
    char *recv[kMaxVRanks];
    uint64_t bytes;   // of a block
};
struct AgvTablesPtr {
    const uint64_t *counts;
    const uint64_t *displs;
    __device__ uint64_t count(uint32_t i) const { return counts[i]; }
    __device__ uint64_t displ(uint32_t i) const { return displs[i]; }
};
// The copy kernel that writes one output at a time.  The tiles of its sources are numbered through as those of the blocks
// above, and a batch of tiles, a few MiB, is copied to its first place, then to the second and so on.  A batch is a multiple of
// eight tiles: workgroups go to the eight XCDs in turn, each with an L2 of its own, and a tile is then copied to all its
// places by the same XCD.
struct PhasedSource {
    const char *src;
    uint64_t bytes;
    uint64_t place;   // table in memory: ndst; tables in the kernel arguments: offset into every rank's receive buffer
    uint32_t begin;   // number of its first tile (of the first source of a launch: wrapped below zero when it begins inside)
    uint32_t reserved;
};
constexpr uint32_t kPhasedGroupTiles = 1024;   // at most: 4 MiB
// A source of so many tiles begins at a multiple of eight of them: HBM is interleaved over its stacks by 4 KiB, and one XCD then
// stays with the same stacks for all of them (100 x 1 MiB to eight places 149.7 us, 155.2 without; no difference for 33 tiles).
constexpr uint32_t kPhasedLongTiles = 192;
// A launch's tables in device memory: sources, start table (an entry and the next one in a word: one load) and nd places per
// source.
struct PhasedTable {
    const PhasedSource *sources;
    const uint32_t *ranges;   // starts[g] | starts[g + 1] << 16
    char *const *dsts;
    uint32_t shift : 8;   // in one word, so that both come with one load
    uint32_t nd : 24;
    uint32_t tiles;
};
constexpr uint32_t kPhasedTableGroups = 4096;
// The same for an AllGather(V), in the kernel arguments: every place of a source is the same offset into the ranks'
// receive buffers.
constexpr uint32_t kPhasedInlineGroups = 480;
struct PhasedInline {
    char *base[kMaxVRanks];
    PhasedSource sources[kMaxVRanks];
    uint32_t ranges[kPhasedInlineGroups / 2];   // sixteen bits each, starts[g] | starts[g + 1] << 8
    uint32_t shift;
    uint32_t tiles;
};
// Tiles of a source whatever the alignment of its places (their tile grids differ by less than a tile).
__host__ __device__ inline uint64_t phased_tiles_of(uint64_t bytes)
{
    return bytes == 0 ? 0 : (bytes / 16 + 63) / (kPhasedTile / 16) + 1;
}
struct AgvTablesInline {
    uint64_t counts[kMaxVRanks];
    uint64_t displs[kMaxVRanks];
    __device__ uint64_t count(uint32_t i) const { return counts[i]; }
    __device__ uint64_t displ(uint32_t i) const { return displs[i]; }
};

// Workgroups of kThreads work-items that one launch takes along x: HIP allows fewer than 2^32 work-items there.
constexpr uint64_t kMostBlocksX = 0xffffffffull / kThreads;

// tiles: of all blocks
hipError_t launch_copy_blocks(const BlockTable &tab, size_t blocks, uint64_t tiles, hipStream_t stream);
hipError_t launch_equal_blocks(const EqualBlocks &tab, uint32_t n, hipStream_t stream);
hipError_t launch_alltoallv_inline(const A2avInline &tab, uint64_t tiles, hipStream_t stream);
// One batch after the other (grid z), each to one place after the other (grid y): per_batch tiles, a multiple of eight.
struct PhasedGrid {
    uint32_t per_batch;
    uint32_t batches;
    uint32_t nd;
};
hipError_t launch_phased_copy(const PhasedTable &tab, const PhasedGrid &grid, hipStream_t stream);
hipError_t launch_phased_copy_inline(const PhasedInline &tab, const PhasedGrid &grid, hipStream_t stream);
hipError_t launch_allgatherv_inline(const VRankPtrs &ptrs, const AgvTablesInline &tabs, uint32_t n, uint32_t esz,
                                    uint32_t grid, uint32_t tiles_per_block, hipStream_t stream);

// send_counts / sdispls / rdispls: device pointers, uint64 elements, row-major n x n.
hipError_t launch_alltoallv(const VRankPtrs &ptrs, const uint64_t *send_counts, const uint64_t *sdispls,
                            const uint64_t *rdispls, uint32_t n, uint32_t esz, uint32_t grid, uint32_t tiles_per_block,
                            hipStream_t stream);

// counts / displs: device pointers, uint64 elements, n entries.
hipError_t launch_displs_from_counts(const uint64_t *counts, uint32_t rows, uint32_t n, uint64_t *displs, uint64_t *totals,
                                     hipStream_t stream);
hipError_t launch_allgatherv(const VRankPtrs &ptrs, const uint64_t *counts, const uint64_t *displs, uint32_t n,
                             uint32_t esz, uint32_t grid, uint32_t tiles_per_block, hipStream_t stream);
}  // namespace hcclx
