// The tables that the copy kernels' launches are made of, checked tile by tile on the CPU (tests/test_host_copy_tables.py
// builds it against the library and runs it; nothing here touches a GPU).
//   blocks n  c00 c01 ...    an AlltoAllV's n x n counts (bytes): every tile of every block is found exactly once
// Prints "tiles <blocks' own> groups <g> bytes <of the table>", or what is wrong.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "hcclx_internal.h"

using namespace hcclx;

namespace {

static_assert((kMostBlocksX + 1) * kThreads > 0xffffffffull && kMostBlocksX * kThreads <= 0xffffffffull, "work-items along x of one launch");

int wrong(const char *what, uint64_t at)
{
    std::printf("wrong: %s at %llu\n", what, static_cast<unsigned long long>(at));
    return 1;
}

// The look-up of k_copy_blocks.
size_t block_of(const std::vector<uint32_t> &starts, uint32_t shift, const std::vector<uint64_t> &begin, uint64_t tile)
{
    uint32_t lo = starts[tile >> shift];
    uint32_t hi = starts[(tile >> shift) + 1];
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (begin[mid] <= tile) {
            lo = mid;
        } else {
            hi = mid - 1;
        }
    }
    return lo;
}

int every_tile(const std::vector<uint32_t> &starts, uint32_t shift, const std::vector<uint64_t> &begin, const std::vector<uint64_t> &tiles)
{
    uint64_t next = 0;
    for (size_t b = 0; b < begin.size(); ++b) {
        if (begin[b] != next) return wrong("first tile of block", b);
        for (uint64_t t = 0; t < tiles[b]; ++t, ++next) {
            if ((next >> shift) + 1 >= starts.size()) return wrong("no group for tile", next);
            if (block_of(starts, shift, begin, next) != b) return wrong("block of tile", next);
        }
    }
    if (starts.size() != ((next - 1) >> shift) + 2) return wrong("number of groups", starts.size());
    return 0;
}

int blocks(int argc, char **argv)
{
    const uint32_t n = static_cast<uint32_t>(std::strtoul(argv[0], nullptr, 10));
    if (argc != static_cast<int>(1 + n * n)) return wrong("argument count", argc);
    std::vector<uint64_t> counts(n * n), sdispls(n * n), rdispls(n * n);
    for (uint32_t k = 0; k < n * n; ++k) counts[k] = std::strtoull(argv[1 + k], nullptr, 10);
    std::vector<const void *> send(n);
    std::vector<void *> recv(n);
    for (uint32_t i = 0; i < n; ++i) {
        send[i] = reinterpret_cast<const void *>((2ull * i + 1) << 44);
        recv[i] = reinterpret_cast<void *>((2ull * i + 2) << 44 | (i * 5 % 64));
        for (uint32_t j = 1; j < n; ++j) {
            sdispls[i * n + j] = sdispls[i * n + j - 1] + counts[i * n + j - 1];
            rdispls[i * n + j] = rdispls[i * n + j - 1] + counts[(j - 1) * n + i];
        }
    }
    BlockLaunch l;
    l.tiles = list_alltoallv_blocks(send.data(), recv.data(), counts.data(), sdispls.data(), rdispls.data(), n, 1, &l.blocks);
    uint64_t own = 0;
    std::vector<uint64_t> begin, tiles;
    for (const CopyBlock &b : l.blocks) {
        begin.push_back(b.begin);
        tiles.push_back(v_tiles_of(b.bytes, reinterpret_cast<uint64_t>(b.dst), 1));
        own += tiles.back();
    }
    if (l.tiles != own) return wrong("number of tiles", l.tiles);
    l.index();
    if (l.starts.size() > kBlockTableGroups + 1) return wrong("groups in memory", l.starts.size());
    if (every_tile(l.starts, l.shift, begin, tiles) != 0) return 1;
    std::vector<char> table(l.bytes());
    l.fill(table.data());
    const BlockTable t = l.table(table.data());
    if (std::memcmp(t.blocks, l.blocks.data(), l.blocks.size() * sizeof(CopyBlock)) != 0 || t.starts[l.starts.size() - 1] != l.blocks.size() - 1) {
        return wrong("table", 0);
    }
    if (n <= kA2avInlineRanks) {   // the table of the kernel arguments lists the empty blocks too
        std::vector<uint64_t> all_begin, all_tiles;
        uint64_t at = 0;
        for (uint32_t i = 0; i < n; ++i) {
            for (uint32_t j = 0; j < n; ++j) {
                all_begin.push_back(at);
                all_tiles.push_back(v_tiles_of(counts[i * n + j], reinterpret_cast<uint64_t>(recv[j]) + rdispls[j * n + i], 1));
                at += all_tiles.back();
            }
        }
        std::vector<uint32_t> starts;
        uint32_t shift = 0;
        index_tiles(all_begin.data(), all_begin.size(), at, kA2avInlineGroups, &starts, &shift);
        if (starts.size() > 4 * (sizeof(A2avInline::starts) / 4)) return wrong("groups in the kernel arguments", starts.size());
        if (every_tile(starts, shift, all_begin, all_tiles) != 0) return 1;
    }
    std::printf("tiles %llu groups %zu bytes %zu\n", static_cast<unsigned long long>(own), l.starts.size() - 1, l.bytes());
    return 0;
}

}  // namespace

int main(int argc, char **argv)
{
    if (argc > 2 && std::string(argv[1]) == "blocks") return blocks(argc - 2, argv + 2);
    return wrong("arguments", 0);
}
