// The tables that the copy kernels' launches are made of, checked tile by tile on the CPU (tests/test_host_copy_tables.py
// builds it against the library and runs it; nothing here touches a GPU).
//   blocks n  c00 c01 ...    an AlltoAllV's n x n counts (bytes): every tile of every block is found exactly once
//       prints "tiles <blocks' own> groups <g> bytes <of the table>"
//   copies max_groups  bytes:places[xtimes] ...    sources that go to several places: every tile of every place is found exactly
//       once; prints "tiles <of all places> workgroups <of all launches> launches <l> bytes <of the largest table>"
//   waves pieces per_tile waves    whether one launch of the wavefront fold takes them: prints 1 or 0
// or what is wrong.
#include <algorithm>
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

int copies(int argc, char **argv)
{
    const uint32_t max_groups = static_cast<uint32_t>(std::strtoul(argv[0], nullptr, 10));
    std::vector<PhasedStream> streams;
    for (int k = 1; k < argc; ++k) {
        unsigned long long bytes = 0;
        unsigned places = 0, times = 1;
        if (std::sscanf(argv[k], "%llu:%ux%u", &bytes, &places, &times) < 2) return wrong("source", k);
        for (unsigned t = 0; t < times; ++t) {
            const uint64_t i = streams.size();
            PhasedStream s{reinterpret_cast<const char *>((i + 1) << 33), bytes, {}};
            for (unsigned d = 0; d < places; ++d) s.dst.push_back(reinterpret_cast<char *>((i + 1) << 33 | (1ull << 56) | (d + 1ull) << 50 | (3 * i + 7 * d) % 64));
            streams.push_back(std::move(s));
        }
    }
    const std::vector<PhasedStream> asked = streams;
    std::vector<PhasedLaunch> launches;
    build_phased(streams, 16ull << 20, max_groups, &launches);
    uint64_t own = 0, workgroups = 0, most_bytes = 0;
    std::vector<std::vector<std::vector<bool>>> moved(asked.size());
    for (size_t s = 0; s < asked.size(); ++s) {
        for (char *dst : asked[s].dst) {
            const uint64_t tiles = v_tiles_of(asked[s].bytes, reinterpret_cast<uint64_t>(dst), kPhasedUnroll);
            own += tiles;
            moved[s].push_back(std::vector<bool>(tiles));
        }
    }
    for (const PhasedLaunch &l : launches) {
        if (l.ranges.size() > max_groups) return wrong("groups of a launch", l.ranges.size());
        if (l.bytes() > 1u << 20) return wrong("table of a launch", l.bytes());
        most_bytes = std::max<uint64_t>(most_bytes, l.bytes());
        const uint64_t x = l.grid.per_batch;
        if (x > kMostBlocksX || x % 8 != 0 || l.grid.nd > 65535 || l.grid.batches > 65535) return wrong("grid", x);
        workgroups += x * l.grid.nd * l.grid.batches;
        std::vector<char> table(l.bytes());
        l.fill(table.data());
        const PhasedTable t = l.table(table.data());
        if (t.tiles > x * l.grid.batches) return wrong("tiles of a launch", t.tiles);
        std::vector<uint32_t> starts;
        for (size_t g = 0; g < l.ranges.size(); ++g) {
            if (g != 0 && starts[g] != (t.ranges[g] & 0xffffu)) return wrong("range of group", g);
            if (g == 0) starts.push_back(t.ranges[0] & 0xffffu);
            starts.push_back(t.ranges[g] >> 16);
        }
        std::vector<uint64_t> begin;
        for (size_t k = 0; k < l.sources.size(); ++k) begin.push_back(k == 0 ? 0 : t.sources[k].begin);
        for (uint64_t tile = 0; tile < t.tiles; ++tile) {
            if ((tile >> t.shift) + 1 >= starts.size()) return wrong("no group for tile", tile);
            const size_t k = block_of(starts, t.shift, begin, tile);
            const PhasedSource &source = t.sources[k];
            const size_t s = (reinterpret_cast<uint64_t>(source.src) >> 33) - 1;
            if (s >= asked.size() || source.bytes != asked[s].bytes || source.place != asked[s].dst.size()) return wrong("source of tile", tile);
            const uint32_t tl = static_cast<uint32_t>(tile) - source.begin;
            for (uint32_t d = 0; d < source.place; ++d) {
                if (t.dsts[static_cast<uint64_t>(k) * t.nd + d] != asked[s].dst[d]) return wrong("place of tile", tile);
                if (tl >= moved[s][d].size()) continue;
                if (moved[s][d][tl]) return wrong("tile moved twice, source", s);
                moved[s][d][tl] = true;
            }
        }
    }
    for (size_t s = 0; s < asked.size(); ++s) {
        for (const auto &tiles : moved[s]) {
            for (bool m : tiles) {
                if (!m) return wrong("tile not moved, source", s);
            }
        }
    }
    std::printf("tiles %llu workgroups %llu launches %zu bytes %llu\n", static_cast<unsigned long long>(own),
                static_cast<unsigned long long>(workgroups), launches.size(), static_cast<unsigned long long>(most_bytes));
    return 0;
}

}  // namespace

int main(int argc, char **argv)
{
    if (argc > 3 && std::string(argv[1]) == "copies") return copies(argc - 2, argv + 2);
    if (argc == 5 && std::string(argv[1]) == "waves") {
        std::printf("%d\n", waves_fit(std::strtoull(argv[2], nullptr, 10), std::atoi(argv[3]), std::atoi(argv[4])) ? 1 : 0);
        return 0;
    }
    if (argc > 2 && std::string(argv[1]) == "blocks") return blocks(argc - 2, argv + 2);
    return wrong("arguments", 0);
}
