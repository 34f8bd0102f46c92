// Ragged data movement of the V collectives: AlltoAllV pack/unpack and AllGatherV, for n virtual ranks
// whose buffers live in one GPU.
//
// Reference behaviour restated (one copy instead of the reference's pack -> CCL slot -> unpack pair):
//   AlltoAllV  in_i[sdispls_i[j] .. +sendCounts_i[j])  ->  out_j[rdispls_j[i] .. )
//              src/ops/all_to_all_v/template/aicpu/ins_temp_all_to_all_v_mesh_1D.cc:304-308 (pack into the
//              peer's CCL slot), :431-438 (unpack), :161-170 (self block)
//   AllGatherV out_j[displs[i] .. +counts[i]) = in_i[0 .. counts[i])   for all i, j
//              src/ops/all_gather_v/template/aicpu/ins_temp_all_gather_v_mesh_1D.cc:97-242;
//              contract include/hccl.h:120-135
//
// The count/displacement tables stay on the device.  Each workgroup stages the per-block tile counts in
// LDS, turns them into an inclusive prefix with a wavefront scan, and then walks tile numbers in a
// grid-stride loop, locating a tile's (source, destination) block by binary search in LDS.  No host
// round trip is needed when the tables come from an on-device router.
//
// Bound: HBM bandwidth.  Algorithmic bytes: AlltoAllV 2 x payload; AllGatherV (1 + n) x payload moved,
// 2n x payload delivered.
#include "fold.h"
#include "vops.h"

namespace hcclx {

namespace {

__device__ __forceinline__ uint64_t wave_inclusive_scan(uint64_t v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t lo = __shfl_up(static_cast<uint32_t>(v), d, 64);
        const uint32_t hi = __shfl_up(static_cast<uint32_t>(v >> 32), d, 64);
        if (lane >= d) v += (static_cast<uint64_t>(hi) << 32) | lo;
    }
    return v;
}

// In place: s_tab[0..m) (per-block tile counts) becomes its inclusive prefix sum.  m <= 4096.
// Each thread sums a contiguous run, a wavefront scan orders the 64 runs of a wave, and the four wave
// totals are combined through LDS.
__device__ void block_inclusive_scan(uint64_t *s_tab, uint32_t m, uint64_t *s_wave)
{
    const uint32_t per = (m + kThreads - 1) / kThreads;
    const uint32_t b = threadIdx.x * per;
    const uint32_t e = (b + per < m) ? b + per : m;
    uint64_t sum = 0;
    for (uint32_t i = b; i < e; ++i) sum += s_tab[i];
    const uint64_t incl = wave_inclusive_scan(sum);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 63) s_wave[wave] = incl;
    __syncthreads();
    uint64_t base = incl - sum;
    for (int w = 0; w < wave; ++w) base += s_wave[w];
    for (uint32_t i = b; i < e; ++i) {
        base += s_tab[i];
        s_tab[i] = base;
    }
    __syncthreads();
}

__device__ __forceinline__ uint32_t find_block(const uint64_t *s_end, uint32_t m, uint64_t t)
{
    uint32_t lo = 0;
    uint32_t hi = m - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (s_end[mid] > t) {
            hi = mid;
        } else {
            lo = mid + 1;
        }
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

// One tile of a block copy: tile `tl` of a block of `bytes` bytes from src to dst[0..ndst) (all
// destinations share dst[0]'s alignment modulo 16, or lose only speed if they do not).
// kCached: the source is read with ordinary loads, so that workgroups that copy the same tile to another
// destination shortly afterwards find it in the L2; otherwise it streams past the caches.
template <bool kCached>
__device__ __forceinline__ u32x4 ld16c(const char *p)
{
    if constexpr (kCached) {
        return ld16_cached(p);
    } else {
        return ld16(p);
    }
}

// kPolicy: how the vectors are stored (fold.h).
template <int kCopyUnroll, bool kCached = false, uint32_t kPolicy = kStoreStream, typename DstFn>
__device__ __forceinline__ void copy_tile(const char *src, uint64_t dst0, uint64_t bytes, uint64_t tl, uint32_t ndst,
                                          DstFn dst_of)
{
    constexpr uint64_t kTileVecs = 256ull * kCopyUnroll;
    const uint64_t head = v_head_of(bytes, dst0);
    const uint64_t body = bytes - head;
    const uint64_t nvec = body / 16;
    const uint32_t shift = v_shift_of(head, dst0);
    // in the first tile of a shifted grid v0 wraps below zero for the vectors in front of the block and
    // fails the bound check below
    const uint64_t v0 = tl * kTileVecs + threadIdx.x - shift;
    const char *sb = src + head;
    if (tl * kTileVecs >= shift && (tl + 1) * kTileVecs - shift <= nvec) {
        u32x4 r[kCopyUnroll];
#pragma unroll
        for (int u = 0; u < kCopyUnroll; ++u) r[u] = ld16c<kCached>(sb + (v0 + static_cast<uint64_t>(u) * kThreads) * 16);
        for (uint32_t d = 0; d < ndst; ++d) {
            char *db = dst_of(d) + head;
#pragma unroll
            for (int u = 0; u < kCopyUnroll; ++u) st16x(db + (v0 + static_cast<uint64_t>(u) * kThreads) * 16, r[u], kPolicy);
        }
        return;
    }
    // first or last tile of the block: the vectors inside it; the last one also moves head and tail bytes
    u32x4 r[kCopyUnroll];
#pragma unroll
    for (int u = 0; u < kCopyUnroll; ++u) {
        const uint64_t vi = v0 + static_cast<uint64_t>(u) * kThreads;
        if (vi < nvec) r[u] = ld16c<kCached>(sb + vi * 16);
    }
    const uint64_t tail = body - nvec * 16;
    char edge = 0;
    uint64_t edge_off = 0;
    const bool has_edge = tl == (nvec + shift) / kTileVecs && threadIdx.x < head + tail;
    if (has_edge) {
        edge_off = (threadIdx.x < head) ? threadIdx.x : head + nvec * 16 + (threadIdx.x - head);
        edge = src[edge_off];
    }
    for (uint32_t d = 0; d < ndst; ++d) {
        char *dp = dst_of(d);
#pragma unroll
        for (int u = 0; u < kCopyUnroll; ++u) {
            const uint64_t vi = v0 + static_cast<uint64_t>(u) * kThreads;
            if (vi < nvec) st16x(dp + head + vi * 16, r[u], kPolicy);
        }
        if (has_edge) dp[edge_off] = edge;
    }
}

template <typename Ptrs, typename Tabs>
__global__ void __launch_bounds__(kThreads)
k_alltoallv(Ptrs ptrs, Tabs tabs, uint32_t n, uint32_t esz, uint32_t tiles_per_block)
{
    extern __shared__ uint64_t s_end[];  // n*n entries, then 4 wave totals
    const uint32_t m = n * n;
    uint64_t *s_wave = s_end + m;
    for (uint32_t p = threadIdx.x; p < m; p += kThreads) {
        const uint32_t i = p / n;
        const uint32_t j = p - i * n;
        const uint64_t dst = reinterpret_cast<uint64_t>(ptrs.recv[j]) + tabs.rdispl(j * n + i) * esz;
        s_end[p] = v_tiles_of(tabs.count(p) * esz, dst, kA2avUnroll);
    }
    __syncthreads();
    block_inclusive_scan(s_end, m, s_wave);
    const uint64_t total = s_end[m - 1];

    // A workgroup takes runs of tiles_per_block consecutive tiles, so that the table set-up above is
    // paid once per run.
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * tiles_per_block;
    for (uint64_t run = static_cast<uint64_t>(blockIdx.x) * tiles_per_block; run < total; run += stride)
    for (uint64_t t = run; t < run + tiles_per_block && t < total; ++t) {
        const uint32_t p = find_block(s_end, m, t);
        const uint64_t tl = uniform64(t - (p ? s_end[p - 1] : 0));
        const uint32_t i = p / n;
        const uint32_t j = p - i * n;
        const uint64_t bytes = tabs.count(p) * esz;
        const char *src = ptrs.send[i] + tabs.sdispl(p) * esz;
        char *dst = ptrs.recv[j] + tabs.rdispl(j * n + i) * esz;
        copy_tile<kA2avUnroll>(src, reinterpret_cast<uint64_t>(dst), bytes, tl, 1, [=](uint32_t) { return dst; });
    }
}

// The first and the last block (or source) that a tile of group g can lie in.
struct Range {
    uint32_t lo, hi;
};
__device__ __forceinline__ Range range_of(const BlockTable &t, uint32_t g) { return {t.starts[g], t.starts[g + 1]}; }
__device__ __forceinline__ Range range_of(const A2avInline &t, uint32_t g)
{
    return {t.starts[g >> 2] >> (g & 3u) * 8 & 255u, t.starts[(g + 1) >> 2] >> ((g + 1) & 3u) * 8 & 255u};
}
__device__ __forceinline__ uint64_t begin_of(const BlockTable &t, uint32_t b) { return t.blocks[b].begin; }
__device__ __forceinline__ uint64_t begin_of(const A2avInline &t, uint32_t b) { return t.begin[b]; }
__device__ __forceinline__ CopyBlock block_of(const BlockTable &t, uint32_t b) { return t.blocks[b]; }
__device__ __forceinline__ CopyBlock block_of(const A2avInline &t, uint32_t b)
{
    const uint32_t i = b * t.inv_n >> 16;
    const uint32_t j = b - i * t.n;
    return {t.send[i] + static_cast<uint64_t>(t.sdispls[b]) * t.esz, t.recv[j] + static_cast<uint64_t>(t.rdispls[b]) * t.esz,
            static_cast<uint64_t>(t.counts[b]) * t.esz, t.begin[b]};
}

__device__ __forceinline__ Range range_of(const PhasedTable &t, uint32_t g) { return {t.ranges[g] & 0xffffu, t.ranges[g] >> 16}; }
__device__ __forceinline__ Range range_of(const PhasedInline &t, uint32_t g)
{
    const uint32_t one = t.ranges[g >> 1] >> (g & 1u) * 16;
    return {one & 255u, one >> 8 & 255u};
}
__device__ __forceinline__ uint32_t begin_of(const PhasedTable &t, uint32_t s) { return t.sources[s].begin; }
__device__ __forceinline__ uint32_t begin_of(const PhasedInline &t, uint32_t s) { return t.sources[s].begin; }

// The last block (or source) that begins at a tile or in front of it.
template <typename Tab, typename N> __device__ __forceinline__ uint32_t at_tile(const Tab &tab, N tile)
{
    const Range r = range_of(tab, static_cast<uint32_t>(tile >> tab.shift));
    uint32_t lo = r.lo;
    uint32_t hi = r.hi;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (begin_of(tab, mid) <= tile) {
            lo = mid;
        } else {
            hi = mid - 1;
        }
    }
    return lo;
}

// Blocks of any lengths, one 4 KiB tile per workgroup and one vector per thread, mostly stored through the L2: bound by HBM.
// A wavefront that loads and stores one vector per lane copies faster than one that moves two (1 GiB: 6.66 against
// 6.22 TB/s with these stores, 6.54 streamed); 8 x 4096 x 7168 bf16 with two vectors, streamed, and the block searched
// in a prefix: 151.3 us, this way 145.4.  One workgroup per tile and none besides: an idle one costs 0.23 ns, and with blocks
// cut into slabs of one size (two scalar loads without a search) 63 ranks that send 512 MiB, Zipf, launch fifteen for
// every tile: 629 us, this way 205; 15 ranks 185 and 178, 32 ranks with blocks of nearly one size 114 and 101.
template <typename Tab, uint32_t kPolicy>
__global__ void __launch_bounds__(kThreads) k_copy_blocks(Tab tab, uint64_t first)
{
    const uint64_t tile = first + blockIdx.x;
    const CopyBlock b = block_of(tab, at_tile(tab, tile));
    char *dst = b.dst;
    copy_tile<1, false, kPolicy>(b.src, reinterpret_cast<uint64_t>(dst), b.bytes, tile - b.begin, 1, [=](uint32_t) { return dst; });
}

// Equal blocks: nothing to look up and no table to bring, the block is the workgroup's place in the grid (x: tile, y:
// destination, z: source).  32 ranks x 32 x 2049 bf16: 3.4 us of table upload in front of the copy less, and the host
// builds no table of 1024 blocks.
__global__ void __launch_bounds__(kThreads) k_equal_blocks(EqualBlocks tab)
{
    const uint64_t bytes = tab.bytes;
    const char *src = tab.send[blockIdx.z] + blockIdx.y * bytes;
    char *dst = tab.recv[blockIdx.y] + blockIdx.z * bytes;
    if (blockIdx.x >= v_tiles_of(bytes, reinterpret_cast<uint64_t>(dst), 1)) return;
    copy_tile<1, false, kStoreThrough>(src, reinterpret_cast<uint64_t>(dst), bytes, blockIdx.x, 1, [=](uint32_t) { return dst; });
}

// null: the source has no such place (the table has nd of them for every source)
__device__ __forceinline__ char *phased_dst(const PhasedTable &t, uint32_t k, const PhasedSource &, uint32_t d)
{
    return t.dsts[k * t.nd + d];
}
__device__ __forceinline__ char *phased_dst(const PhasedInline &t, uint32_t, const PhasedSource &source, uint32_t d) { return t.base[d] + source.place; }

// Sources to several places, one place at a time.  Workgroups start in the order of their numbers (x: tile of the
// batch, y: place, z: batch), so a batch is written to its first place, then to the second, and so on.  At any moment
// the GPU writes ONE output instead of n at once, which HBM takes faster (one source to eight outputs, every workgroup
// storing to all eight: 5.5 TB/s at the pins; this way 6.4-6.5); the re-reads of the batch come from the L2s, not from
// HBM.  The place of a workgroup follows from its number with mostly two dependent scalar loads: a table search in front
// of a tile costs a fifth of the kernel's time.  No workgroup is idle but at the end of a batch and of a place that is aligned
// better than the worst; with sources cut into slabs of one size, 5000 x 64 KiB to eight places took 15214 us (this way 565),
// 64 MiB beside 4090 x 4 KiB 12567 (140), 900 x 70001 bytes to three 47.4 (40), and the AllGather of 8 x 64 MiB 754 (755).
template <typename Tab>
__global__ void __launch_bounds__(kThreads) k_phased_copy(Tab tab, uint32_t per_batch)
{
    const uint32_t tile = blockIdx.z * per_batch + blockIdx.x;
    if (tile >= tab.tiles) return;
    const uint32_t k = at_tile(tab, tile);
    const PhasedSource source = tab.sources[k];
    char *dst = phased_dst(tab, k, source, blockIdx.y);
    const uint32_t tl = tile - source.begin;
    // (one test: with a branch for each the look-ups would wait for one another)
    if ((dst == nullptr) | (tl > v_last_tile_of(source.bytes, reinterpret_cast<uint64_t>(dst), kPhasedUnroll))) return;
    copy_tile<kPhasedUnroll, true>(source.src, reinterpret_cast<uint64_t>(dst), source.bytes, tl, 1, [=](uint32_t) { return dst; });
}

template <typename Tabs>
__global__ void __launch_bounds__(kThreads)
k_allgatherv(VRankPtrs ptrs, Tabs tabs, uint32_t n, uint32_t esz, uint32_t tiles_per_block)
{
    extern __shared__ uint64_t s_end[];  // n entries, then 4 wave totals
    uint64_t *s_wave = s_end + n;
    for (uint32_t i = threadIdx.x; i < n; i += kThreads) {
        const uint64_t dst = reinterpret_cast<uint64_t>(ptrs.recv[0]) + tabs.displ(i) * esz;
        s_end[i] = v_tiles_of(tabs.count(i) * esz, dst, kAgvUnroll);
    }
    __syncthreads();
    block_inclusive_scan(s_end, n, s_wave);
    const uint64_t total = s_end[n - 1];

    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * tiles_per_block;
    for (uint64_t run = static_cast<uint64_t>(blockIdx.x) * tiles_per_block; run < total; run += stride)
    for (uint64_t t = run; t < run + tiles_per_block && t < total; ++t) {
        const uint32_t i = find_block(s_end, n, t);
        const uint64_t tl = uniform64(t - (i ? s_end[i - 1] : 0));
        const uint64_t bytes = tabs.count(i) * esz;
        const uint64_t off = tabs.displ(i) * esz;
        const char *src = ptrs.send[i];
        copy_tile<kAgvUnroll>(src, reinterpret_cast<uint64_t>(ptrs.recv[0]) + off, bytes, tl, n,
                  [&](uint32_t d) { return ptrs.recv[d] + off; });
    }
}

}  // namespace

hipError_t launch_alltoallv(const VRankPtrs &ptrs, const uint64_t *send_counts, const uint64_t *sdispls,
                            const uint64_t *rdispls, uint32_t n, uint32_t esz, uint32_t grid, uint32_t tiles_per_block,
                            hipStream_t stream)
{
    const size_t lds = (static_cast<size_t>(n) * n + 4) * sizeof(uint64_t);
    const A2avTablesPtr tabs{send_counts, sdispls, rdispls};
    HCCLX_LAUNCH((k_alltoallv<VRankPtrs, A2avTablesPtr>), dim3(grid), dim3(kThreads), lds, stream, ptrs, tabs, n,
                       esz, tiles_per_block);
    return hipGetLastError();
}

namespace {
// 64 GiB and more take several launches.
template <uint32_t kPolicy, typename Tab> hipError_t launch_tiles(const Tab &tab, uint64_t tiles, hipStream_t stream)
{
    for (uint64_t first = 0; first < tiles; first += kMostBlocksX) {
        const uint64_t take = tiles - first < kMostBlocksX ? tiles - first : kMostBlocksX;
        HCCLX_LAUNCH((k_copy_blocks<Tab, kPolicy>), dim3(static_cast<uint32_t>(take)), dim3(kThreads), 0, stream, tab, first);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
}  // namespace

// Many blocks (more than 22 ranks) and more than the Infinity Cache takes up: streamed.  Plans, before the blocks were stored
// through the L2 : through : streamed, us: 32 ranks with blocks of nearly one size 384 MiB in all 141 : 146 : 139, 256 MiB
// 98.9 : 98.8 : 93; 48 x 192 MiB 72.9 : 74.7 : 72.2; 64 x 384 MiB 144 : 152 : 144, Zipf 256 MiB 94.1 : 103.5 : 96.1.  128 MiB and less
// through the L2 (64 ranks 48.0 : 49.4 : 49.1, 32 ranks 48.0 : 46.2 : 47.8, 16 x 32 MiB 14.2 : 13.1 : 14.2), and few blocks at
// every size (16 ranks, Zipf, 1 GiB 365 : 333 : 341; 8 ranks 351 : 328 : 333).
hipError_t launch_copy_blocks(const BlockTable &tab, size_t blocks, uint64_t tiles, hipStream_t stream)
{
    constexpr size_t kStreamBlocks = 512;
    constexpr uint64_t kStreamTiles = (160ull << 20) / 4096;
    return blocks >= kStreamBlocks && tiles >= kStreamTiles ? launch_tiles<kStoreStream>(tab, tiles, stream)
                                                            : launch_tiles<kStoreThrough>(tab, tiles, stream);
}

hipError_t launch_equal_blocks(const EqualBlocks &tab, uint32_t n, hipStream_t stream)
{
    // tiles of a block whatever the alignment of its place: up to 63 vectors in front of it in the tile grid
    const uint64_t tiles = (tab.bytes / 16 + 63) / 256 + 1;
    HCCLX_LAUNCH(k_equal_blocks, dim3(static_cast<uint32_t>(tiles), n, n), dim3(kThreads), 0, stream, tab);
    return hipGetLastError();
}

hipError_t launch_alltoallv_inline(const A2avInline &tab, uint64_t tiles, hipStream_t stream)
{
    return launch_tiles<kStoreThrough>(tab, tiles, stream);
}

namespace {
template <typename Tab> hipError_t launch_phased(const Tab &tab, const PhasedGrid &g, hipStream_t stream)
{
    HCCLX_LAUNCH((k_phased_copy<Tab>), dim3(g.per_batch, g.nd, g.batches), dim3(kThreads), 0, stream, tab, g.per_batch);
    return hipGetLastError();
}
}  // namespace

hipError_t launch_phased_copy(const PhasedTable &tab, const PhasedGrid &grid, hipStream_t stream)
{
    return launch_phased(tab, grid, stream);
}

hipError_t launch_phased_copy_inline(const PhasedInline &tab, const PhasedGrid &grid, hipStream_t stream)
{
    return launch_phased(tab, grid, stream);
}

// One wavefront per row of n <= 64 counts: displs = exclusive prefix sum, totals[row] = the row's sum.
__global__ void __launch_bounds__(64)
k_displs_from_counts(const uint64_t *__restrict__ counts, uint32_t n, uint64_t *__restrict__ displs,
                     uint64_t *__restrict__ totals)
{
    const uint64_t row = blockIdx.x;
    const uint32_t lane = threadIdx.x;
    const uint64_t c = lane < n ? counts[row * n + lane] : 0;
    const uint64_t incl = wave_inclusive_scan(c);
    if (lane < n) displs[row * n + lane] = incl - c;
    if (totals != nullptr && lane == n - 1) totals[row] = incl;
}

hipError_t launch_displs_from_counts(const uint64_t *counts, uint32_t rows, uint32_t n, uint64_t *displs, uint64_t *totals,
                                     hipStream_t stream)
{
    HCCLX_LAUNCH(k_displs_from_counts, dim3(rows), dim3(64), 0, stream, counts, n, displs, totals);
    return hipGetLastError();
}

hipError_t launch_allgatherv(const VRankPtrs &ptrs, const uint64_t *counts, const uint64_t *displs, uint32_t n,
                             uint32_t esz, uint32_t grid, uint32_t tiles_per_block, hipStream_t stream)
{
    const size_t lds = (static_cast<size_t>(n) + 4) * sizeof(uint64_t);
    const AgvTablesPtr tabs{counts, displs};
    HCCLX_LAUNCH((k_allgatherv<AgvTablesPtr>), dim3(grid), dim3(kThreads), lds, stream, ptrs, tabs, n, esz,
                       tiles_per_block);
    return hipGetLastError();
}

hipError_t launch_allgatherv_inline(const VRankPtrs &ptrs, const AgvTablesInline &tabs, uint32_t n, uint32_t esz,
                                    uint32_t grid, uint32_t tiles_per_block, hipStream_t stream)
{
    const size_t lds = (static_cast<size_t>(n) + 4) * sizeof(uint64_t);
    HCCLX_LAUNCH((k_allgatherv<AgvTablesInline>), dim3(grid), dim3(kThreads), lds, stream, ptrs, tabs, n, esz,
                       tiles_per_block);
    return hipGetLastError();
}

}  // namespace hcclx
