// The caller side of an MoE AlltoAllV, for n virtual ranks at once: routing tables from per-entry
// destinations (stable grouping by destination rank), the row gather that packs the send buffers, and the
// inverse that combines what comes back.  C-ABI entry points: hcclx_moe_* in include/hcclx.h.
//
// The reference has no such step: its AlltoAllV takes finished send buffers and tables.  The nearest code is
// the staging either side of the transfer, PreCopy / PostCopy of InsTempAlltoAllVMesh1D
// (src/ops/all_to_all_v/template/aicpu/ins_temp_all_to_all_v_mesh_1D.cc:412-440).
//
// Bound: HBM bandwidth (pack / combine move rows of several KiB); the routing kernels touch 4 bytes per
// entry and are latency-bound.  Algorithmic bytes: pack 2 x entries x row bytes; combine (topk + 1) x
// tokens x row bytes.  hcclx_moe_dispatch and hcclx_moe_gather_combine do pack + AlltoAllV, and AlltoAllV back
// + combine, in one pass each: the rows go straight to (come straight from) the place the AlltoAllV would
// have put them, which halves the traffic of either direction.
#include "hcclx.h"
#include "hcclx_internal.h"
#include "kernels/elem.h"
#include "kernels/fold.h"

#include <cstring>

using namespace hcclx;

namespace {

constexpr uint32_t kMoeMaxRanks = 64;
constexpr uint32_t kMoeChunk = 256;        // entries per workgroup of the routing kernels
constexpr uint32_t kDropped = 0xffffffffu;  // perm value of an entry whose destination is out of range

struct MoeConstPtrs {
    const void *p[kMoeMaxRanks];
};
struct MoePtrs {
    void *p[kMoeMaxRanks];
};

__device__ __forceinline__ const MoePtrs &as_mutable_dev(const MoeConstPtrs &c)
{
    return reinterpret_cast<const MoePtrs &>(c);   // same layout; the landing addresses are only read through
}

MoePtrs as_mutable(const MoeConstPtrs &c)
{
    MoePtrs m;
    for (uint32_t i = 0; i < kMoeMaxRanks; ++i) m.p[i] = const_cast<void *>(c.p[i]);
    return m;
}

// Workspace layout (uint32): base[n][n][chunks] (chunk fastest) -- first the per-chunk histogram, then,
// in place, its exclusive prefix over the chunks -- followed by row_start[n][n].
__host__ __device__ inline uint32_t chunks_of(uint32_t entries) { return (entries + kMoeChunk - 1) / kMoeChunk; }

__global__ void __launch_bounds__(kMoeChunk)
k_moe_hist(MoeConstPtrs dest, uint32_t n, uint32_t entries, uint32_t chunks, uint32_t *base)
{
    __shared__ uint32_t s_hist[kMoeMaxRanks];
    const uint32_t c = blockIdx.x;
    const uint32_t i = blockIdx.y;
    if (threadIdx.x < kMoeMaxRanks) s_hist[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t e = c * kMoeChunk + threadIdx.x;
    if (e < entries) {
        const int32_t d = static_cast<const int32_t *>(dest.p[i])[e];
        if (d >= 0 && static_cast<uint32_t>(d) < n) atomicAdd(&s_hist[d], 1u);
    }
    __syncthreads();
    if (threadIdx.x < n) base[(static_cast<uint64_t>(i) * n + threadIdx.x) * chunks + c] = s_hist[threadIdx.x];
}

__device__ __forceinline__ uint32_t wave_scan_u32(uint32_t v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(v, d, 64);
        if (lane >= d) v += o;
    }
    return v;
}

// One workgroup per rank i: every (i, d) histogram row becomes its exclusive prefix over the chunks (a
// wavefront scans 64 chunks at a time); the row totals give send counts and displacements.
__global__ void __launch_bounds__(256)
k_moe_scan(uint32_t n, uint32_t chunks, uint64_t row_elems, uint32_t *base, uint32_t *row_start, uint64_t *send_counts,
           uint64_t *sdispls, uint64_t *recv_counts)
{
    __shared__ uint32_t s_total[kMoeMaxRanks];
    const uint32_t i = blockIdx.x;
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t lane = threadIdx.x & 63;
    for (uint32_t d = wave; d < n; d += 4) {
        uint32_t *row = base + (static_cast<uint64_t>(i) * n + d) * chunks;
        uint32_t running = 0;
        for (uint32_t c0 = 0; c0 < chunks; c0 += 64) {
            const uint32_t c = c0 + lane;
            const uint32_t v = c < chunks ? row[c] : 0;
            const uint32_t incl = wave_scan_u32(v);
            if (c < chunks) row[c] = running + incl - v;
            running += __shfl(incl, 63, 64);
        }
        if (lane == 0) s_total[d] = running;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t start = 0;
        for (uint32_t d = 0; d < n; ++d) {
            const uint32_t t = s_total[d];
            row_start[i * n + d] = start;
            send_counts[i * n + d] = static_cast<uint64_t>(t) * row_elems;
            sdispls[i * n + d] = static_cast<uint64_t>(start) * row_elems;
            recv_counts[d * n + i] = static_cast<uint64_t>(t) * row_elems;
            start += t;
        }
    }
}

// perm[e] = first row of the destination's group + entries of earlier chunks with that destination + rank of
// e among the entries of its own chunk with that destination (index order: the grouping is stable).
__global__ void __launch_bounds__(kMoeChunk)
k_moe_perm(MoeConstPtrs dest, MoePtrs perm, uint32_t n, uint32_t entries, uint32_t chunks, const uint32_t *base,
           const uint32_t *row_start, const uint64_t *send_counts, uint64_t *rdispls)
{
    // one workgroup also writes rdispls[j][i] = what ranks 0 .. i-1 send to rank j (the send counts are complete:
    // the scan kernel ran before this one)
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < n) {
        const uint32_t j = threadIdx.x;
        uint64_t run = 0;
        for (uint32_t i = 0; i < n; ++i) {
            rdispls[j * n + i] = run;
            run += send_counts[i * n + j];
        }
    }
    __shared__ uint32_t s_cnt[4][kMoeMaxRanks];
    const uint32_t c = blockIdx.x;
    const uint32_t i = blockIdx.y;
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t e = c * kMoeChunk + threadIdx.x;
    int32_t d = -1;
    if (e < entries) d = static_cast<const int32_t *>(dest.p[i])[e];
    const bool valid = d >= 0 && static_cast<uint32_t>(d) < n;
    uint32_t rank = 0;
    const unsigned long long below = (1ull << lane) - 1ull;
    for (uint32_t dd = 0; dd < n; ++dd) {
        const unsigned long long m = __ballot(valid && static_cast<uint32_t>(d) == dd);
        if (valid && static_cast<uint32_t>(d) == dd) rank = __popcll(m & below);
        if (lane == 0) s_cnt[wave][dd] = __popcll(m);
    }
    __syncthreads();
    if (e < entries) {
        uint32_t out = kDropped;
        if (valid) {
            uint32_t off = rank;
            for (uint32_t w = 0; w < wave; ++w) off += s_cnt[w][d];
            out = row_start[i * n + d] + base[(static_cast<uint64_t>(i) * n + d) * chunks + c] + off;
        }
        static_cast<uint32_t *>(perm.p[i])[e] = out;
    }
}

// The scan and permutation kernels in one launch, for tables small enough that every workgroup can afford to sum
// its rank's rows of the per-chunk histogram itself (at most kFusedChunks chunks per rank and kFusedCells histogram
// cells in all): two dependent launches instead of three.  Workgroup (c, i): per destination the entries of rank i
// in all chunks and in the chunks before c (one wavefront per destination, one lane per chunk), from them the first
// row of each destination's group, then the permutation of chunk c as in k_moe_perm.  The workgroups of chunk 0
// write their rank's rows of the count and displacement tables; workgroup (0, 0) also sums every rank's rows and
// writes rdispls.  base keeps the raw histogram.
constexpr uint32_t kFusedChunks = 64;
constexpr uint32_t kFusedCells = 16384;

__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}

__global__ void __launch_bounds__(kMoeChunk)
k_moe_scan_perm(MoeConstPtrs dest, MoePtrs perm, uint32_t n, uint32_t entries, uint32_t chunks, uint64_t row_elems,
                const uint32_t *base, uint64_t *send_counts, uint64_t *sdispls, uint64_t *recv_counts, uint64_t *rdispls)
{
    __shared__ uint32_t s_total[kMoeMaxRanks];
    __shared__ uint32_t s_before[kMoeMaxRanks];
    __shared__ uint32_t s_start[kMoeMaxRanks];
    __shared__ uint32_t s_cnt[4][kMoeMaxRanks];
    __shared__ uint32_t s_all[kMoeMaxRanks * kMoeMaxRanks];   // workgroup (0, 0): entries of rank i for destination j
    const uint32_t c = blockIdx.x;
    const uint32_t i = blockIdx.y;
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t lane = threadIdx.x & 63;
    for (uint32_t d = wave; d < n; d += 4) {
        const uint32_t v = lane < chunks ? base[(static_cast<uint64_t>(i) * n + d) * chunks + lane] : 0;
        const uint32_t total = wave_sum_u32(v);
        const uint32_t before = wave_sum_u32(lane < c ? v : 0);
        if (lane == 0) {
            s_total[d] = total;
            s_before[d] = before;
        }
    }
    if (c == 0 && i == 0) {
        for (uint32_t cell = threadIdx.x; cell < n * n; cell += kMoeChunk) {
            uint32_t t = 0;
            for (uint32_t k = 0; k < chunks; ++k) t += base[static_cast<uint64_t>(cell) * chunks + k];
            s_all[cell] = t;
        }
    }
    __syncthreads();
    if (wave == 0) {
        const uint32_t t = lane < n ? s_total[lane] : 0;
        const uint32_t incl = wave_scan_u32(t);
        s_start[lane] = incl - t;
        if (c == 0 && lane < n) {
            send_counts[i * n + lane] = static_cast<uint64_t>(t) * row_elems;
            sdispls[i * n + lane] = static_cast<uint64_t>(incl - t) * row_elems;
            recv_counts[lane * n + i] = static_cast<uint64_t>(t) * row_elems;
        }
    }
    if (c == 0 && i == 0 && threadIdx.x < n) {
        const uint32_t j = threadIdx.x;
        uint64_t run = 0;
        for (uint32_t r = 0; r < n; ++r) {
            rdispls[j * n + r] = run * row_elems;
            run += s_all[r * n + j];
        }
    }
    const uint32_t e = c * kMoeChunk + threadIdx.x;
    int32_t d = -1;
    if (e < entries) d = static_cast<const int32_t *>(dest.p[i])[e];
    const bool valid = d >= 0 && static_cast<uint32_t>(d) < n;
    uint32_t rank = 0;
    const unsigned long long below = (1ull << lane) - 1ull;
    for (uint32_t dd = 0; dd < n; ++dd) {
        const unsigned long long m = __ballot(valid && static_cast<uint32_t>(d) == dd);
        if (valid && static_cast<uint32_t>(d) == dd) rank = __popcll(m & below);
        if (lane == 0) s_cnt[wave][dd] = __popcll(m);
    }
    __syncthreads();
    if (e < entries) {
        uint32_t out = kDropped;
        if (valid) {
            uint32_t off = rank;
            for (uint32_t w = 0; w < wave; ++w) off += s_cnt[w][d];
            out = s_start[d] + s_before[d] + off;
        }
        static_cast<uint32_t *>(perm.p[i])[e] = out;
    }
}

// The whole routing in one launch, for so few entries per rank (kOneLaunchEntries) that every workgroup can count for
// itself.  Workgroup (c, i): a pass over the destinations of rank i gives, per destination, its
// entries and those in front of chunk c; then the permutation of chunk c as in k_moe_perm.  The workgroups of chunk 0 write
// their rank's rows of the count and displacement tables and, from a pass over all ranks' destinations, what every rank
// sends to rank i in front of which.  Bound by the latency of one launch and its rounds of loads.  Two launches : one, us: 8 ranks x 64
// entries 6.28 : 4.60, x 512 6.16 : 4.48, x 1024 6.21 : 4.96; 16 x 1024 8.00 : 6.64; 64 x 1024 25.2 : 18.2; 2 x 512 5.10 : 3.64,
// x 1024 5.30 : 4.06.
// No launch has more entries than kOneLaunchEntries: a thread holds that many / kMoeChunk of its rank's destinations and counts no
// others.  (In a loop over more of them two launches were faster: 8 x 4096 7.6 : 9.4, 16 x 2048 8.9 : 9.7.)
constexpr uint32_t kOneLaunchEntries = 1024;
static_assert(kOneLaunchEntries % kMoeChunk == 0, "every thread of a workgroup holds as many entries");

__global__ void __launch_bounds__(kMoeChunk)
k_moe_route_one(MoeConstPtrs dest, MoePtrs perm, uint32_t n, uint32_t entries, uint64_t row_elems, uint64_t *send_counts,
                uint64_t *sdispls, uint64_t *recv_counts, uint64_t *rdispls)
{
    __shared__ uint32_t s_total[kMoeMaxRanks];
    __shared__ uint32_t s_before[kMoeMaxRanks];
    __shared__ uint32_t s_start[kMoeMaxRanks];
    __shared__ uint32_t s_cnt[4][kMoeMaxRanks];
    __shared__ uint32_t s_from[kMoeMaxRanks];   // chunk 0: entries of each rank for destination i
    const uint32_t c = blockIdx.x;
    const uint32_t i = blockIdx.y;
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t lane = threadIdx.x & 63;
    const int32_t *mine = static_cast<const int32_t *>(dest.p[i]);
    // Every load that does not depend on another is issued here: the launch is little more than these round trips.  An entry
    // behind the last repeats it and is not counted.
    const uint32_t e = c * kMoeChunk + threadIdx.x;
    uint32_t d = static_cast<uint32_t>(mine[e < entries ? e : entries - 1]);
    constexpr int kPerThread = kOneLaunchEntries / kMoeChunk;
    uint32_t all[kPerThread];
#pragma unroll
    for (int u = 0; u < kPerThread; ++u) {
        const uint32_t at = u * kMoeChunk + threadIdx.x;
        all[u] = static_cast<uint32_t>(mine[at < entries ? at : entries - 1]);
    }
    // chunk 0: entries of rank r for rank i, a wavefront per rank, the loads of its next rank ahead of the count of this one
    constexpr int kAhead = 8;
    auto load_from = [&](uint32_t r, uint32_t first, uint32_t (&f)[kAhead]) {
        const int32_t *from = static_cast<const int32_t *>(dest.p[r]);
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const uint32_t at = first + u * 64 + lane;
            f[u] = static_cast<uint32_t>(from[at < entries ? at : entries - 1]);
        }
    };
    auto count_from = [&](uint32_t first, const uint32_t (&f)[kAhead]) {
        uint32_t count = 0;
#pragma unroll
        for (int u = 0; u < kAhead; ++u) count += first + u * 64 + lane < entries && f[u] == i ? 1u : 0u;
        return count;
    };
    uint32_t f[kAhead];
    if (c == 0) load_from(wave < n ? wave : 0, 0, f);
    if (threadIdx.x < kMoeMaxRanks) {
        s_total[threadIdx.x] = 0;
        s_before[threadIdx.x] = 0;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPerThread; ++u) {
        const uint32_t at = u * kMoeChunk + threadIdx.x;
        if (at < entries && all[u] < n) {
            atomicAdd(&s_total[all[u]], 1u);
            if (at < c * kMoeChunk) atomicAdd(&s_before[all[u]], 1u);
        }
    }
    if (c == 0) {
        for (uint32_t r = wave; r < n; r += 4) {
            uint32_t ahead[kAhead];
            load_from(r + 4 < n ? r + 4 : r, 0, ahead);
            uint32_t count = count_from(0, f);
            for (uint32_t first = kAhead * 64; first < entries; first += kAhead * 64) {
                load_from(r, first, f);
                count += count_from(first, f);
            }
            count = wave_sum_u32(count);
            if (lane == 0) s_from[r] = count;
#pragma unroll
            for (int u = 0; u < kAhead; ++u) f[u] = ahead[u];
        }
    }
    if (e >= entries) d = n;
    uint32_t rank = 0;
    const unsigned long long below = (1ull << lane) - 1ull;
    for (uint32_t dd = 0; dd < n; ++dd) {
        const unsigned long long m = __ballot(d == dd);
        if (d == dd) rank = __popcll(m & below);
        if (lane == 0) s_cnt[wave][dd] = __popcll(m);
    }
    __syncthreads();
    if (wave == 0) {
        const uint32_t t = lane < n ? s_total[lane] : 0;
        const uint32_t incl = wave_scan_u32(t);
        s_start[lane] = incl - t;
        if (c == 0) {
            const uint32_t from = lane < n ? s_from[lane] : 0;
            const uint32_t upto = wave_scan_u32(from);
            if (lane < n) {
                send_counts[i * n + lane] = static_cast<uint64_t>(t) * row_elems;
                sdispls[i * n + lane] = static_cast<uint64_t>(incl - t) * row_elems;
                recv_counts[i * n + lane] = static_cast<uint64_t>(from) * row_elems;
                rdispls[i * n + lane] = static_cast<uint64_t>(upto - from) * row_elems;
            }
        }
    }
    __syncthreads();
    if (e < entries) {
        uint32_t out = kDropped;
        if (d < n) {
            out = s_start[d] + s_before[d] + rank;
            for (uint32_t w = 0; w < wave; ++w) out += s_cnt[w][d];
        }
        static_cast<uint32_t *>(perm.p[i])[e] = out;
    }
}

// Row gather / scatter: 512 vectors of 16 bytes per workgroup, rows of vpr vectors.
//   PACK:    packed[perm[e]] = tokens[e / topk]      (g runs over entries x vpr)
//   UNPACK:  out[t] = packed[perm[t]]                (topk == 1; g runs over tokens x vpr)
template <bool PACK>
__global__ void __launch_bounds__(256)
k_moe_rows(MoeConstPtrs src, MoeConstPtrs perm, MoePtrs dst, uint32_t rows, uint32_t topk, uint32_t vpr)
{
    const uint32_t i = blockIdx.y;
    const uint64_t total = static_cast<uint64_t>(rows) * vpr;
    const uint32_t *pm = static_cast<const uint32_t *>(perm.p[i]);
    const char *s = static_cast<const char *>(src.p[i]);
    char *o = static_cast<char *>(dst.p[i]);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const uint64_t g = static_cast<uint64_t>(blockIdx.x) * 512 + u * 256 + threadIdx.x;
        if (g >= total) continue;
        const uint32_t e = static_cast<uint32_t>(g / vpr);
        const uint32_t v = static_cast<uint32_t>(g - static_cast<uint64_t>(e) * vpr);
        const uint32_t p = pm[e];
        if (PACK) {
            if (p == kDropped) continue;
            st16(o + (static_cast<uint64_t>(p) * vpr + v) * 16, ld16(s + (static_cast<uint64_t>(e / topk) * vpr + v) * 16));
        } else {
            u32x4 x = {0, 0, 0, 0};
            if (p != kDropped) x = ld16(s + (static_cast<uint64_t>(p) * vpr + v) * 16);
            st16(o + (static_cast<uint64_t>(e) * vpr + v) * 16, x);
        }
    }
}

// out[t] = sum over j of packed[perm[t * topk + j]], j ascending, starting from the first entry that was
// not dropped; accumulated in the compute type (fp32 for 16-bit floats), narrowed once.
template <int DT>
__global__ void __launch_bounds__(256)
k_moe_combine(MoeConstPtrs packed, MoeConstPtrs perm, MoePtrs out, uint32_t tokens, uint32_t topk, uint32_t vpr)
{
    using V = Vec16<DT>;
    using C = typename V::C;
    constexpr int NE = V::NE;
    const uint32_t i = blockIdx.y;
    const uint64_t total = static_cast<uint64_t>(tokens) * vpr;
    const uint32_t *pm = static_cast<const uint32_t *>(perm.p[i]);
    const char *s = static_cast<const char *>(packed.p[i]);
    char *o = static_cast<char *>(out.p[i]);
    const uint64_t g = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (g >= total) return;
    const uint32_t t = static_cast<uint32_t>(g / vpr);
    const uint32_t v = static_cast<uint32_t>(g - static_cast<uint64_t>(t) * vpr);
    C acc[NE];
    bool have = false;
#pragma unroll
    for (int e = 0; e < NE; ++e) acc[e] = C(0);
    for (uint32_t j = 0; j < topk; ++j) {
        const uint32_t p = pm[static_cast<uint64_t>(t) * topk + j];
        if (p == kDropped) continue;
        C x[NE];
        V::unpack(ld16(s + (static_cast<uint64_t>(p) * vpr + v) * 16), x);
        if (!have) {
#pragma unroll
            for (int e = 0; e < NE; ++e) acc[e] = x[e];
            have = true;
        } else {
#pragma unroll
            for (int e = 0; e < NE; ++e) acc[e] = V::template combine<HCCL_REDUCE_SUM>(x[e], acc[e]);
        }
    }
    st16(o + (static_cast<uint64_t>(t) * vpr + v) * 16, V::pack(acc));
}

// Where rank i's rows for destination j land: packed row p of rank i sits at landing(...) + p rows, i.e. at the
// first row of the block from i in recv[j] minus the first row of the group for j in i's packed order.  The
// tables are a few hundred bytes and stay in the caches.
__device__ __forceinline__ char *landing(const MoePtrs &recv, uint32_t i, uint32_t j, uint32_t n, uint32_t esz,
                                         const uint64_t *sdispls, const uint64_t *rdispls)
{
    const int64_t elems = static_cast<int64_t>(rdispls[j * n + i]) - static_cast<int64_t>(sdispls[i * n + j]);
    return static_cast<char *>(recv.p[j]) + elems * static_cast<int64_t>(esz);
}

// Dispatch in one pass (what the pack kernel followed by the AlltoAllV kernel does in two):
// recv[dest[e]] row (landing + perm[e]) = tokens[e / topk].
__global__ void __launch_bounds__(256)
k_moe_dispatch(MoeConstPtrs tokens, MoeConstPtrs dest, MoeConstPtrs perm, MoePtrs recv, uint32_t n, uint32_t entries,
               uint32_t topk, uint32_t vpr, uint32_t esz, const uint64_t *sdispls, const uint64_t *rdispls)
{
    const uint32_t i = blockIdx.y;
    const uint64_t total = static_cast<uint64_t>(entries) * vpr;
    const uint32_t *pm = static_cast<const uint32_t *>(perm.p[i]);
    const int32_t *dt = static_cast<const int32_t *>(dest.p[i]);
    const char *s = static_cast<const char *>(tokens.p[i]);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const uint64_t g = static_cast<uint64_t>(blockIdx.x) * 512 + u * 256 + threadIdx.x;
        if (g >= total) continue;
        const uint32_t e = static_cast<uint32_t>(g / vpr);
        const uint32_t v = static_cast<uint32_t>(g - static_cast<uint64_t>(e) * vpr);
        const uint32_t p = pm[e];
        const uint32_t j = static_cast<uint32_t>(dt[e]);
        if (p == kDropped || j >= n) continue;   // perm marks entries with a destination outside 0 .. n-1 as dropped
        char *o = landing(recv, i, j, n, esz, sdispls, rdispls);
        st16(o + (static_cast<uint64_t>(p) * vpr + v) * 16, ld16(s + (static_cast<uint64_t>(e / topk) * vpr + v) * 16));
    }
}

// The way back in one pass (what the AlltoAllV kernel followed by the combine kernel does in two):
// out[t] = sum over j < topk of the row of entry t * topk + j where dispatch put it, in the buffers `expert`.
// DT = int8 moves bytes (topk == 1: nothing is added).
template <int DT>
__global__ void __launch_bounds__(256)
k_moe_gather_combine(MoeConstPtrs expert, MoeConstPtrs dest, MoeConstPtrs perm, MoePtrs out, uint32_t n, uint32_t tokens,
                     uint32_t topk, uint32_t vpr, uint32_t esz, const uint64_t *sdispls, const uint64_t *rdispls)
{
    using V = Vec16<DT>;
    using C = typename V::C;
    constexpr int NE = V::NE;
    const uint32_t i = blockIdx.y;
    const uint64_t total = static_cast<uint64_t>(tokens) * vpr;
    const uint32_t *pm = static_cast<const uint32_t *>(perm.p[i]);
    const int32_t *dt = static_cast<const int32_t *>(dest.p[i]);
    char *o = static_cast<char *>(out.p[i]);
    const uint64_t g = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (g >= total) return;
    const uint32_t t = static_cast<uint32_t>(g / vpr);
    const uint32_t v = static_cast<uint32_t>(g - static_cast<uint64_t>(t) * vpr);
    C acc[NE];
    bool have = false;
#pragma unroll
    for (int e = 0; e < NE; ++e) acc[e] = C(0);
    for (uint32_t j = 0; j < topk; ++j) {
        const uint64_t e = static_cast<uint64_t>(t) * topk + j;
        const uint32_t p = pm[e];
        const uint32_t d = static_cast<uint32_t>(dt[e]);
        if (p == kDropped || d >= n) continue;
        const char *from = landing(as_mutable_dev(expert), i, d, n, esz, sdispls, rdispls);
        C x[NE];
        V::unpack(ld16(from + (static_cast<uint64_t>(p) * vpr + v) * 16), x);
        if (!have) {
#pragma unroll
            for (int k = 0; k < NE; ++k) acc[k] = x[k];
            have = true;
        } else {
#pragma unroll
            for (int k = 0; k < NE; ++k) acc[k] = V::template combine<HCCL_REDUCE_SUM>(x[k], acc[k]);
        }
    }
    st16(o + (static_cast<uint64_t>(t) * vpr + v) * 16, V::pack(acc));
}

// ---- rows of at least kLongRow vectors ----------------------------------------------------------------------
// A wavefront moves one piece (64 vectors, 1 KiB) of ONE row, so the entry, its destination and where it lands are the
// same for every lane: they are fetched with scalar loads, and no lane divides or looks anything up.  Pieces and not
// runs of a workgroup's width: a row of 7168 bf16 is 14 whole pieces, but 3.5 runs of 256 vectors.
// From 48 vectors on: 8 x 2000 tokens, top-2, routing and both directions with rows of 48 vectors 24.1 us against 32.6 for
// the kernels above, with 32 (half of every wavefront idle) 23.7 against 24.9 and 8 x 2000 with 17 24.7 against 20.7.
constexpr uint32_t kLongRow = 48;
constexpr uint32_t kPieceVecs = 64;
constexpr uint32_t kPiecesPerBlock = 4;
constexpr uint32_t kXcds = 8;

struct RowPieces {
    uint32_t per_row;   // pieces of a row
    uint32_t total;     // pieces of all rows of a rank
    uint32_t groups;    // dispatch: wavefronts that share a token's piece, S entries of it each
};
// A launch has at most 2^32 work-items along x: more rows than that take several launches, each with its pointers moved on.
constexpr uint64_t kMostBlocks = 0xffff00;
// Rows of one launch at most; 0: not even one row fits.
inline uint32_t rows_per_launch(uint32_t vpr, uint32_t groups)
{
    const uint64_t per_row = (static_cast<uint64_t>(vpr) + kPieceVecs - 1) / kPieceVecs;
    const uint64_t rows = kMostBlocks / kXcds / groups * kXcds * kPiecesPerBlock / per_row;
    return rows > 0xffffffffull ? 0xffffffffu : static_cast<uint32_t>(rows);
}
inline RowPieces row_pieces(uint32_t rows, uint32_t vpr, uint32_t groups)
{
    const uint32_t per_row = static_cast<uint32_t>((static_cast<uint64_t>(vpr) + kPieceVecs - 1) / kPieceVecs);
    return {per_row, rows * per_row, groups};
}
// The same arrays from `bytes` on.
inline MoeConstPtrs moved_on(MoeConstPtrs a, uint32_t n, uint64_t bytes)
{
    for (uint32_t i = 0; i < n; ++i) a.p[i] = static_cast<const char *>(a.p[i]) + bytes;
    return a;
}

// Dispatch: a piece of a token goes to S of its entries' rows, loaded once; what is left of topk / S goes to other
// workgroups, eight apart, so that they run on the same XCD and find the piece in its L2 (kCached).  Bound: HBM.  8 x 4096
// tokens, top-2, 7168 bf16 (1409 MB): 219 us where two vectors of two entries per thread, each read by itself, took 293;
// 8 x 64 tokens, top-8: 11.5 against 22.5.
template <int S, uint32_t kPolicy, bool kCached>
__global__ void __launch_bounds__(kPieceVecs * kPiecesPerBlock)
k_moe_scatter_pieces(MoeConstPtrs tokens, MoeConstPtrs dest, MoeConstPtrs perm, MoePtrs recv, uint32_t n, uint32_t topk, uint32_t vpr,
                     RowPieces pieces, uint32_t esz, const uint64_t *sdispls, const uint64_t *rdispls)
{
    const uint32_t i = blockIdx.y;
    const uint32_t span = kXcds * pieces.groups;
    const uint32_t hi = blockIdx.x / span;
    const uint32_t in_span = blockIdx.x - hi * span;
    const uint32_t block = hi * kXcds + in_span % kXcds;
    const uint32_t piece = __builtin_amdgcn_readfirstlane(block * kPiecesPerBlock + threadIdx.x / kPieceVecs);
    if (piece >= pieces.total) return;
    const uint32_t t = piece / pieces.per_row;
    const uint32_t v0 = (piece - t * pieces.per_row) * kPieceVecs;
    const uint32_t lane = threadIdx.x % kPieceVecs;
    const uint32_t lane_off = lane * 16;
    const bool inside = lane < vpr - v0;
    const char *from = static_cast<const char *>(tokens.p[i]) + (static_cast<uint64_t>(t) * vpr + v0) * 16;
    u32x4 x = {0, 0, 0, 0};
    if (inside) x = kCached ? ld16_cached(from + lane_off) : ld16(from + lane_off);
    const uint32_t *pm = static_cast<const uint32_t *>(perm.p[i]) + static_cast<uint64_t>(t) * topk;
    const int32_t *dt = static_cast<const int32_t *>(dest.p[i]) + static_cast<uint64_t>(t) * topk;
    const uint32_t first = in_span / kXcds * S;
    uint32_t p[S];
    uint32_t j[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const uint32_t e = first + s;
        const uint32_t at = e < topk ? e : topk - 1;   // an entry behind the token's last repeats it and stores nothing
        p[s] = pm[at];
        j[s] = static_cast<uint32_t>(dt[at]);
        if (e >= topk) p[s] = kDropped;
    }
    char *to[S];
    bool ok[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        ok[s] = p[s] != kDropped && j[s] < n;
        to[s] = landing(recv, i, ok[s] ? j[s] : 0u, n, esz, sdispls, rdispls) + (static_cast<uint64_t>(ok[s] ? p[s] : 0u) * vpr + v0) * 16;
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if (ok[s] && inside) st16x(to[s] + lane_off, x, kPolicy);
    }
}

// Gather the rows of a token's entries from where dispatch put them in expert[dest[.]] and add them, K entries at a time: their
// look-ups are in flight together, and their rows too where all K are there.  (A branch per entry makes the compiler wait for
// every load before the next.)  Where one is dropped or behind the last, those that are left are read one after the other, so
// that what is dropped costs no bytes.  K by gather_entries.  DT = int8 moves bytes (topk == 1).
// ALL: tokens have K entries (top-2).  There is one round, and no branch between the look-ups and the rows: in the place of a
// dropped entry the lanes load the row of one that is there, which the caches then hold.  Exchange of 8 x 4096 x 7168 bf16, the
// other form : this, us: 451.8 : 449.8, 16 x 695 152.6 : 152.1; gather with half of the entries dropped 151.5 : 148.6, all 113.7 : 85.3.
// Of more entries the other form is the faster one (8 x 96 top-8 41.7 : 41.2, 8 x 16 15.8 : 15.2, 8 x 64 top-3 19.8 : 18.9).
template <int DT, int K, bool ALL>
__global__ void __launch_bounds__(kPieceVecs * kPiecesPerBlock)
k_moe_gather_pieces(MoeConstPtrs rows, MoeConstPtrs dest, MoeConstPtrs perm, MoePtrs out, uint32_t n, uint32_t any_topk, uint32_t vpr,
                    RowPieces pieces, uint32_t esz, const uint64_t *sdispls, const uint64_t *rdispls)
{
    const uint32_t topk = ALL ? K : any_topk;
    using V = Vec16<DT>;
    using C = typename V::C;
    constexpr int NE = V::NE;
    const uint32_t i = blockIdx.y;
    const uint32_t piece = __builtin_amdgcn_readfirstlane(blockIdx.x * kPiecesPerBlock + threadIdx.x / kPieceVecs);
    if (piece >= pieces.total) return;
    const uint32_t t = piece / pieces.per_row;
    const uint32_t v0 = (piece - t * pieces.per_row) * kPieceVecs;
    const uint32_t lane = threadIdx.x % kPieceVecs;
    const uint32_t lane_off = lane * 16;
    if (lane >= vpr - v0) return;
    const uint32_t *pm = static_cast<const uint32_t *>(perm.p[i]) + static_cast<uint64_t>(t) * topk;
    const int32_t *dt = static_cast<const int32_t *>(dest.p[i]) + static_cast<uint64_t>(t) * topk;
    C acc[NE];
    bool have = false;
#pragma unroll
    for (int k = 0; k < NE; ++k) acc[k] = C(0);
    char *to = static_cast<char *>(out.p[i]) + (static_cast<uint64_t>(t) * vpr + v0) * 16 + lane_off;
    auto row = [&](uint32_t d, uint32_t p) {
        return ld16(landing(as_mutable_dev(rows), i, d, n, esz, sdispls, rdispls) + (static_cast<uint64_t>(p) * vpr + v0) * 16 + lane_off);
    };
    auto add = [&](u32x4 raw) {
        C x[NE];
        V::unpack(raw, x);
        if (!have) {
#pragma unroll
            for (int q = 0; q < NE; ++q) acc[q] = x[q];
        } else {
#pragma unroll
            for (int q = 0; q < NE; ++q) acc[q] = V::template combine<HCCL_REDUCE_SUM>(x[q], acc[q]);
        }
        have = true;
    };
    for (uint32_t first = 0; first < topk; first += K) {
        uint32_t p[K];
        uint32_t d[K];
        bool ok[K];
        bool all = true;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint32_t e = first + k < topk ? first + k : topk - 1;   // an entry behind the last repeats it and is not added
            p[k] = pm[e];
            d[k] = static_cast<uint32_t>(dt[e]);
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {
            ok[k] = (first + k < topk) & (p[k] != kDropped) & (d[k] < n);   // without branches between the look-ups
            all = all & ok[k];
        }
        if constexpr (ALL) {
            uint32_t there_p = kDropped;
            uint32_t there_d = 0;
#pragma unroll
            for (int k = K - 1; k >= 0; --k) {
                there_p = ok[k] ? p[k] : there_p;
                there_d = ok[k] ? d[k] : there_d;
            }
            if (there_p == kDropped) continue;   // no entry is there
            u32x4 raw[K];
#pragma unroll
            for (int k = 0; k < K; ++k) raw[k] = row(ok[k] ? d[k] : there_d, ok[k] ? p[k] : there_p);
#pragma unroll
            for (int k = 0; k < K; ++k) {
                if (ok[k]) add(raw[k]);
            }
        } else if (K > 1 && all) {
            u32x4 raw[K];
#pragma unroll
            for (int k = 0; k < K; ++k) raw[k] = row(d[k], p[k]);
#pragma unroll
            for (int k = 0; k < K; ++k) add(raw[k]);
        } else {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                if (ok[k]) add(row(d[k], p[k]));
            }
        }
    }
    st16(to, V::pack(acc));
}

// Entries of a token that the gather takes at a time.  Two of two (exchange of the rows, one : two entries, us: 8 x 4096 tokens of
// 7168 bf16 458.4 : 449.8, 8 x 1024 115.4 : 115.2, 4 x 300 25.9 : 25.2).  Of more, four of four and more while the launch is so
// small that it is bound by its round trips (top-8, one : two : four: 8 x 16 18.2 : 16.1 : 15.1, 8 x 40 23.8 : 22.3 : 22.5; top-4, 8 x
// 32 16.5 : 15.2 : 15.0), then two (top-8, 8 x 64 29.5 : 29.2 : 29.4, 8 x 96 42.9 : 41.0 : 41.1, 8 x 128 51.0 : 50.7 : 50.9, 4 x 1000 x 2880
// 77.3 : 76.7 : 76.6; top-4, 16 x 128 x 4096 37.8 : 37.0 : 36.8), and one where the rows come near to what the Infinity Cache holds:
// more of them open more rows at once than HBM likes (top-8, 8 x 256 91.0 : 91.3 : 91.8, 8 x 400 134.6 : 136.5 : 137.3, 8 x 4096 x 4096 807 : 825 :
// 830; top-4, 2 x 2000 97.8 : 99.1 : 99.7, 4 x 3683 x 4096 212.5 : 217.4 : 217.7).
inline int gather_entries(const DeviceCtx *ctx, uint32_t topk, uint64_t waves, uint64_t row_bytes)
{
    constexpr uint64_t kTwoUpto = 192ull << 20;
    if (topk <= 2) return static_cast<int>(topk);
    const uint64_t cus = ctx ? static_cast<uint64_t>(ctx->num_cus) : 256;
    if (topk >= 4 && waves <= 16 * cus) return 4;
    return row_bytes < kTwoUpto ? 2 : 1;
}

// Which entries share a wavefront, and how rows are stored.  Tokens of up to kWarmTokens in all are usually still in the
// Infinity Cache, just written by the layer in front, and stay there when the stores stream past it: with four entries
// and more, two per wavefront (8 x 1024 tokens, top-8, 4096 bf16: 84 us; 131 with the caches flushed).  Everything else
// reads each piece past the caches, once for up to four entries, and writes through the L2 (the same case: 104 and 106;
// top-2 of 8 x 4096 x 7168: 222 against 235 to 240; 8 x 4096 x 4096, top-8: 403 against 481).
constexpr uint64_t kWarmTokens = 128ull << 20;

int launch_scatter_pieces(uint32_t per_wave, hipStream_t st, const MoeConstPtrs &tokens, const MoeConstPtrs &dest,
                          const MoeConstPtrs &perm, const MoePtrs &recv, uint32_t n, uint32_t rows, uint32_t topk, uint32_t vpr,
                          uint32_t esz, const uint64_t *sdispls, const uint64_t *rdispls)
{
    const bool warm = per_wave == 0 && topk >= 4 && static_cast<uint64_t>(rows) * n <= kWarmTokens / 16 / vpr;
    const uint32_t s = per_wave != 0 ? per_wave : warm ? 2u : topk >= 3 ? 4u : topk;
    const uint32_t groups = (topk + s - 1) / s;
    const uint32_t most = rows_per_launch(vpr, groups);
    if (most == 0) return fail(HCCL_E_PARA, "too much data for one launch");
    const dim3 block(kPieceVecs * kPiecesPerBlock);
    for (uint32_t at = 0; at < rows;) {
        const uint32_t take = rows - at < most ? rows - at : most;
        const RowPieces pieces = row_pieces(take, vpr, groups);
        const MoeConstPtrs tk = moved_on(tokens, n, static_cast<uint64_t>(at) * vpr * 16);
        const MoeConstPtrs ds = moved_on(dest, n, static_cast<uint64_t>(at) * topk * 4);
        const MoeConstPtrs pm = moved_on(perm, n, static_cast<uint64_t>(at) * topk * 4);
        const dim3 grid((pieces.total + kPiecesPerBlock * kXcds - 1) / (kPiecesPerBlock * kXcds) * kXcds * groups, n);
        if (warm) {
            HCCLX_LAUNCH((k_moe_scatter_pieces<2, kStoreStream, true>), grid, block, 0, st, tk, ds, pm, recv, n, topk, vpr, pieces, esz,
                         sdispls, rdispls);
        } else if (s == 1) {
            HCCLX_LAUNCH((k_moe_scatter_pieces<1, kStoreThrough, false>), grid, block, 0, st, tk, ds, pm, recv, n, topk, vpr, pieces,
                         esz, sdispls, rdispls);
        } else if (s == 2) {
            HCCLX_LAUNCH((k_moe_scatter_pieces<2, kStoreThrough, false>), grid, block, 0, st, tk, ds, pm, recv, n, topk, vpr, pieces,
                         esz, sdispls, rdispls);
        } else {
            HCCLX_LAUNCH((k_moe_scatter_pieces<4, kStoreThrough, false>), grid, block, 0, st, tk, ds, pm, recv, n, topk, vpr, pieces,
                         esz, sdispls, rdispls);
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return fail_hip(e, "moe dispatch kernel");
        at += take;
    }
    return HCCL_SUCCESS;
}

template <int DT>
void launch_gather_k(int k, dim3 grid, dim3 block, hipStream_t st, const MoeConstPtrs &rows, const MoeConstPtrs &dest, const MoeConstPtrs &perm,
                     const MoePtrs &out, uint32_t n, uint32_t topk, uint32_t vpr, const RowPieces &pieces, uint32_t esz,
                     const uint64_t *sdispls, const uint64_t *rdispls)
{
    if (k == 4) {
        HCCLX_LAUNCH((k_moe_gather_pieces<DT, 4, false>), grid, block, 0, st, rows, dest, perm, out, n, topk, vpr, pieces, esz, sdispls, rdispls);
    } else if (k == 2 && topk == 2) {
        HCCLX_LAUNCH((k_moe_gather_pieces<DT, 2, true>), grid, block, 0, st, rows, dest, perm, out, n, topk, vpr, pieces, esz, sdispls, rdispls);
    } else if (k == 2) {
        HCCLX_LAUNCH((k_moe_gather_pieces<DT, 2, false>), grid, block, 0, st, rows, dest, perm, out, n, topk, vpr, pieces, esz, sdispls, rdispls);
    } else {
        HCCLX_LAUNCH((k_moe_gather_pieces<DT, 1, false>), grid, block, 0, st, rows, dest, perm, out, n, topk, vpr, pieces, esz, sdispls, rdispls);
    }
}

int launch_gather_pieces(int kind, hipStream_t st, const MoeConstPtrs &rows, const MoeConstPtrs &dest, const MoeConstPtrs &perm,
                         const MoeConstPtrs &out, uint32_t n, uint32_t tokens, uint32_t topk, uint32_t vpr, uint32_t esz,
                         const uint64_t *sdispls, const uint64_t *rdispls)
{
    const uint32_t most = rows_per_launch(vpr, 1);
    if (most == 0) return fail(HCCL_E_PARA, "too much data for one launch");
    const dim3 block(kPieceVecs * kPiecesPerBlock);
    const uint64_t row_bytes = static_cast<uint64_t>(n) * tokens * topk * vpr * 16;
    for (uint32_t at = 0; at < tokens;) {
        const uint32_t take = tokens - at < most ? tokens - at : most;
        const RowPieces pieces = row_pieces(take, vpr, 1);
        const MoePtrs to = as_mutable(moved_on(out, n, static_cast<uint64_t>(at) * vpr * 16));
        const MoeConstPtrs ds = moved_on(dest, n, static_cast<uint64_t>(at) * topk * 4);
        const MoeConstPtrs pm = moved_on(perm, n, static_cast<uint64_t>(at) * topk * 4);
        const dim3 grid((pieces.total + kPiecesPerBlock - 1) / kPiecesPerBlock, n);
        const int k = gather_entries(device_ctx(), topk, static_cast<uint64_t>(pieces.total) * n, row_bytes);
        if (kind == HCCL_DATA_TYPE_FP32) {
            launch_gather_k<HCCL_DATA_TYPE_FP32>(k, grid, block, st, rows, ds, pm, to, n, topk, vpr, pieces, esz, sdispls, rdispls);
        } else if (kind == HCCL_DATA_TYPE_FP16) {
            launch_gather_k<HCCL_DATA_TYPE_FP16>(k, grid, block, st, rows, ds, pm, to, n, topk, vpr, pieces, esz, sdispls, rdispls);
        } else if (kind == HCCL_DATA_TYPE_BFP16) {
            launch_gather_k<HCCL_DATA_TYPE_BFP16>(k, grid, block, st, rows, ds, pm, to, n, topk, vpr, pieces, esz, sdispls, rdispls);
        } else {
            HCCLX_LAUNCH((k_moe_gather_pieces<HCCL_DATA_TYPE_INT8, 1, false>), grid, block, 0, st, rows, ds, pm, to, n, topk, vpr, pieces, esz,
                         sdispls, rdispls);
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return fail_hip(e, "moe gather-combine kernel");
        at += take;
    }
    return HCCL_SUCCESS;
}

int check_ranks(uint32_t n)
{
    if (n == 0 || n > kMoeMaxRanks) return fail(HCCL_E_PARA, "rank count outside 1.." + std::to_string(kMoeMaxRanks));
    return HCCL_SUCCESS;
}

int fill(const void *const *in, uint32_t n, MoeConstPtrs *out, const char *what, bool align16)
{
    if (in == nullptr) return fail(HCCL_E_PTR, std::string(what) + " pointer array is null");
    std::memset(out, 0, sizeof(*out));
    for (uint32_t i = 0; i < n; ++i) {
        if (in[i] == nullptr) return fail(HCCL_E_PTR, std::string(what) + "[" + std::to_string(i) + "] is null");
        if (align16 && (reinterpret_cast<uint64_t>(in[i]) & 15) != 0) {
            return fail(HCCL_E_PARA, std::string(what) + "[" + std::to_string(i) + "] is not 16-byte aligned");
        }
        out->p[i] = in[i];
    }
    return HCCL_SUCCESS;
}

}  // namespace

extern "C" {

uint64_t hcclx_moe_workspace_bytes(uint32_t n, uint32_t entries)
{
    return (static_cast<uint64_t>(n) * n * chunks_of(entries) + static_cast<uint64_t>(n) * n) * sizeof(uint32_t);
}

int hcclx_moe_route(const int32_t *const *dest, uint32_t n, uint32_t entries, uint64_t row_elems, uint64_t *send_counts,
                    uint64_t *sdispls, uint64_t *recv_counts, uint64_t *rdispls, uint32_t *const *perm, void *workspace,
                    void *stream)
{
    if (!device_ctx()) return HCCL_E_RUNTIME;
    int rc = check_ranks(n);
    if (rc != HCCL_SUCCESS) return rc;
    if (!send_counts || !sdispls || !recv_counts || !rdispls || !workspace) return fail(HCCL_E_PTR, "output table or workspace is null");
    if (entries == 0) return fail(HCCL_E_PARA, "no entries to route");
    if (static_cast<uint64_t>(entries) >= kDropped) return fail(HCCL_E_PARA, "too many entries");
    MoeConstPtrs d, p;
    rc = fill(reinterpret_cast<const void *const *>(dest), n, &d, "dest", false);
    if (rc != HCCL_SUCCESS) return rc;
    rc = fill(reinterpret_cast<const void *const *>(perm), n, &p, "perm", false);
    if (rc != HCCL_SUCCESS) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const uint32_t chunks = chunks_of(entries);
    uint32_t *base = static_cast<uint32_t *>(workspace);
    uint32_t *row_start = base + static_cast<uint64_t>(n) * n * chunks;
    // perm may lie on top of the destinations: then every entry is read a launch before, and by the thread that writes it
    bool in_place = false;
    for (uint32_t i = 0; i < n; ++i) in_place = in_place || d.p[i] == p.p[i];
    if (entries <= kOneLaunchEntries && !in_place) {
        HCCLX_LAUNCH(k_moe_route_one, dim3(chunks, n), dim3(kMoeChunk), 0, st, d, as_mutable(p), n, entries, row_elems, send_counts,
                     sdispls, recv_counts, rdispls);
        const hipError_t oe = hipGetLastError();
        if (oe != hipSuccess) return fail_hip(oe, "moe routing kernel");
        return HCCL_SUCCESS;
    }
    HCCLX_LAUNCH(k_moe_hist, dim3(chunks, n), dim3(kMoeChunk), 0, st, d, n, entries, chunks, base);
    if (chunks <= kFusedChunks && static_cast<uint64_t>(n) * n * chunks <= kFusedCells) {
        HCCLX_LAUNCH(k_moe_scan_perm, dim3(chunks, n), dim3(kMoeChunk), 0, st, d, as_mutable(p), n, entries, chunks,
                           row_elems, base, send_counts, sdispls, recv_counts, rdispls);
        hipError_t fe = hipGetLastError();
        if (fe != hipSuccess) return fail_hip(fe, "moe routing kernels");
        return HCCL_SUCCESS;
    }
    HCCLX_LAUNCH(k_moe_scan, dim3(n), dim3(256), 0, st, n, chunks, row_elems, base, row_start, send_counts, sdispls,
                       recv_counts);
    HCCLX_LAUNCH(k_moe_perm, dim3(chunks, n), dim3(kMoeChunk), 0, st, d, as_mutable(p), n, entries, chunks, base,
                       row_start, send_counts, rdispls);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail_hip(e, "moe routing kernels");
    return HCCL_SUCCESS;
}

int hcclx_moe_pack(const void *const *tokens, const uint32_t *const *perm, uint32_t n, uint32_t entries, uint32_t topk,
                   uint64_t row_bytes, void *const *packed, void *stream)
{
    if (!device_ctx()) return HCCL_E_RUNTIME;
    int rc = check_ranks(n);
    if (rc != HCCL_SUCCESS) return rc;
    if (topk == 0 || entries == 0 || entries % topk != 0) return fail(HCCL_E_PARA, "entries must be a positive multiple of topk");
    if (row_bytes == 0 || row_bytes % 16 != 0) return fail(HCCL_E_PARA, "row size must be a positive multiple of 16 bytes");
    if (row_bytes / 16 > 0xffffffffull) return fail(HCCL_E_PARA, "row too long");
    MoeConstPtrs s, p, o;
    rc = fill(tokens, n, &s, "tokens", true);
    if (rc != HCCL_SUCCESS) return rc;
    rc = fill(reinterpret_cast<const void *const *>(perm), n, &p, "perm", false);
    if (rc != HCCL_SUCCESS) return rc;
    rc = fill(packed, n, &o, "packed", true);
    if (rc != HCCL_SUCCESS) return rc;
    const uint32_t vpr = static_cast<uint32_t>(row_bytes / 16);
    const uint64_t blocks = (static_cast<uint64_t>(entries) * vpr + 511) / 512;
    if (blocks > 0x7fffffffull) return fail(HCCL_E_PARA, "too much data for one launch");
    HCCLX_LAUNCH(k_moe_rows<true>, dim3(static_cast<uint32_t>(blocks), n), dim3(256), 0, static_cast<hipStream_t>(stream),
                       s, p, as_mutable(o), entries, topk, vpr);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail_hip(e, "moe pack kernel");
    return HCCL_SUCCESS;
}

int hcclx_moe_combine(const void *const *packed, const uint32_t *const *perm, uint32_t n, uint32_t tokens, uint32_t topk,
                      uint64_t row_elems, int dtype, void *const *out, void *stream)
{
    if (!device_ctx()) return HCCL_E_RUNTIME;
    int rc = check_ranks(n);
    if (rc != HCCL_SUCCESS) return rc;
    const int esz = dtype_size(dtype);
    if (esz == 0) return fail(HCCL_E_NOT_SUPPORT, "unknown data type " + std::to_string(dtype));
    if (topk == 0 || tokens == 0) return fail(HCCL_E_PARA, "tokens and topk must be positive");
    const uint64_t row_bytes = row_elems * esz;
    if (row_bytes == 0 || row_bytes % 16 != 0) return fail(HCCL_E_PARA, "row size must be a positive multiple of 16 bytes");
    if (row_bytes / 16 > 0xffffffffull) return fail(HCCL_E_PARA, "row too long");
    if (topk > 1 && dtype != HCCL_DATA_TYPE_FP32 && dtype != HCCL_DATA_TYPE_FP16 && dtype != HCCL_DATA_TYPE_BFP16) {
        return fail(HCCL_E_NOT_SUPPORT, "combining several rows needs fp32, fp16 or bf16");
    }
    MoeConstPtrs s, p, o;
    rc = fill(packed, n, &s, "packed", true);
    if (rc != HCCL_SUCCESS) return rc;
    rc = fill(reinterpret_cast<const void *const *>(perm), n, &p, "perm", false);
    if (rc != HCCL_SUCCESS) return rc;
    rc = fill(out, n, &o, "out", true);
    if (rc != HCCL_SUCCESS) return rc;
    const uint32_t vpr = static_cast<uint32_t>(row_bytes / 16);
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (topk == 1) {
        const uint64_t blocks = (static_cast<uint64_t>(tokens) * vpr + 511) / 512;
        if (blocks > 0x7fffffffull) return fail(HCCL_E_PARA, "too much data for one launch");
        HCCLX_LAUNCH(k_moe_rows<false>, dim3(static_cast<uint32_t>(blocks), n), dim3(256), 0, st, s, p, as_mutable(o),
                           tokens, 1u, vpr);
    } else {
        const uint64_t blocks = (static_cast<uint64_t>(tokens) * vpr + 255) / 256;
        if (blocks > 0x7fffffffull) return fail(HCCL_E_PARA, "too much data for one launch");
        const dim3 grid(static_cast<uint32_t>(blocks), n);
        if (dtype == HCCL_DATA_TYPE_FP32) {
            HCCLX_LAUNCH(k_moe_combine<HCCL_DATA_TYPE_FP32>, grid, dim3(256), 0, st, s, p, as_mutable(o), tokens, topk, vpr);
        } else if (dtype == HCCL_DATA_TYPE_FP16) {
            HCCLX_LAUNCH(k_moe_combine<HCCL_DATA_TYPE_FP16>, grid, dim3(256), 0, st, s, p, as_mutable(o), tokens, topk, vpr);
        } else {
            HCCLX_LAUNCH(k_moe_combine<HCCL_DATA_TYPE_BFP16>, grid, dim3(256), 0, st, s, p, as_mutable(o), tokens, topk, vpr);
        }
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail_hip(e, "moe combine kernel");
    return HCCL_SUCCESS;
}

int hcclx_moe_dispatch(const void *const *tokens, const int32_t *const *dest, const uint32_t *const *perm, uint32_t n,
                       uint32_t entries, uint32_t topk, uint64_t row_elems, int dtype, const uint64_t *sdispls,
                       const uint64_t *rdispls, void *const *recv, void *stream)
{
    if (!device_ctx()) return HCCL_E_RUNTIME;
    int rc = check_ranks(n);
    if (rc != HCCL_SUCCESS) return rc;
    const int esz = dtype_size(dtype);
    if (esz == 0) return fail(HCCL_E_NOT_SUPPORT, "unknown data type " + std::to_string(dtype));
    if (topk == 0 || entries == 0 || entries % topk != 0) return fail(HCCL_E_PARA, "entries must be a positive multiple of topk");
    const uint64_t row_bytes = row_elems * esz;
    if (row_bytes == 0 || row_bytes % 16 != 0) return fail(HCCL_E_PARA, "row size must be a positive multiple of 16 bytes");
    if (row_bytes / 16 > 0xffffffffull) return fail(HCCL_E_PARA, "row too long");
    if (!sdispls || !rdispls) return fail(HCCL_E_PTR, "displacement table is null");
    MoeConstPtrs s, d, p, o;
    rc = fill(tokens, n, &s, "tokens", true);
    if (rc != HCCL_SUCCESS) return rc;
    rc = fill(reinterpret_cast<const void *const *>(dest), n, &d, "dest", false);
    if (rc != HCCL_SUCCESS) return rc;
    rc = fill(reinterpret_cast<const void *const *>(perm), n, &p, "perm", false);
    if (rc != HCCL_SUCCESS) return rc;
    rc = fill(recv, n, &o, "recv", true);
    if (rc != HCCL_SUCCESS) return rc;
    const uint32_t vpr = static_cast<uint32_t>(row_bytes / 16);
    if (vpr >= kLongRow) {
        return launch_scatter_pieces(device_ctx()->moe_scatter_rows, static_cast<hipStream_t>(stream), s, d, p, as_mutable(o), n,
                                     entries / topk, topk, vpr, static_cast<uint32_t>(esz), sdispls, rdispls);
    }
    const uint64_t blocks = (static_cast<uint64_t>(entries) * vpr + 511) / 512;
    if (blocks > 0x7fffffffull) return fail(HCCL_E_PARA, "too much data for one launch");
    HCCLX_LAUNCH(k_moe_dispatch, dim3(static_cast<uint32_t>(blocks), n), dim3(256), 0, static_cast<hipStream_t>(stream), s, d,
                       p, as_mutable(o), n, entries, topk, vpr, static_cast<uint32_t>(esz), sdispls, rdispls);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail_hip(e, "moe dispatch kernel");
    return HCCL_SUCCESS;
}

int hcclx_moe_gather_combine(const void *const *expert, const int32_t *const *dest, const uint32_t *const *perm, uint32_t n,
                             uint32_t tokens, uint32_t topk, uint64_t row_elems, int dtype, const uint64_t *sdispls,
                             const uint64_t *rdispls, void *const *out, void *stream)
{
    if (!device_ctx()) return HCCL_E_RUNTIME;
    int rc = check_ranks(n);
    if (rc != HCCL_SUCCESS) return rc;
    const int esz = dtype_size(dtype);
    if (esz == 0) return fail(HCCL_E_NOT_SUPPORT, "unknown data type " + std::to_string(dtype));
    if (topk == 0 || tokens == 0) return fail(HCCL_E_PARA, "tokens and topk must be positive");
    const uint64_t row_bytes = row_elems * esz;
    if (row_bytes == 0 || row_bytes % 16 != 0) return fail(HCCL_E_PARA, "row size must be a positive multiple of 16 bytes");
    if (row_bytes / 16 > 0xffffffffull) return fail(HCCL_E_PARA, "row too long");
    if (topk > 1 && dtype != HCCL_DATA_TYPE_FP32 && dtype != HCCL_DATA_TYPE_FP16 && dtype != HCCL_DATA_TYPE_BFP16) {
        return fail(HCCL_E_NOT_SUPPORT, "combining several rows needs fp32, fp16 or bf16");
    }
    if (!sdispls || !rdispls) return fail(HCCL_E_PTR, "displacement table is null");
    MoeConstPtrs s, d, p, o;
    rc = fill(expert, n, &s, "expert", true);
    if (rc != HCCL_SUCCESS) return rc;
    rc = fill(reinterpret_cast<const void *const *>(dest), n, &d, "dest", false);
    if (rc != HCCL_SUCCESS) return rc;
    rc = fill(reinterpret_cast<const void *const *>(perm), n, &p, "perm", false);
    if (rc != HCCL_SUCCESS) return rc;
    rc = fill(out, n, &o, "out", true);
    if (rc != HCCL_SUCCESS) return rc;
    const uint32_t vpr = static_cast<uint32_t>(row_bytes / 16);
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int kind = topk == 1 ? HCCL_DATA_TYPE_INT8 : dtype;
    if (vpr >= kLongRow) {
        return launch_gather_pieces(kind, st, s, d, p, o, n, tokens, topk, vpr, static_cast<uint32_t>(esz), sdispls, rdispls);
    }
    const uint64_t blocks = (static_cast<uint64_t>(tokens) * vpr + 255) / 256;
    if (blocks > 0x7fffffffull) return fail(HCCL_E_PARA, "too much data for one launch");
    const dim3 grid(static_cast<uint32_t>(blocks), n);
    if (kind == HCCL_DATA_TYPE_FP32) {
        HCCLX_LAUNCH(k_moe_gather_combine<HCCL_DATA_TYPE_FP32>, grid, dim3(256), 0, st, s, d, p, as_mutable(o), n, tokens, topk,
                           vpr, static_cast<uint32_t>(esz), sdispls, rdispls);
    } else if (kind == HCCL_DATA_TYPE_FP16) {
        HCCLX_LAUNCH(k_moe_gather_combine<HCCL_DATA_TYPE_FP16>, grid, dim3(256), 0, st, s, d, p, as_mutable(o), n, tokens, topk,
                           vpr, static_cast<uint32_t>(esz), sdispls, rdispls);
    } else if (kind == HCCL_DATA_TYPE_BFP16) {
        HCCLX_LAUNCH(k_moe_gather_combine<HCCL_DATA_TYPE_BFP16>, grid, dim3(256), 0, st, s, d, p, as_mutable(o), n, tokens, topk,
                           vpr, static_cast<uint32_t>(esz), sdispls, rdispls);
    } else {
        HCCLX_LAUNCH(k_moe_gather_combine<HCCL_DATA_TYPE_INT8>, grid, dim3(256), 0, st, s, d, p, as_mutable(o), n, tokens, topk,
                           vpr, static_cast<uint32_t>(esz), sdispls, rdispls);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail_hip(e, "moe gather-combine kernel");
    return HCCL_SUCCESS;
}

}  // extern "C"
