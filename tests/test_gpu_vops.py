"""GPU parity of the V-collective kernels (hcclx_alltoallv, hcclx_allgatherv) against the API contract."""
import json
import os

import numpy as np
import pytest
import torch

from oracle import templates as T
from hccl_amd import hcclx
from hccl_amd._lib import HcclError

from gpu_util import DevBuf

pytestmark = pytest.mark.gpu
GOLD = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "st_cases.json")))
NAME2DT = {"int8": T.INT8, "fp16": T.FP16, "bf16": T.BFP16, "int32": T.INT32, "fp32": T.FP32, "fp64": T.FP64}


def run_a2av(m, dtype, rng, on_device=False, send_pad=0):
    n = len(m)
    esz = T.DTYPE_SIZE[dtype]
    npd = {1: np.uint8, 2: np.uint16, 4: np.uint32, 8: np.uint64}[esz]
    v = [T.alltoallvc_to_v(m, r) for r in range(n)]
    ins = [rng.integers(0, np.iinfo(npd).max, size=sum(m[i]), dtype=npd, endpoint=True) for i in range(n)]
    want = T.run_alltoallv(ins, [x[0] for x in v], [x[1] for x in v], [x[2] for x in v], [x[3] for x in v],
                           [sum(x[2]) for x in v])
    send = [DevBuf(x, offset=send_pad) for x in ins]
    recv = [DevBuf(nbytes=sum(x[2]) * esz) for x in v]
    sc = np.array([x[0] for x in v], dtype=np.uint64).ravel()
    sd = np.array([x[1] for x in v], dtype=np.uint64).ravel()
    rd = np.array([x[3] for x in v], dtype=np.uint64).ravel()
    if on_device:
        tab = torch.from_numpy(np.concatenate([sc, sd, rd]).astype(np.int64)).to("cuda:0")
        p = tab.data_ptr()
        hcclx.alltoallv([s.ptr for s in send], [r.ptr for r in recv], p, p + 8 * n * n, p + 16 * n * n, dtype,
                        on_device=True)
    else:
        hcclx.alltoallv([s.ptr for s in send], [r.ptr for r in recv], sc, sd, rd, dtype)
    torch.cuda.synchronize()
    for j in range(n):
        assert np.array_equal(recv[j].get(npd), want[j]), f"rank {j}"
        assert recv[j].guard_intact()


@pytest.mark.parametrize("case", GOLD["alltoallv"], ids=lambda c: c["name"])
@pytest.mark.parametrize("on_device", [False, True])
def test_alltoallv_reference_matrices(case, on_device):
    # counts of the reference's system tests divided by 2^13 (rounded up): zero cells stay zero
    m = [[-(-c // (1 << 13)) for c in row] for row in case["matrix"]]
    run_a2av(m, NAME2DT[case["dtype"]], np.random.default_rng(len(m)), on_device)


def test_alltoallv_odd_counts_and_misaligned_blocks():
    rng = np.random.default_rng(4)
    for n in (2, 3, 8, 13):
        m = rng.integers(0, 5000, size=(n, n)).tolist()
        m[0][0] = 0
        m[n - 1][0] = 1
        run_a2av(m, T.INT8, rng, send_pad=3)
        run_a2av(m, T.BFP16, rng)


@pytest.mark.parametrize("n", [2, 8, 16, 24, 40, 64])
def test_alltoallv_host_tables_of_any_rank_count_and_as_a_plan(n):
    """Up to 15 ranks the tables ride in the kernel arguments; beyond, the non-empty blocks become a list in device
    memory.  The same exchange as a plan moves new data at every launch, also from a captured graph."""
    rng = np.random.default_rng(n)
    m = rng.integers(0, 3000, size=(n, n))
    m[rng.random((n, n)) < 0.3] = 0                     # empty blocks
    m = m.tolist()
    run_a2av(m, T.BFP16, rng, send_pad=2)
    run_a2av(m, T.INT8, rng, send_pad=1)
    v = [T.alltoallvc_to_v(m, r) for r in range(n)]
    sc = np.array([x[0] for x in v], dtype=np.uint64).ravel()
    sd = np.array([x[1] for x in v], dtype=np.uint64).ravel()
    rd = np.array([x[3] for x in v], dtype=np.uint64).ravel()
    send = [DevBuf(nbytes=max(1, sum(m[i])) * 4) for i in range(n)]
    recv = [DevBuf(nbytes=max(1, sum(x[2])) * 4) for x in v]
    plan = hcclx.AlltoAllVPlan([s.ptr for s in send], [r.ptr for r in recv], sc, sd, rd, T.FP32)
    assert plan.bytes == 2 * 4 * int(sc.sum()) and plan.table_bytes > 0
    stream = torch.cuda.Stream()
    graph = None
    for rep in range(4):
        ins = [rng.integers(0, 2**32 - 1, size=max(1, sum(m[i])), dtype=np.uint32) for i in range(n)]
        for i in range(n):
            send[i].t[:ins[i].nbytes] = torch.from_numpy(ins[i].view(np.uint8).copy()).to("cuda:0")
        for r in recv:
            r.t.fill_(0xA5)
        torch.cuda.synchronize()
        if rep < 2:
            plan.launch(stream.cuda_stream)
        else:
            if graph is None:
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.stream(stream):
                    graph.capture_begin()
                    plan.launch(stream.cuda_stream)
                    graph.capture_end()
            graph.replay()
        torch.cuda.synchronize()
        want = T.run_alltoallv([x[:sum(m[i])] for i, x in enumerate(ins)], [x[0] for x in v], [x[1] for x in v],
                               [x[2] for x in v], [x[3] for x in v], [sum(x[2]) for x in v])
        for j in range(n):
            assert np.array_equal(recv[j].get(np.uint32)[:sum(v[j][2])], want[j]), (rep, j)
            assert recv[j].guard_intact()
    del graph
    plan.close()


@pytest.mark.parametrize("n,least,most,hot", [
    (2, 1, 9, 5 << 20),             # one block with more than 256 tiles and three of a few bytes
    (3, 4095, 4097, 0),             # one or two tiles each
    (15, 0, 60000, 3 << 20),        # the most ranks whose tables ride in the kernel arguments, 225 blocks
    (16, 0, 60000, 3 << 20),        # the fewest whose tables lie in memory
    (64, 0, 9000, 1 << 20),         # a table of more than 16 KiB, read by a kernel from pinned memory
])
def test_alltoallv_slabs_of_unequal_blocks(n, least, most, hot):
    rng = np.random.default_rng(n)
    m = rng.integers(least, most + 1, size=(n, n))
    if hot:
        m[n - 1][0] = hot + 13
    run_a2av(m.tolist(), T.INT8, rng, send_pad=n % 7)


@pytest.mark.parametrize("n,hot", [(64, 16 << 20), (63, 9 << 20), (60, 3 << 20), (15, 16 << 20)])
def test_alltoallv_one_long_block_among_many_short_ones(n, hot):
    """No block empty: as many workgroups as there are tiles, also where one block has most of them; the call and the plan.  One
    kernel is counted, whether or not the table is large enough to be brought to the device by a kernel of its own."""
    rng = np.random.default_rng(n)
    m = rng.integers(1, 300, size=(n, n))
    m[n // 2][n - 1] = hot + 5
    m = m.tolist()
    before = hcclx.kernels_launched()
    run_a2av(m, T.INT8, rng, send_pad=1)
    assert hcclx.kernels_launched() - before == 1
    v = [T.alltoallvc_to_v(m, r) for r in range(n)]
    ins = [rng.integers(0, 256, size=sum(m[i]), dtype=np.uint8) for i in range(n)]
    want = T.run_alltoallv(ins, [x[0] for x in v], [x[1] for x in v], [x[2] for x in v], [x[3] for x in v], [sum(x[2]) for x in v])
    send = [DevBuf(x) for x in ins]
    recv = [DevBuf(nbytes=sum(x[2]), offset=j % 17) for j, x in enumerate(v)]
    plan = hcclx.AlltoAllVPlan([s.ptr for s in send], [r.ptr for r in recv], np.array([x[0] for x in v], np.uint64).ravel(),
                               np.array([x[1] for x in v], np.uint64).ravel(), np.array([x[3] for x in v], np.uint64).ravel(), T.INT8)
    plan.launch()
    torch.cuda.synchronize()
    plan.close()
    for j in range(n):
        assert np.array_equal(recv[j].get(np.uint8), want[j]) and recv[j].guard_intact(), j


@pytest.mark.parametrize("n,count", [(15, 78643201), (64, 4456449)])
def test_alltoallv_of_more_tiles_than_one_launch_takes(n, count):
    """More than 64 GiB (2^24 tiles) in two launches, tables in the kernel arguments and in memory.  All blocks are copies of
    the same few MiB, and those of the first launch go to the same place; the blocks of the last rows, where the second launch
    begins, each have a place of their own."""
    own = n - (1 if n == 15 else 4)     # from this row on
    g = torch.Generator(device="cuda:0")
    g.manual_seed(n)
    src = torch.randint(-2**31, 2**31 - 1, (count + 1,), device="cuda:0", generator=g, dtype=torch.int32)
    rest = (n - own) * n
    dst = torch.zeros((rest + 1) * count + 1, device="cuda:0", dtype=torch.int32)
    sdispls = [1 if i >= own else 0 for i in range(n) for _ in range(n)]
    rdispls = [(1 + (i - own) * n + j) * count if i >= own else 0 for j in range(n) for i in range(n)]
    counts = [count] * (n * n)
    torch.cuda.synchronize()
    send, recv = [src.data_ptr()] * n, [dst.data_ptr()] * n
    plan = hcclx.AlltoAllVPlan(send, recv, counts, sdispls, rdispls, T.FP32)
    for go in (lambda: hcclx.alltoallv(send, recv, counts, sdispls, rdispls, T.FP32), plan.launch):
        before = hcclx.kernels_launched()
        go()
        assert hcclx.kernels_launched() - before >= 2
        torch.cuda.synchronize()
        assert torch.equal(dst[:count], src[:-1])
        for k in range(1, rest + 1):
            assert torch.equal(dst[k * count:(k + 1) * count], src[1:]), k
        assert int(dst[-1]) == 0
        dst.zero_()
    plan.close()


@pytest.mark.parametrize("n,rows", [(23, 168), (24, 144), (40, 56)])
def test_alltoallv_of_many_blocks_and_160_mib_is_streamed(n, rows):
    """529 and 576 blocks, 40960 tiles and more; blocks of half to one and a half KiB times rows, at any alignment."""
    rng = np.random.default_rng(n)
    m = rng.integers(rows * 1024, rows * 3072, size=(n, n))
    assert m.sum() > 160 << 20 and (m > 0).sum() >= 512
    run_a2av(m.tolist(), T.INT8, rng, send_pad=3)


def test_alltoallv_all_zero_and_single_rank():
    rng = np.random.default_rng(1)
    run_a2av([[0, 0], [0, 0]], T.FP32, rng)
    run_a2av([[777]], T.FP32, rng)


def test_alltoallv_moe_dispatch_shape_small():
    """4 ranks x 96 tokens x hidden 7168 bf16, destinations Zipf(1.2): the MoE dispatch layout."""
    rng = np.random.default_rng(12)
    n, tokens, hidden = 4, 96, 7168
    w = 1.0 / np.arange(1, n + 1) ** 1.2
    w /= w.sum()
    m = [(np.bincount(rng.choice(n, size=tokens, p=w), minlength=n) * hidden).tolist() for _ in range(n)]
    run_a2av(m, T.BFP16, rng, on_device=True)


def run_agv(counts, displs, dtype, rng, on_device=False, total=None):
    n = len(counts)
    esz = T.DTYPE_SIZE[dtype]
    npd = {1: np.uint8, 2: np.uint16, 4: np.uint32, 8: np.uint64}[esz]
    total = total if total is not None else max(d + c for d, c in zip(displs, counts))
    ins = [rng.integers(0, np.iinfo(npd).max, size=c, dtype=npd, endpoint=True) for c in counts]
    fill = np.frombuffer(bytes([0xA5]) * (total * esz), dtype=npd)
    want = T.run_allgatherv(ins, counts, displs, total, fill)
    send = [DevBuf(x) for x in ins]
    recv = [DevBuf(nbytes=total * esz) for _ in range(n)]
    c64, d64 = np.array(counts, dtype=np.uint64), np.array(displs, dtype=np.uint64)
    if on_device:
        tab = torch.from_numpy(np.concatenate([c64, d64]).astype(np.int64)).to("cuda:0")
        hcclx.allgatherv([s.ptr for s in send], [r.ptr for r in recv], tab.data_ptr(), tab.data_ptr() + 8 * n, dtype,
                         on_device=True)
    else:
        hcclx.allgatherv([s.ptr for s in send], [r.ptr for r in recv], c64, d64, dtype)
    torch.cuda.synchronize()
    for j in range(n):
        assert np.array_equal(recv[j].get(npd), want[j]), f"rank {j}"
        assert recv[j].guard_intact()


@pytest.mark.parametrize("case", GOLD["allgatherv"], ids=lambda c: c["name"])
def test_allgatherv_reference_lists(case):
    div = 1 << 8 if max(case["counts"]) > 100000 else 1
    counts = [-(-c // div) for c in case["counts"]]
    displs = [sum(counts[:i]) for i in range(len(counts))] if div > 1 else case["displs"]
    run_agv(counts, displs, NAME2DT[case["dtype"]], np.random.default_rng(3))


def test_allgatherv_ragged_with_gaps_and_zero_counts():
    rng = np.random.default_rng(6)
    counts = [0, 1, 4097, 0, 33, 70001, 15, 2]
    displs, off = [], 5
    for c in counts:
        displs.append(off)
        off += c + 3          # holes between blocks must stay untouched
    run_agv(counts, displs, T.FP16, rng, total=off + 9)
    run_agv(counts, displs, T.INT8, rng, on_device=True, total=off + 9)
    run_agv([0, 0, 0], [0, 0, 0], T.FP32, rng, total=4)


def test_allgatherv_16_ranks_random_counts():
    rng = np.random.default_rng(16)
    counts = rng.integers(0, 40000, size=16).tolist()
    displs = [sum(counts[:i]) for i in range(16)]
    run_agv(counts, displs, T.FP16, rng, on_device=True)


@pytest.mark.parametrize("rows,n", [(1, 1), (1, 16), (8, 8), (64, 64), (5, 37)])
def test_displacements_from_counts_on_the_device(rows, n):
    """The exclusive prefix sum per row, by one wavefront: against numpy, with zeros and counts beyond 32 bits."""
    rng = np.random.default_rng(rows * 100 + n)
    counts = rng.integers(0, 1 << 20, size=(rows, n)).astype(np.uint64)
    counts[rng.random((rows, n)) < 0.2] = 0
    counts[0, n // 2] = (1 << 35) + 7
    dc = torch.from_numpy(counts.view(np.int64)).to("cuda:0")
    dd = torch.full((rows, n), -1, dtype=torch.int64, device="cuda:0")
    dt = torch.full((rows,), -1, dtype=torch.int64, device="cuda:0")
    hcclx.displs_from_counts(dc.data_ptr(), rows, n, dd.data_ptr(), dt.data_ptr())
    torch.cuda.synchronize()
    want = np.cumsum(counts, axis=1) - counts
    assert np.array_equal(dd.cpu().numpy().view(np.uint64), want)
    assert np.array_equal(dt.cpu().numpy().view(np.uint64), counts.sum(axis=1))
    dd.fill_(-1)
    hcclx.displs_from_counts(dc.data_ptr(), rows, n, dd.data_ptr())          # totals are optional
    torch.cuda.synchronize()
    assert np.array_equal(dd.cpu().numpy().view(np.uint64), want)


def test_allgatherv_with_counts_and_displacements_that_never_leave_the_device():
    """Config 3 of the baseline in small: 16 ranks, ragged fp16 blocks packed back to back; the displacements come
    from the counts by the device prefix sum and feed hcclx_allgatherv with tables_on_device."""
    rng = np.random.default_rng(3)
    n = 16
    counts = rng.integers(0, 50000, size=n).astype(np.uint64)
    counts[5] = 0
    ins = [rng.integers(0, 65536, size=int(c), dtype=np.uint16) for c in counts]
    total = int(counts.sum())
    send = [DevBuf(x) if x.size else DevBuf(nbytes=2) for x in ins]
    recv = [DevBuf(nbytes=total * 2) for _ in range(n)]
    dc = torch.from_numpy(counts.view(np.int64)).to("cuda:0")
    dd = torch.empty(n, dtype=torch.int64, device="cuda:0")
    hcclx.displs_from_counts(dc.data_ptr(), 1, n, dd.data_ptr())
    hcclx.allgatherv([s.ptr for s in send], [r.ptr for r in recv], dc.data_ptr(), dd.data_ptr(), T.FP16, on_device=True)
    torch.cuda.synchronize()
    displs = (np.cumsum(counts) - counts).astype(np.int64).tolist()
    want = T.run_allgatherv(ins, [int(c) for c in counts], displs, total, 0)
    for j in range(n):
        assert np.array_equal(recv[j].get(np.uint16), want[j]), f"rank {j}"
        assert recv[j].guard_intact()


SLAB = 32768    # eight tiles, one for each XCD, of the copy kernel that writes one output at a time


@pytest.mark.parametrize("n,sizes,pad", [
    (2, [(4 << 20) + 1, 1], 0),                                                     # one long source, one of a byte
    (5, [SLAB - 1, SLAB, SLAB + 1, 3 * SLAB + 1008, 4 << 20], 5),                   # around whole tiles, shifted places
    (16, [300000 + 4099 * k for k in range(16)], 3),                                # no two sources of one length
    (64, [(k % 7) * SLAB + (k * 37) % 1031 + (0 if k % 9 else -1) for k in range(64)], 2),   # most ranks, empty sources
])
def test_allgatherv_written_one_output_at_a_time(n, sizes, pad):
    """From 4 MiB of payload: the tiles of the sources, batch by batch to one receive buffer after the other; receive
    buffers of different alignment, holes between the blocks."""
    counts = [max(0, c) for c in sizes]
    counts[0] += max(0, (4 << 20) - sum(counts))
    displs = [sum(counts[:i]) + i * pad for i in range(n)]
    rng = np.random.default_rng(n)
    total = displs[-1] + counts[-1] + 7
    ins = [rng.integers(0, 256, size=c, dtype=np.uint8) for c in counts]
    want = T.run_allgatherv(ins, counts, displs, total, np.full(total, 0xA5, np.uint8))
    send = [DevBuf(x, offset=i % 3) for i, x in enumerate(ins)]
    recv = [DevBuf(nbytes=total, offset=(j * 5) % 48) for j in range(n)]
    hcclx.allgatherv([b.ptr for b in send], [b.ptr for b in recv], np.array(counts, np.uint64), np.array(displs, np.uint64), T.INT8)
    torch.cuda.synchronize()
    for j in range(n):
        assert np.array_equal(recv[j].get(np.uint8), want[j]), f"rank {j}"
        assert recv[j].guard_intact()


def test_allgatherv_payload_beyond_one_launch_of_the_largest_slabs():
    counts = [(1 << 30) + 4099, (1 << 30) + 77]
    g = torch.Generator(device="cuda:0")
    g.manual_seed(4)
    send = [torch.randint(0, 256, (c,), device="cuda:0", generator=g, dtype=torch.uint8) for c in counts]
    recv = [torch.zeros(sum(counts), device="cuda:0", dtype=torch.uint8) for _ in counts]
    torch.cuda.synchronize()
    before = hcclx.kernels_launched()
    hcclx.allgatherv([t.data_ptr() for t in send], [t.data_ptr() for t in recv], counts, [0, counts[0]], T.INT8)
    assert hcclx.kernels_launched() - before == 2
    torch.cuda.synchronize()
    for t in recv:
        assert torch.equal(t[:counts[0]], send[0]) and torch.equal(t[counts[0]:], send[1])


@pytest.mark.parametrize("nseg", [1, 37, 200])
def test_copies_to_several_places_of_different_number(nseg):
    """The same kernel with its tables in memory: segments that only copy, 1 to 16 places each, 4 MiB and more."""
    rng = np.random.default_rng(nseg)
    counts = [int(c) for c in rng.integers(1, 2 * (5 << 20) // nseg, size=nseg)]
    counts[0] += max(0, (5 << 20) - sum(counts))
    fans = [int(f) for f in rng.integers(2, 17, size=nseg)]
    if nseg > 1:
        fans[1] = 1
    ins = [rng.integers(0, 256, size=c, dtype=np.uint8) for c in counts]
    src = [DevBuf(x, offset=i % 5) for i, x in enumerate(ins)]
    dst = [[DevBuf(nbytes=c, offset=(3 * i + 7 * k) % 21) for k in range(f)] for i, (c, f) in enumerate(zip(counts, fans))]
    segs = [(c, [s.ptr], [d.ptr for d in ds]) for c, s, ds in zip(counts, src, dst)]
    plan = hcclx.Plan(segs, T.INT8)
    for go in (lambda: hcclx.fold(segs, T.INT8), plan.launch):
        go()
        torch.cuda.synchronize()
        for x, ds in zip(ins, dst):
            for d in ds:
                assert np.array_equal(d.get(np.uint8), x) and d.guard_intact()
                d.t.fill_(0xA5)
    plan.close()


@pytest.mark.parametrize("n,count,dtype", [(1, 5, T.INT8), (2, 1, T.INT8), (3, 4095, T.INT8), (8, 2049, T.BFP16), (16, 4097, T.FP32),
                                           (33, 1023, T.INT16), (64, 7, T.INT64), (5, 700001, T.INT8)])
def test_alltoall_of_equal_blocks_needs_no_table(n, count, dtype):
    """Equal blocks back to back: one launch, no upload; one byte, whole tiles and one element more or less, blocks at any
    alignment."""
    esz = T.DTYPE_SIZE[dtype]
    rng = np.random.default_rng(n + count)
    ins = [rng.integers(0, 256, size=n * count * esz, dtype=np.uint8) for _ in range(n)]
    src = [DevBuf(x, offset=(i * esz) % 32) for i, x in enumerate(ins)]
    dst = [DevBuf(nbytes=n * count * esz, offset=(3 * i * esz) % 40) for i in range(n)]
    displs = [j * count for j in range(n)] * n
    before = hcclx.kernels_launched()
    hcclx.alltoallv([s.ptr for s in src], [d.ptr for d in dst], [count] * (n * n), displs, displs, dtype)
    torch.cuda.synchronize()
    assert hcclx.kernels_launched() - before == 1
    for j in range(n):
        want = np.concatenate([ins[i][j * count * esz:(j + 1) * count * esz] for i in range(n)])
        assert np.array_equal(dst[j].get(np.uint8), want) and dst[j].guard_intact(), j


def test_v_ops_reject_bad_arguments():
    b = DevBuf(nbytes=64)
    with pytest.raises(HcclError) as e:
        hcclx.alltoallv([b.ptr] * 65, [b.ptr] * 65, [0] * 65 * 65, [0] * 65 * 65, [0] * 65 * 65, T.INT8)
    assert e.value.code == 1
    with pytest.raises(HcclError) as e:
        hcclx.allgatherv([b.ptr], [b.ptr], [1], [0], 99)
    assert e.value.code == 5
