"""GPU parity of the MoE dispatch entry points (hcclx_moe_route / _pack / _combine) against the oracle, and the
dispatch -> AlltoAllV -> AlltoAllV back -> combine round trip at the size of the baseline's MoE configuration."""
import numpy as np
import pytest
import torch

from oracle import templates as T
from hccl_amd import hcclx
from hccl_amd._lib import HcclError

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def dev_i32(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).to(DEV)


def route_on_gpu(dests, n, entries, row_elems, skew=0):
    """`skew`: rank i's destination array starts (i * skew) % 4 entries into its allocation, so that some arrays
    are not 16-byte aligned."""
    whole = [dev_i32(np.concatenate([np.zeros((i * skew) % 4, dtype=np.int32), np.asarray(x, dtype=np.int32)]))
             for i, x in enumerate(dests)]
    d = [w[(i * skew) % 4:] for i, w in enumerate(whole)]
    tabs = [torch.full((n * n,), -1, dtype=torch.int64, device=DEV) for _ in range(4)]
    perm = [torch.full((entries,), 12345, dtype=torch.int32, device=DEV) for _ in range(n)]
    ws = torch.empty(hcclx.moe_workspace_bytes(n, entries), dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    hcclx.moe_route([x.data_ptr() for x in d], entries, row_elems, tabs[0].data_ptr(), tabs[1].data_ptr(),
                    tabs[2].data_ptr(), tabs[3].data_ptr(), [p.data_ptr() for p in perm], ws.data_ptr())
    torch.cuda.synchronize()
    return tabs, perm


@pytest.mark.parametrize("n,entries", [(1, 5), (2, 256), (3, 257), (8, 4096), (8, 70001), (16, 1000), (64, 33333),
                                       (64, 3001), (33, 7942), (16, 16384), (16, 16385), (5, 3), (12, 4099)])
@pytest.mark.parametrize("skew", [0, 1])
def test_route_tables_and_stable_permutation(n, entries, skew):
    """Both routing paths (two launches while a rank has at most 64 chunks of 256 entries and the per-chunk histogram at
    most 16384 cells, three beyond), with destination arrays that are and are not 16-byte aligned."""
    rng = np.random.default_rng(n * 1000 + entries)
    p = 1.0 / np.arange(1, n + 1) ** 1.2
    dests = [rng.choice(n, size=entries, p=p / p.sum()) for _ in range(n)]
    dests[0][::7] = -1                      # dropped entries
    if n > 1:
        dests[1][::5] = n
    tabs, perm = route_on_gpu(dests, n, entries, 24, skew)
    sc, sd, rc, rd, perms = T.moe_route(dests, n, 24)
    for got, want in zip(tabs, (sc, sd, rc, rd)):
        assert np.array_equal(got.cpu().numpy().reshape(n, n), np.array(want, dtype=np.int64))
    for i in range(n):
        assert np.array_equal(perm[i].cpu().numpy().view(np.uint32), perms[i]), i


@pytest.mark.parametrize("topk,dtype,width", [(1, T.BFP16, 64), (2, T.BFP16, 40), (4, T.FP32, 12), (3, T.FP16, 8),
                                              (1, T.INT8, 48), (2, T.BFP16, 3000), (1, T.FP32, 1032), (4, T.FP16, 1024)])
def test_pack_and_combine_match_the_oracle(topk, dtype, width):
    rng = np.random.default_rng(topk * 10 + dtype)
    n, tokens = 4, 777
    entries = tokens * topk
    npd = T.NP_STORAGE[dtype]
    esz = T.DTYPE_SIZE[dtype]
    dests = [rng.integers(0, n + 1, size=entries) for _ in range(n)]            # n = dropped
    if dtype == T.FP32:
        toks = [rng.standard_normal((tokens, width)).astype(np.float32) for _ in range(n)]
    elif dtype == T.INT8:
        toks = [rng.integers(-128, 127, size=(tokens, width), dtype=np.int8) for _ in range(n)]
    else:
        toks = [T.narrow16(rng.standard_normal(tokens * width).astype(np.float32), dtype).reshape(tokens, width)
                for _ in range(n)]
    tabs, perm = route_on_gpu(dests, n, entries, width)
    _, _, _, _, perms = T.moe_route(dests, n, width)
    kept = [int(np.count_nonzero(p != T.MOE_DROPPED)) for p in perms]
    d_tok = [torch.from_numpy(t.view(np.uint8).reshape(-1).copy()).to(DEV) for t in toks]
    d_pack = [torch.full((max(1, k) * width * esz + 64,), 0xEE, dtype=torch.uint8, device=DEV) for k in kept]
    torch.cuda.synchronize()
    hcclx.moe_pack([t.data_ptr() for t in d_tok], [p.data_ptr() for p in perm], entries, topk, width * esz,
                   [t.data_ptr() for t in d_pack])
    torch.cuda.synchronize()
    packed = []
    for i in range(n):
        want = T.moe_pack(toks[i], perms[i], topk, max(1, kept[i]))
        got = d_pack[i].cpu().numpy()
        assert np.array_equal(got[:kept[i] * width * esz].view(npd), want[:kept[i]].reshape(-1)), i
        assert (got[max(1, kept[i]) * width * esz:] == 0xEE).all()              # nothing past the last row
        packed.append(want)
    d_out = [torch.full((tokens * width * esz + 64,), 0xEE, dtype=torch.uint8, device=DEV) for _ in range(n)]
    torch.cuda.synchronize()
    hcclx.moe_combine([t.data_ptr() for t in d_pack], [p.data_ptr() for p in perm], tokens, topk, width, dtype,
                      [t.data_ptr() for t in d_out])
    torch.cuda.synchronize()
    for i in range(n):
        want = T.moe_combine(packed[i], perms[i], topk, dtype)
        got = d_out[i].cpu().numpy()
        assert np.array_equal(got[:tokens * width * esz].view(npd).reshape(tokens, width).view(np.uint8),
                              want.view(np.uint8)), i
        assert (got[tokens * width * esz:] == 0xEE).all()


@pytest.mark.parametrize("topk,dtype,width,n,tokens", [(1, T.BFP16, 64, 4, 777), (2, T.BFP16, 40, 5, 300),
                                                        (4, T.FP32, 12, 3, 513), (3, T.FP16, 8, 8, 1000),
                                                        (1, T.INT8, 48, 2, 257), (2, T.FP32, 4, 64, 96),
                                                        # rows of 128 vectors and more: the kernels that move one row per workgroup
                                                        (2, T.BFP16, 3000, 4, 61), (1, T.FP32, 1032, 3, 100),
                                                        (3, T.FP16, 1024, 5, 40), (1, T.INT8, 16 * 129, 2, 33)])
def test_fused_dispatch_and_gather_combine_equal_the_two_pass_pipeline(topk, dtype, width, n, tokens):
    """hcclx_moe_dispatch puts every row where pack + AlltoAllV would; hcclx_moe_gather_combine gives what
    AlltoAllV back + combine would: checked against the oracle's pack -> alltoallv -> alltoallv -> combine."""
    rng = np.random.default_rng(topk * 100 + dtype + n)
    entries = tokens * topk
    npd = T.NP_STORAGE[dtype]
    esz = T.DTYPE_SIZE[dtype]
    dests = [rng.integers(-1, n + 1, size=entries) for _ in range(n)]            # -1 and n are dropped
    if dtype == T.FP32:
        toks = [rng.standard_normal((tokens, width)).astype(np.float32) for _ in range(n)]
    elif dtype == T.INT8:
        toks = [rng.integers(-128, 127, size=(tokens, width), dtype=np.int8) for _ in range(n)]
    else:
        toks = [T.narrow16(rng.standard_normal(tokens * width).astype(np.float32), dtype).reshape(tokens, width)
                for _ in range(n)]
    tabs, perm = route_on_gpu(dests, n, entries, width)
    sc, sd, rc, rd, perms = T.moe_route(dests, n, width)
    kept = [int(np.count_nonzero(p != T.MOE_DROPPED)) for p in perms]
    inbound = [sum(rc[j]) // width for j in range(n)]
    # the oracle's two-pass pipeline, in elements
    packed = [T.moe_pack(toks[i], perms[i], topk, max(1, kept[i])).reshape(-1) for i in range(n)]
    recv_want = T.run_alltoallv(packed, sc, sd, rc, rd, [max(1, r) * width for r in inbound], fill=0)
    d_dest = [dev_i32(x) for x in dests]
    d_tok = [torch.from_numpy(t.view(np.uint8).reshape(-1).copy()).to(DEV) for t in toks]
    d_recv = [torch.full((max(1, r) * width * esz + 64,), 0xEE, dtype=torch.uint8, device=DEV) for r in inbound]
    torch.cuda.synchronize()
    ptrs = lambda ts: [t.data_ptr() for t in ts]
    hcclx.moe_dispatch(ptrs(d_tok), ptrs(d_dest), ptrs(perm), entries, topk, width, dtype, tabs[1].data_ptr(),
                       tabs[3].data_ptr(), ptrs(d_recv))
    torch.cuda.synchronize()
    for j in range(n):
        got = d_recv[j].cpu().numpy()
        assert np.array_equal(got[:inbound[j] * width * esz].view(npd), recv_want[j][:inbound[j] * width]), j
        assert (got[max(1, inbound[j]) * width * esz:] == 0xEE).all()
    # the experts' results: any function of the received rows; here the rows with their bytes reversed per row pair
    expert = [np.ascontiguousarray(r[:inbound[j] * width].reshape(-1, width)[:, ::-1]).reshape(-1) for j, r in enumerate(recv_want)]
    back = T.run_alltoallv([np.concatenate([e, np.zeros(width, dtype=npd)]) for e in expert], rc, rd, sc, sd,
                           [max(1, k) * width for k in kept], fill=0)
    d_exp = [torch.from_numpy(np.concatenate([e, np.zeros(width, dtype=npd)]).view(np.uint8).copy()).to(DEV) for e in expert]
    d_out = [torch.full((tokens * width * esz + 64,), 0xEE, dtype=torch.uint8, device=DEV) for _ in range(n)]
    torch.cuda.synchronize()
    hcclx.moe_gather_combine(ptrs(d_exp), ptrs(d_dest), ptrs(perm), tokens, topk, width, dtype, tabs[1].data_ptr(),
                             tabs[3].data_ptr(), ptrs(d_out))
    torch.cuda.synchronize()
    for i in range(n):
        want = T.moe_combine(back[i].reshape(-1, width), perms[i], topk, dtype)
        got = d_out[i].cpu().numpy()
        assert np.array_equal(got[:tokens * width * esz].view(npd).reshape(tokens, width).view(np.uint8),
                              want.view(np.uint8)), i
        assert (got[tokens * width * esz:] == 0xEE).all()


def test_errors():
    t = torch.zeros(4096, dtype=torch.uint8, device=DEV)
    p = t.data_ptr()
    with pytest.raises(HcclError) as e:
        hcclx.moe_pack([p], [p], 8, 3, 64, [p])              # entries not a multiple of topk
    assert e.value.code == 1
    with pytest.raises(HcclError) as e:
        hcclx.moe_pack([p], [p], 8, 1, 24, [p])              # rows must be multiples of 16 bytes
    assert e.value.code == 1
    with pytest.raises(HcclError) as e:
        hcclx.moe_pack([p + 4], [p], 8, 1, 64, [p])          # 16-byte aligned buffers
    assert e.value.code == 1
    with pytest.raises(HcclError) as e:
        hcclx.moe_combine([p], [p], 8, 2, 16, T.INT32, [p])  # several rows can only be added as floats
    assert e.value.code == 5
    with pytest.raises(HcclError) as e:
        hcclx.moe_pack([p, 0], [p, p], 8, 1, 64, [p, p])
    assert e.value.code == 2


def test_moe_dispatch_round_trip_at_baseline_size():
    """8 ranks x 4096 tokens x hidden 7168 bf16, Zipf(1.2) destinations, routed on the device: pack, AlltoAllV
    with device tables, AlltoAllV back with the transposed tables, combine: every rank gets its tokens back;
    what rank j receives is, rank by rank, the senders' tokens for j in token order."""
    n, tokens, hidden = 8, 4096, 7168
    rng = np.random.default_rng(0)
    p = 1.0 / np.arange(1, n + 1) ** 1.2
    dests = [rng.choice(n, size=tokens, p=p / p.sum()) for _ in range(n)]
    d_dest = [dev_i32(x) for x in dests]
    toks = [torch.randint(-32768, 32767, (tokens, hidden), device=DEV, dtype=torch.int16) for _ in range(n)]
    packed = [torch.empty(tokens * hidden, device=DEV, dtype=torch.int16) for _ in range(n)]
    tabs = [torch.zeros(n * n, dtype=torch.int64, device=DEV) for _ in range(4)]     # send_counts, sdispls, recv_counts, rdispls
    perm = [torch.empty(tokens, dtype=torch.int32, device=DEV) for _ in range(n)]
    ws = torch.empty(hcclx.moe_workspace_bytes(n, tokens), dtype=torch.uint8, device=DEV)
    inbound = np.zeros(n, dtype=np.int64)
    for i in range(n):
        inbound += np.bincount(dests[i], minlength=n)
    recv = [torch.full((max(1, int(inbound[j])) * hidden,), 0x2222, device=DEV, dtype=torch.int16) for j in range(n)]
    back = [torch.full((tokens * hidden,), 0x3333, device=DEV, dtype=torch.int16) for _ in range(n)]
    out = [torch.full((tokens, hidden), 0x4444, device=DEV, dtype=torch.int16) for _ in range(n)]
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    st = s.cuda_stream
    ptrs = lambda ts: [t.data_ptr() for t in ts]
    hcclx.moe_route(ptrs(d_dest), tokens, hidden, tabs[0].data_ptr(), tabs[1].data_ptr(), tabs[2].data_ptr(),
                    tabs[3].data_ptr(), ptrs(perm), ws.data_ptr(), stream=st)
    hcclx.moe_pack(ptrs(toks), ptrs(perm), tokens, 1, hidden * 2, ptrs(packed), stream=st)
    hcclx.alltoallv(ptrs(packed), ptrs(recv), tabs[0].data_ptr(), tabs[1].data_ptr(), tabs[3].data_ptr(), T.BFP16,
                    on_device=True, stream=st)
    hcclx.alltoallv(ptrs(recv), ptrs(back), tabs[2].data_ptr(), tabs[3].data_ptr(), tabs[1].data_ptr(), T.BFP16,
                    on_device=True, stream=st)
    hcclx.moe_combine(ptrs(back), ptrs(perm), tokens, 1, hidden, T.BFP16, ptrs(out), stream=st)
    s.synchronize()
    for i in range(n):
        assert torch.equal(out[i], toks[i]), i
    for j in range(n):
        pos = 0
        for i in range(n):
            mine = toks[i][torch.from_numpy(dests[i] == j).to(DEV)].reshape(-1)
            assert torch.equal(recv[j][pos:pos + mine.numel()], mine), (i, j)
            pos += mine.numel()
        assert pos == int(inbound[j]) * hidden


def test_one_pass_round_trip_at_baseline_size():
    """The same configuration through the one-pass entry points: route, dispatch straight into the receive buffers,
    gather-combine straight out of them: every rank gets its tokens back, and the receive buffers hold what the
    AlltoAllV delivers."""
    n, tokens, hidden = 8, 4096, 7168
    rng = np.random.default_rng(1)
    p = 1.0 / np.arange(1, n + 1) ** 1.2
    dests = [rng.choice(n, size=tokens, p=p / p.sum()) for _ in range(n)]
    d_dest = [dev_i32(x) for x in dests]
    toks = [torch.randint(-32768, 32767, (tokens, hidden), device=DEV, dtype=torch.int16) for _ in range(n)]
    tabs = [torch.zeros(n * n, dtype=torch.int64, device=DEV) for _ in range(4)]
    perm = [torch.empty(tokens, dtype=torch.int32, device=DEV) for _ in range(n)]
    ws = torch.empty(hcclx.moe_workspace_bytes(n, tokens), dtype=torch.uint8, device=DEV)
    inbound = np.zeros(n, dtype=np.int64)
    for i in range(n):
        inbound += np.bincount(dests[i], minlength=n)
    recv = [torch.full((max(1, int(inbound[j])) * hidden + 32,), 0x2222, device=DEV, dtype=torch.int16) for j in range(n)]
    out = [torch.full((tokens, hidden), 0x4444, device=DEV, dtype=torch.int16) for _ in range(n)]
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    st = s.cuda_stream
    ptrs = lambda ts: [t.data_ptr() for t in ts]
    hcclx.moe_route(ptrs(d_dest), tokens, hidden, tabs[0].data_ptr(), tabs[1].data_ptr(), tabs[2].data_ptr(),
                    tabs[3].data_ptr(), ptrs(perm), ws.data_ptr(), stream=st)
    hcclx.moe_dispatch(ptrs(toks), ptrs(d_dest), ptrs(perm), tokens, 1, hidden, T.BFP16, tabs[1].data_ptr(),
                       tabs[3].data_ptr(), ptrs(recv), stream=st)
    hcclx.moe_gather_combine(ptrs(recv), ptrs(d_dest), ptrs(perm), tokens, 1, hidden, T.BFP16, tabs[1].data_ptr(),
                             tabs[3].data_ptr(), ptrs(out), stream=st)
    s.synchronize()
    for i in range(n):
        assert torch.equal(out[i], toks[i]), i
    for j in range(n):
        pos = 0
        for i in range(n):
            mine = toks[i][torch.from_numpy(dests[i] == j).to(DEV)].reshape(-1)
            assert torch.equal(recv[j][pos:pos + mine.numel()], mine), (i, j)
            pos += mine.numel()
        assert pos == int(inbound[j]) * hidden
        assert bool((recv[j][pos:] == 0x2222).all())


@pytest.mark.parametrize("topk,dtype,width,n,tokens", [(4, T.BFP16, 1024, 2, 37), (5, T.FP32, 516, 3, 65), (8, T.BFP16, 1536, 8, 16),
                                                        (9, T.FP16, 1032, 2, 33), (2, T.FP32, 512, 64, 3), (6, T.BFP16, 1528, 1, 1),
                                                        (3, T.BFP16, 376, 4, 50), (3, T.BFP16, 384, 4, 50), (2, T.FP16, 392, 2, 31)])
def test_rows_cut_into_pieces(topk, dtype, width, n, tokens):
    """Rows of 48 vectors and more are moved a piece of 64 vectors per wavefront: whole pieces, one vector more and one
    less, rows around the 48 vectors, token numbers around the 32 pieces of eight workgroups, entries that do not divide by those of a wavefront."""
    test_fused_dispatch_and_gather_combine_equal_the_two_pass_pipeline(topk, dtype, width, n, tokens)


# rows of 64 vectors are one piece, so the wavefronts of a gather are tokens x ranks: those that fit 256 CUs 20 and 32 deep, and one token more
@pytest.mark.parametrize("topk,dtype,width,n,tokens", [(3, T.BFP16, 512, 8, 640), (3, T.BFP16, 512, 8, 641), (5, T.FP16, 512, 8, 1024),
                                                        (5, T.FP32, 256, 8, 1025), (2, T.BFP16, 512, 8, 1025), (8, T.FP32, 256, 1, 1),
                                                        (7, T.FP16, 520, 1, 9), (1, T.BFP16, 512, 16, 5)])
def test_entries_of_a_token_in_flight_together(topk, dtype, width, n, tokens):
    """The gather takes four, two or one of a token's entries at a time, by the launch's wavefronts: around both limits, with
    entries that four and two do not divide, and (one rank: two of three entries dropped) tokens that keep none.  The order of
    the sum is the oracle's whatever is loaded together, so the results are equal to the bit."""
    test_fused_dispatch_and_gather_combine_equal_the_two_pass_pipeline(topk, dtype, width, n, tokens)


# rows of 64 vectors: the wavefronts that fit 256 CUs 16 deep, and one token more; and 192 MiB of rows (4 x 8192 elements x 384
# tokens x 8 ranks)
@pytest.mark.parametrize("topk,dtype,width,n,tokens", [(5, T.FP16, 512, 8, 512), (5, T.FP16, 512, 8, 513), (4, T.BFP16, 8192, 8, 384),
                                                        (2, T.FP32, 260, 1, 7), (2, T.FP16, 4096, 3, 33)])
def test_entries_in_flight_together_at_the_limits(topk, dtype, width, n, tokens):
    """How many entries the gather takes at a time goes by the launch's wavefronts and by its rows: on both sides of the limits."""
    test_fused_dispatch_and_gather_combine_equal_the_two_pass_pipeline(topk, dtype, width, n, tokens)


def gather_time(n, tokens, topk, hidden, dropped):
    """us of a gather in which this share of the entries is dropped, the least of several groups of launches."""
    entries = tokens * topk
    rng = np.random.default_rng(5)
    dests = [np.where(rng.random(entries) < dropped, n, rng.integers(0, n, size=entries)) for _ in range(n)]
    tabs, perm = route_on_gpu(dests, n, entries, hidden)
    d = [dev_i32(x) for x in dests]
    landed = (tabs[2].view(n, n).sum(1) // hidden).tolist()
    rows = [torch.zeros(max(1, r) * hidden, dtype=torch.int16, device=DEV) for r in landed]
    out = [torch.zeros(tokens * hidden, dtype=torch.int16, device=DEV) for _ in range(n)]
    ptrs = [[x.data_ptr() for x in t] for t in (rows, d, perm, out)]
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    times = []
    for _ in range(8):
        torch.cuda.synchronize()
        start.record()
        for _ in range(5):
            hcclx.moe_gather_combine(*ptrs[:3], tokens, topk, hidden, T.BFP16, tabs[1].data_ptr(), tabs[3].data_ptr(), ptrs[3])
        end.record()
        torch.cuda.synchronize()
        times.append(start.elapsed_time(end) / 5e-3)
    return min(times)


@pytest.mark.parametrize("topk,share", [(1, 0.75), (2, 0.62)])
def test_entries_that_are_dropped_cost_no_bytes(topk, share):
    """A gather of which every entry is dropped only writes.  Measured 0.48 and 0.52 of the time with none dropped; 0.95 and 0.75
    when a dropped entry read something from HBM."""
    assert gather_time(8, 4096, topk, 7168, 1.0) < share * gather_time(8, 4096, topk, 7168, 0.0)


@pytest.mark.parametrize("topk,tokens,hidden", [(5, 4200, 8192), (3, 700, 7168)])
def test_dispatch_of_tokens_beyond_the_cache(topk, tokens, hidden):
    """The first: 264 MiB of tokens, four entries per wavefront and a rest of one, stored through the L2."""
    n, entries = 2, tokens * topk
    g = torch.Generator(device=DEV)
    g.manual_seed(topk)
    toks = [torch.randint(-2**31, 2**31 - 1, (tokens, hidden), device=DEV, dtype=torch.int32, generator=g) for _ in range(n)]
    dest = [torch.randint(0, n + 1, (entries,), device=DEV, dtype=torch.int32, generator=g) for _ in range(n)]   # n = dropped
    tabs, perm = route_on_gpu([d.cpu().numpy() for d in dest], n, entries, hidden)
    inbound = [sum(int((d == j).sum()) for d in dest) for j in range(n)]
    recv = [torch.full((r + 1, hidden), 7, device=DEV, dtype=torch.int32) for r in inbound]
    ptrs = lambda ts: [t.data_ptr() for t in ts]
    torch.cuda.synchronize()
    hcclx.moe_dispatch(ptrs(toks), ptrs(dest), ptrs(perm), entries, topk, hidden, T.FP32, tabs[1].data_ptr(), tabs[3].data_ptr(), ptrs(recv))
    torch.cuda.synchronize()
    for j in range(n):
        want = torch.cat([toks[i][(dest[i] == j).nonzero().reshape(-1) // topk] for i in range(n)])
        assert torch.equal(recv[j][:-1], want), j
        assert bool((recv[j][-1] == 7).all()), j


def test_dispatch_and_gather_combine_in_several_launches():
    """More work-items than one launch takes along x (2^32): 33000 tokens of two pieces, 4096 entries each, nearly all
    dropped; the entries kept lie at both ends and around the first launch's last token."""
    n, topk, tokens, width = 1, 4096, 33000, 512
    tok = torch.arange(tokens * width, device=DEV, dtype=torch.float32).reshape(tokens, width)
    dest = torch.full((tokens, topk), -1, device=DEV, dtype=torch.int32)
    perm = torch.full((tokens, topk), -1, device=DEV, dtype=torch.int32)
    kept = [(0, 0), (1, 4095), (32763, 17), (32764, 0), (32764, 4095), (32999, 2048)]
    for row, (t, e) in enumerate(kept):
        dest[t, e], perm[t, e] = 0, row
    zero = torch.zeros(1, device=DEV, dtype=torch.int64)
    recv = torch.full((len(kept) + 1, width), -1.0, device=DEV)
    out = torch.full((tokens + 1, width), -1.0, device=DEV)
    torch.cuda.synchronize()
    hcclx.moe_dispatch([tok.data_ptr()], [dest.data_ptr()], [perm.data_ptr()], tokens * topk, topk, width, T.FP32, zero.data_ptr(),
                       zero.data_ptr(), [recv.data_ptr()])
    torch.cuda.synchronize()
    rows = torch.tensor([t for t, _ in kept], device=DEV)
    assert torch.equal(recv[:-1], tok[rows]) and bool((recv[-1] == -1).all())
    hcclx.moe_gather_combine([recv.data_ptr()], [dest.data_ptr()], [perm.data_ptr()], tokens, topk, width, T.FP32, zero.data_ptr(),
                             zero.data_ptr(), [out.data_ptr()])
    torch.cuda.synchronize()
    want = torch.zeros_like(tok).index_add_(0, rows, tok[rows])
    assert torch.equal(out[:-1], want) and bool((out[-1] == -1).all())


@pytest.mark.parametrize("n,entries", [(1, 1), (8, 64), (8, 511), (8, 512), (4, 513), (64, 1024), (3, 1024), (3, 1025), (33, 257)])
@pytest.mark.parametrize("skew", [0, 1])
def test_route_in_one_launch(n, entries, skew):
    """Up to 1024 entries per rank: around whole chunks of 256, whole rounds of eight loads and the size from which two
    launches take over."""
    before = hcclx.kernels_launched()
    rng = np.random.default_rng(n + entries)
    dests = [rng.integers(-1, n + 1, size=entries) for _ in range(n)]
    tabs, perm = route_on_gpu(dests, n, entries, 8, skew)
    assert hcclx.kernels_launched() - before == (1 if entries <= 1024 else 2)
    sc, sd, rc, rd, perms = T.moe_route(dests, n, 8)
    for got, want in zip(tabs, (sc, sd, rc, rd)):
        assert np.array_equal(got.cpu().numpy().reshape(n, n), np.array(want, dtype=np.int64))
    for i in range(n):
        assert np.array_equal(perm[i].cpu().numpy().view(np.uint32), perms[i]), i


@pytest.mark.parametrize("n,entries", [(1, 1), (8, 512), (64, 1024), (5, 300), (3, 1025), (3, 20000)])
def test_route_with_perm_in_the_place_of_dest(n, entries):
    """A caller that only packs and combines needs no destinations afterwards: the histogram runs a launch before the
    permutation then, at every size."""
    rng = np.random.default_rng(n + entries)
    dests = [rng.integers(-1, n + 1, size=entries) for _ in range(n)]
    both = [dev_i32(x) for x in dests]
    tabs = [torch.full((n * n,), -1, dtype=torch.int64, device=DEV) for _ in range(4)]
    ws = torch.empty(hcclx.moe_workspace_bytes(n, entries), dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    before = hcclx.kernels_launched()
    hcclx.moe_route([b.data_ptr() for b in both], entries, 8, *[t.data_ptr() for t in tabs], [b.data_ptr() for b in both], ws.data_ptr())
    assert hcclx.kernels_launched() - before >= 2
    torch.cuda.synchronize()
    sc, sd, rc, rd, perms = T.moe_route(dests, n, 8)
    for got, want in zip(tabs, (sc, sd, rc, rd)):
        assert np.array_equal(got.cpu().numpy().reshape(n, n), np.array(want, dtype=np.int64))
    for i in range(n):
        assert np.array_equal(both[i].cpu().numpy().view(np.uint32), perms[i]), i


def test_the_scatter_knob_can_be_taken_back():
    """1 and 2 entries per wavefront, then chosen per launch again: the same rows; anything else is refused."""
    n, topk, tokens, width = 3, 4, 50, 512
    rng = np.random.default_rng(8)
    dests = [rng.integers(0, n, size=tokens * topk) for _ in range(n)]
    tabs, perm = route_on_gpu(dests, n, tokens * topk, width)
    dest = [dev_i32(d) for d in dests]
    tok = [torch.arange(tokens * width, device=DEV, dtype=torch.int32) + i * 1000003 for i in range(n)]
    ptrs = lambda ts: [t.data_ptr() for t in ts]
    got = []
    for value in (0, 1, 2, 0):
        hcclx.tune("moe_scatter_rows", value)
        recv = [torch.zeros(int(tabs[2].reshape(n, n)[j].sum()), device=DEV, dtype=torch.int32) for j in range(n)]
        torch.cuda.synchronize()
        hcclx.moe_dispatch(ptrs(tok), ptrs(dest), ptrs(perm), tokens * topk, topk, width, T.FP32, tabs[1].data_ptr(), tabs[3].data_ptr(), ptrs(recv))
        torch.cuda.synchronize()
        got.append(recv)
    for recv in got[1:]:
        assert all(torch.equal(a, b) for a, b in zip(got[0], recv))
    with pytest.raises(HcclError):
        hcclx.tune("moe_scatter_rows", 3)
