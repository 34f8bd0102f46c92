"""The shapes of the wide chain kernel for launches with one destination (small, one, large; chosen by size and alignment):
whole and partial tiles of each, segments of unequal length, sources that share the destination's alignment and sources that
straddle it, against the same fold step by step in torch.  Bit-exact: the order is the same."""
import numpy as np
import pytest
import torch

from oracle import templates as T
from hccl_amd import hcclx

from gpu_util import TORCH_STORAGE, device_payload

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def step(dtype, op, src, dst):
    """src (+) dst as the kernels combine: sums in fp32 for bf16 (narrowed once, at the end), max as (s < d) ? d : s."""
    return torch.where(src < dst, dst, src) if op == T.MAX else src + dst


def chain(xs, dtype, op, flips):
    wide = (lambda x: x.float()) if dtype == T.BFP16 else (lambda x: x)
    acc = wide(xs[0])
    for k in range(1, len(xs)):
        acc = step(dtype, op, acc, wide(xs[k])) if flips[k] else step(dtype, op, wide(xs[k]), acc)
    return acc.to(TORCH_STORAGE[dtype])


@pytest.mark.parametrize("dtype,op", [(T.FP32, T.SUM), (T.BFP16, T.SUM), (T.INT32, T.MAX), (T.FP32, T.MAX)])
@pytest.mark.parametrize("nsrc,mib,straddle", [(5, 4, True), (17, 8, False), (9, 31, True), (5, 33, True), (8, 127, False),
                                               (5, 128, False), (5, 129, True)])
def test_chain_to_one_destination(nsrc, mib, straddle, dtype, op):
    esz = T.DTYPE_SIZE[dtype]
    edge = 65536 // esz                       # elements of the largest tile
    whole = mib * MIB // esz
    lengths = [edge - 1, whole - 3 * edge - 7, 1, 2 * edge + 3] if straddle else [edge, whole - 2 * edge, edge - 16 // esz]
    total = sum(lengths) + 64
    xs = [device_payload(dtype, total + k, 10 * k + mib) for k in range(nsrc)]
    if op == T.MAX and dtype == T.FP32:       # values that max tells apart only by the order of its operands
        for k, x in enumerate(xs):
            x[k::7] = -0.0
            x[k + 1::7] = 0.0
            x[2 * k::5] = float("nan")
    flips = [op == T.MAX and dtype == T.FP32 and k % 3 == 1 for k in range(nsrc)]
    out = torch.full((total,), 77, device="cuda:0", dtype=TORCH_STORAGE[dtype])
    torch.cuda.synchronize()
    segs, at = [], 0
    for n in lengths:
        srcs = [x.data_ptr() + (at + (k % 3 if straddle else 0)) * esz for k, x in enumerate(xs)]
        segs.append((n, srcs, [out.data_ptr() + at * esz], [int(f) for f in flips]))
        at += n
    before = hcclx.kernels_launched()
    hcclx.fold_wide(segs, dtype, op)
    assert hcclx.kernels_launched() == before + 1
    torch.cuda.synchronize()
    want = chain([x[k % 3 if straddle else 0:][:at] for k, x in enumerate(xs)], dtype, op, flips)
    got = out[:at]
    if dtype == T.BFP16:
        got, want = got.view(torch.int16), want.view(torch.int16)
    elif dtype == T.FP32:
        assert torch.equal(got.isnan(), want.isnan())
        got, want = (torch.where(v.isnan(), torch.zeros_like(v), v).view(torch.int32) for v in (got, want))
    assert torch.equal(got, want)
    assert bool((out[at:] == 77).all())
