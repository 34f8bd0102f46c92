"""The shapes of the wide chain kernel for launches with one destination (chosen by size, alignment and what is read):
whole and partial tiles of each, segments of unequal length, sources that share the destination's alignment and sources that
straddle it, against the same fold step by step in torch.  Bit-exact: the order is the same."""
import numpy as np
import pytest
import torch

from oracle import templates as T
from hccl_amd import hcclx

from gpu_util import TORCH_STORAGE, device_payload
from wide_shape_cases import CASES, segment_lengths

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


HALF = (T.FP16, T.BFP16)


def any_step(dtype, op, src, dst):
    """src (+) dst as the kernels combine: 16-bit floats in fp32 (sums narrowed once, at the end; products every time), max as
    (s < d) ? d : s, min as (d < s) ? d : s."""
    if op == T.MAX:
        return torch.where(src < dst, dst, src)
    if op == T.MIN:
        return torch.where(dst < src, dst, src)
    if op == T.PROD:
        return (src * dst).to(TORCH_STORAGE[dtype]).float() if dtype in HALF else src * dst
    return src + dst


def any_chain(xs, dtype, op, flips):
    wide = (lambda x: x.float()) if dtype in HALF else (lambda x: x)
    acc = wide(xs[0])
    for k in range(1, len(xs)):
        acc = any_step(dtype, op, acc, wide(xs[k])) if flips[k] else any_step(dtype, op, wide(xs[k]), acc)
    return acc.to(TORCH_STORAGE[dtype])


def assert_same(got, want):
    """Equal to the bit; NaNs where NaNs are."""
    if got.is_floating_point():
        bits = {2: torch.int16, 4: torch.int32, 8: torch.int64}[got.element_size()]
        assert torch.equal(got.isnan(), want.isnan())
        got, want = (torch.where(v.isnan(), torch.zeros_like(v), v).view(bits) for v in (got, want))
    assert torch.equal(got, want)


TYPES = {"int8": T.INT8, "int16": T.INT16, "int32": T.INT32, "int64": T.INT64, "fp16": T.FP16, "bf16": T.BFP16, "fp32": T.FP32, "fp64": T.FP64}
OPS = {"sum": T.SUM, "prod": T.PROD, "max": T.MAX, "min": T.MIN}


def run_case(dtype, op, nsrc, total, straddle, in_place=None):
    esz = T.DTYPE_SIZE[dtype]
    lengths = segment_lengths(esz, total, straddle)
    whole = sum(lengths)
    assert whole * esz == total
    off = [k % 2 if straddle else 0 for k in range(nsrc)]
    if in_place is not None:
        off[in_place] = 0
    xs = [device_payload(dtype, whole + 64, 10 * k + nsrc) for k in range(nsrc)]
    if op in (T.MAX, T.MIN) and xs[0].is_floating_point():   # values that they tell apart only by the order of the operands
        for k, x in enumerate(xs):
            x[k::7] = -0.0
            x[k + 1::7] = 0.0
            x[2 * k::5] = float("nan")
            x[3 * k::11] = float("-inf")
    flips = [op in (T.MAX, T.MIN) and xs[0].is_floating_point() and k % 3 == 1 for k in range(nsrc)]
    want = any_chain([x[o:o + whole] for x, o in zip(xs, off)], dtype, op, flips)
    out = xs[in_place] if in_place is not None else torch.full((whole + 64,), 77, device="cuda:0", dtype=TORCH_STORAGE[dtype])
    behind = out[whole:].clone()
    segs, at = [], 0
    for n in lengths:
        segs.append((n, [x.data_ptr() + (at + o) * esz for x, o in zip(xs, off)], [out.data_ptr() + at * esz], [int(f) for f in flips]))
        at += n
    torch.cuda.synchronize()
    hcclx.fold_wide(segs, dtype, op)
    torch.cuda.synchronize()
    assert_same(out[:whole], want)
    assert_same(out[whole:], behind)


@pytest.mark.parametrize("dtype,op,nsrc,total,straddle,shape", CASES)
def test_every_shape_of_a_chain(dtype, op, nsrc, total, straddle, shape):
    """The shape is what test_host_wide_shapes.py finds the rule to give for these launches."""
    run_case(TYPES[dtype], OPS[op], nsrc, total, straddle)


@pytest.mark.parametrize("dtype,op", [("fp32", "sum"), ("bf16", "max")])
def test_the_largest_chains_without_lds_of_their_own(dtype, op):
    """fold_lds_hold 0: they run in the next smaller shape; what was planned before keeps its kernel."""
    hcclx.tune("fold_lds_hold", 0)
    try:
        run_case(TYPES[dtype], OPS[op], 9, 144 * MIB, False)
    finally:
        hcclx.tune("fold_lds_hold", 1)


@pytest.mark.parametrize("place", ["first", "last"])
@pytest.mark.parametrize("dtype,op,nsrc,total,straddle,shape", [c for c in CASES if c[:2] == ("fp32", "min")])
def test_every_shape_of_a_chain_in_place(dtype, op, nsrc, total, straddle, shape, place):
    """The destination is one of the sources."""
    run_case(TYPES[dtype], OPS[op], nsrc, total, straddle, in_place=0 if place == "first" else nsrc - 1)


def nhr_like_tree(n):
    """The steps (dst, src) of a tree over n registers in which each round halves what is left: ceil(log2 n) levels."""
    steps, left = [], list(range(n))
    while len(left) > 1:
        half = (len(left) + 1) // 2
        steps += [(left[k], left[half + k]) for k in range(len(left) - half)]
        left = left[:half]
    return steps


@pytest.mark.parametrize("dtype,nsrc,mib", [(T.FP32, 17, 16), (T.FP32, 33, 15), (T.FP64, 20, 17), (T.BFP16, 32, 4), (T.BFP16, 33, 4),
                                            (T.FP16, 64, 1)])
def test_wide_tree_shapes(dtype, nsrc, mib):
    """Both shapes of the wide tree kernel (by size; the 16-bit floats by their number of leaves): partial tiles at both ends of
    unequal segments, against the same tree in torch."""
    esz = T.DTYPE_SIZE[dtype]
    whole = mib * MIB // esz
    edge = 512 * 16 // esz                    # elements of the larger tile
    lengths = [edge - 1, whole, edge + 1, 3]
    xs = [device_payload(dtype, sum(lengths) + 8, 100 * k + mib) for k in range(nsrc)]
    out = torch.full((sum(lengths) + 8,), 77, device="cuda:0", dtype=TORCH_STORAGE[dtype])
    torch.cuda.synchronize()
    steps = nhr_like_tree(nsrc)
    prog = [r for st in steps for r in st]
    segs, at = [], 1
    for n in lengths:
        segs.append((n, [x.data_ptr() + at * esz for x in xs], [out.data_ptr() + at * esz], prog))
        at += n
    hcclx.fold_wide(segs, dtype, T.SUM, hcclx.FOLD_TREE)
    torch.cuda.synchronize()
    val = [x.float() if esz == 2 else x.clone() for x in xs]
    for d, s in steps:
        val[d] = val[s] + val[d]
    want = val[0].to(TORCH_STORAGE[dtype])
    bits = {2: torch.int16, 4: torch.int32, 8: torch.int64}[esz]
    assert torch.equal(out[1:at].view(bits), want[1:at].view(bits))
    assert bool((out[at:] == 77).all()) and bool((out[:1] == 77).all())


@pytest.mark.parametrize("dtype", [T.FP16, T.BFP16])
@pytest.mark.parametrize("op", [T.SUM, T.PROD, T.MAX, T.MIN])
def test_wide_trees_of_16_bit_floats_over_all_values(dtype, op):
    """Both forms (whole vectors up to 32 leaves, pairs of elements above) over every bit pattern: infinities, NaNs, subnormals."""
    for nsrc in (24, 40):
        n = 65536 + 24
        xs = [torch.randint(-32768, 32768, (n,), device="cuda:0", dtype=torch.int16).view(TORCH_STORAGE[dtype]) for _ in range(nsrc)]
        for k, x in enumerate(xs[:4]):   # positions at which nothing is a NaN by chance
            x[k * 5000:(k + 1) * 5000] = float("inf") if k % 2 else float("-inf")
        for x in xs[4:]:
            x[:20000] = torch.randn(20000, device="cuda:0").to(x.dtype)
        out = torch.full((n,), 77, device="cuda:0", dtype=TORCH_STORAGE[dtype])
        torch.cuda.synchronize()
        steps = nhr_like_tree(nsrc)
        hcclx.fold_wide([(n, [x.data_ptr() for x in xs], [out.data_ptr()], [r for st in steps for r in st])], dtype, op, hcclx.FOLD_TREE)
        torch.cuda.synchronize()
        val = [x.float() for x in xs]
        for d, s in steps:
            val[d] = any_step(dtype, op, val[s], val[d])
        assert_same(out, val[0].to(TORCH_STORAGE[dtype]))


@pytest.mark.parametrize("nsrc,mib", [(12, 64), (16, 63)])
def test_tree_to_one_destination_with_fewer_workgroups(nsrc, mib):
    """Trees over more than eight slots: from 64 MiB on fewer workgroups share a CU, the tiles are the same."""
    n = mib * MIB // 4 + 5
    xs = [device_payload(T.FP32, n, k) for k in range(nsrc)]
    out = torch.zeros(n, device="cuda:0")
    torch.cuda.synchronize()
    steps = nhr_like_tree(nsrc)
    hcclx.fold([(n, [x.data_ptr() for x in xs], [out.data_ptr()], [r for st in steps for r in st])], T.FP32, T.SUM, hcclx.FOLD_TREE)
    torch.cuda.synchronize()
    for d, s in steps:
        xs[d] = xs[s] + xs[d]
    assert torch.equal(out.view(torch.int32), xs[0].view(torch.int32))


@pytest.mark.parametrize("nsrc", [9, 10, 16, 17, 18, 25, 33, 57, 64])
@pytest.mark.parametrize("ndst", [1, 3])
def test_chain_in_groups_of_sources(nsrc, ndst):
    """Small chains take eight sources at a time behind the first: last groups of one, of eight and in between, with the operands of
    every third step turned round."""
    n = 5003
    xs = [device_payload(T.FP32, n + 8, 100 + k) for k in range(nsrc)]
    for k, x in enumerate(xs):
        x[k::11] = -0.0
        x[k + 1::11] = 0.0
    flips = [k % 3 == 2 for k in range(nsrc)]
    outs = [torch.full((n + 8,), 77.0, device="cuda:0") for _ in range(ndst)]
    torch.cuda.synchronize()
    hcclx.fold_wide([(n, [x.data_ptr() + 4 for x in xs], [o.data_ptr() + 4 for o in outs], [int(f) for f in flips])], T.FP32, T.MAX)
    torch.cuda.synchronize()
    want = chain([x[1:n + 1] for x in xs], T.FP32, T.MAX, flips)
    for o in outs:
        assert torch.equal(o[1:n + 1].view(torch.int32), want.view(torch.int32))
        assert bool((o[n + 1:] == 77).all()) and bool((o[:1] == 77).all())
