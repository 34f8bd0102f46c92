"""The collectives whose speed is followed from change to change, called the way a program calls them: one call per
virtual rank on the program's communication stream, host tables converted once, buffers resident in HBM.

listed() names the cases, draw() makes more of the same kinds; prepare() builds what a program holds before the call
(buffers, tables, the communicator), run() is one collective (or one MoE exchange) and returns every output whole.
Communicators and the stream live as long as the process, as in a training or serving program, so that a case on new
buffers is a known communicator that meets new buffers."""
import math
import random

import torch

from hccl_amd import api, hcclx
from hccl_amd import types as T

DTYPES = {"fp32": (T.FP32, torch.float32, 4), "bf16": (T.BFP16, torch.bfloat16, 2), "fp16": (T.FP16, torch.float16, 2),
          "int32": (T.INT32, torch.int32, 4)}
OPS = {"sum": T.SUM, "prod": T.PROD, "max": T.MAX}

# what a drawn case moves at most (the largest listed one moves 25.8 GB)
DRAW_BYTES = 4 << 30


def listed():
    return [
        # a scalar-sized AllReduce (loss, gradient norm, found-inf flags): all latency
        {"name": "all_reduce_small", "kind": "all_reduce", "ranks": 8, "count": 1001, "dtype": "fp32", "op": "sum",
         "topology": "mesh"},
        # one gradient bucket of a data-parallel step (25 MiB, an odd number of elements)
        {"name": "all_reduce_bucket", "kind": "all_reduce", "ranks": 8, "count": 13107203, "dtype": "bf16", "op": "sum",
         "topology": "mesh"},
        # product over 12 ranks: twelve results in twelve orders (benchmark configuration 5)
        {"name": "all_reduce_prod", "kind": "all_reduce", "ranks": 12, "count": 16777216, "dtype": "fp32", "op": "prod",
         "topology": "clos"},
        # the largest of the 12-rank size sweep: 1 GiB per rank
        {"name": "all_reduce_largest", "kind": "all_reduce", "ranks": 12, "count": 268435456, "dtype": "int32", "op": "max",
         "topology": "clos"},
        # more than 16 ranks, log-step order (a tree per slice)
        {"name": "all_reduce_32_ranks", "kind": "all_reduce", "ranks": 32, "count": 4194304, "dtype": "fp32", "op": "sum",
         "topology": "clos"},
        # sharded gradients: the benchmark's own workload
        {"name": "reduce_scatter", "kind": "reduce_scatter", "ranks": 8, "count": 4194304, "dtype": "bf16", "op": "sum",
         "topology": "mesh"},
        # sharded weights gathered before use
        {"name": "all_gather", "kind": "all_gather", "ranks": 8, "count": 33554432, "dtype": "fp16"},
        # ragged shards (0 .. 8 Mi elements), most blocks at addresses that are only 2-byte aligned
        {"name": "all_gather_ragged", "kind": "all_gather_v", "ranks": 16, "most": 8388608, "dtype": "fp16"},
        # MoE token exchange with finished host tables: 8 ranks x 4096 tokens x hidden 7168
        {"name": "all_to_all_tokens", "kind": "all_to_all_v", "ranks": 8, "tokens": 4096, "hidden": 7168, "dtype": "bf16"},
        # many small blocks (heads against sequence among 32 ranks), an odd number of elements each
        {"name": "all_to_all_small", "kind": "all_to_all", "ranks": 32, "count": 2049, "dtype": "bf16"},
        # an MoE layer's exchange in prefill, both directions: routing tables, dispatch, combine of top-2
        {"name": "moe_prefill", "kind": "moe", "ranks": 8, "tokens": 4096, "topk": 2, "hidden": 7168, "dtype": "bf16"},
        # the same in decode: few tokens per rank, top-8
        {"name": "moe_decode", "kind": "moe", "ranks": 8, "tokens": 64, "topk": 8, "hidden": 7168, "dtype": "bf16"},
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["all_reduce"] * 4 + ["reduce_scatter", "all_gather", "all_gather_v", "all_to_all_v", "all_to_all",
                                            "moe", "moe"])
    c = {"kind": kind}
    if kind == "all_reduce":
        c["ranks"] = rng.choice([2, 4, 8, 8, 12, 16, 24, 32, 64])
        c["dtype"], c["op"] = rng.choice([("fp32", "sum"), ("bf16", "sum"), ("fp16", "sum"), ("fp32", "prod"),
                                          ("int32", "max"), ("fp32", "max")])
        c["topology"] = rng.choice(["mesh", "clos"])
        c["count"] = _log_int(rng, 1, DRAW_BYTES // (2 * c["ranks"] * DTYPES[c["dtype"]][2]))
    elif kind == "reduce_scatter":
        c["ranks"] = rng.choice([2, 4, 8, 8, 16, 32])
        c["dtype"], c["op"] = rng.choice([("bf16", "sum"), ("fp32", "sum"), ("fp16", "sum"), ("int32", "max")])
        c["topology"] = rng.choice(["mesh", "mesh", "clos"])
        c["count"] = _log_int(rng, 1, DRAW_BYTES // ((c["ranks"] + 1) * c["ranks"] * DTYPES[c["dtype"]][2]))
    elif kind in ("all_gather", "all_gather_v"):
        c["ranks"] = rng.choice([2, 4, 8, 8, 16, 32])
        c["dtype"] = rng.choice(["fp16", "bf16", "fp32"])
        most = DRAW_BYTES // ((c["ranks"] + 1) * c["ranks"] * DTYPES[c["dtype"]][2])
        c["most" if kind == "all_gather_v" else "count"] = _log_int(rng, 16, most)
    elif kind == "all_to_all_v":
        c["ranks"] = rng.choice([2, 4, 8, 8, 16, 32])
        c["hidden"] = rng.choice([64, 1024, 2880, 4096, 7168])
        c["tokens"] = _log_int(rng, 1, 4608)
        c["dtype"] = rng.choice(["bf16", "fp16", "fp32"])
    elif kind == "all_to_all":
        c["ranks"] = rng.choice([2, 4, 8, 16, 32])
        c["dtype"] = rng.choice(["bf16", "fp16", "fp32"])
        c["count"] = _log_int(rng, 1, DRAW_BYTES // (2 * c["ranks"] ** 2 * DTYPES[c["dtype"]][2]))
    else:
        c["ranks"] = rng.choice([2, 4, 8, 8, 16])
        c["topk"] = rng.choice([1, 2, 4, 8])
        c["hidden"] = rng.choice([1024, 2880, 4096, 7168])
        c["dtype"] = rng.choice(["bf16", "fp16", "fp32"])
        row = c["hidden"] * DTYPES[c["dtype"]][2]
        c["tokens"] = _log_int(rng, 1, min(4608, DRAW_BYTES // (2 * c["ranks"] * (c["topk"] + 1) * row)))
    return c


_stream = None
_worlds = {}


def _comm_stream():
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


def _world(case):
    """The program's communicator of that many ranks on that topology."""
    key = (case["ranks"], case.get("topology", "mesh"))
    if key not in _worlds:
        w = api.World(case["ranks"])
        if key[1] == "clos":
            w.set_topo(1, api.SHAPE_CLOS)
        _worlds[key] = w
    return _worlds[key]


def _values(gen, count, case):
    """Gradients, activations and weights are normal, factors lie around one, whole numbers take their whole range."""
    dtype = DTYPES[case["dtype"]][1]
    if case["dtype"] == "int32":
        return torch.randint(-2**31, 2**31 - 1, (count,), device="cuda", generator=gen, dtype=torch.int32)
    if case.get("op") == "prod":
        return torch.rand(count, device="cuda", generator=gen) * 0.2 + 0.9
    return torch.randn(count, device="cuda", generator=gen, dtype=dtype)


def _zipf(ranks):
    """How tokens fall on ranks: Zipf with exponent 1.2."""
    return (torch.arange(1, ranks + 1, dtype=torch.float64) ** -1.2).cuda()


def _ragged(case):
    """The shard sizes of a ragged gather, uniform up to the largest; which rank holds which comes from the seed."""
    rng = random.Random(case["most"] * 64 + case["ranks"])
    return [rng.randint(0, case["most"]) for _ in range(case["ranks"])]


def _excl(row):
    out, at = [], 0
    for x in row:
        out.append(at)
        at += x
    return out


def _ptrs(tensors):
    return [t.data_ptr() for t in tensors]


def _arena(empty, sizes):
    """One buffer for what all ranks receive (how much each gets is the routing's matter, the sum is not) and its parts."""
    whole = empty(sum(sizes))
    return whole, [whole[at:at + size] for at, size in zip(_excl(sizes), sizes)]


def prepare(case, seed):
    n = case["ranks"]
    hccl, dtype, _ = DTYPES[case["dtype"]]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    s = {"case": case, "dtype": hccl, "stream": _comm_stream().cuda_stream}
    empty = lambda count: torch.zeros(max(1, count), device="cuda", dtype=dtype)[:count]  # noqa: E731
    kind = case["kind"]
    if kind != "moe":
        s["world"] = _world(case)
    if kind == "all_reduce":
        send = [_values(gen, case["count"], case) for _ in range(n)]
        recv = [empty(case["count"]) for _ in range(n)]
    elif kind == "reduce_scatter":
        send = [_values(gen, n * case["count"], case) for _ in range(n)]
        recv = [empty(case["count"]) for _ in range(n)]
    elif kind == "all_gather":
        send = [_values(gen, case["count"], case) for _ in range(n)]
        recv = [empty(n * case["count"]) for _ in range(n)]
    elif kind == "all_gather_v":
        sizes = _ragged(case)
        counts = [sizes[i] for i in torch.randperm(n, device="cuda", generator=gen).tolist()]
        s["counts"], s["tables"] = counts, (api.u64_table(counts), api.u64_table(_excl(counts)))
        send = [_values(gen, max(1, c), case) for c in counts]
        recv = [empty(sum(counts)) for _ in range(n)]
    elif kind == "all_to_all_v":
        dest = torch.multinomial(_zipf(n).expand(n, n), case["tokens"], replacement=True, generator=gen)
        matrix = [[int(x) * case["hidden"] for x in torch.bincount(d, minlength=n).tolist()] for d in dest]
        columns = [[matrix[i][j] for i in range(n)] for j in range(n)]
        s["tables"] = [[api.u64_table(t) for t in (matrix[r], _excl(matrix[r]), columns[r], _excl(columns[r]))]
                       for r in range(n)]
        send = [_values(gen, case["tokens"] * case["hidden"], case) for _ in range(n)]
        s["arrived"], recv = _arena(empty, [sum(c) for c in columns])
    elif kind == "all_to_all":
        send = [_values(gen, n * case["count"], case) for _ in range(n)]
        recv = [empty(n * case["count"]) for _ in range(n)]
    else:
        entries = case["tokens"] * case["topk"]
        dest = torch.multinomial(_zipf(n).expand(n, n), entries, replacement=True, generator=gen)
        landed = torch.stack([torch.bincount(d, minlength=n) for d in dest]).sum(0).tolist()
        send = [_values(gen, case["tokens"] * case["hidden"], case) for _ in range(n)]
        s["arrived"], recv = _arena(empty, [rows * case["hidden"] for rows in landed])
        s["entries"] = entries
        s["dest"] = [d.to(torch.int32) for d in dest]
        s["perm"] = [torch.zeros(entries, device="cuda", dtype=torch.int32) for _ in range(n)]
        s["out"] = [empty(case["tokens"] * case["hidden"]) for _ in range(n)]
        s["counts"] = [torch.zeros(n * n, device="cuda", dtype=torch.int64) for _ in range(4)]
        s["workspace"] = torch.zeros(hcclx.moe_workspace_bytes(n, entries), device="cuda", dtype=torch.uint8)
        s["dest_ptrs"], s["perm_ptrs"], s["out_ptrs"] = _ptrs(s["dest"]), _ptrs(s["perm"]), _ptrs(s["out"])
        s["count_ptrs"] = _ptrs(s["counts"])
    s["send"], s["recv"] = send, recv
    # a rank that receives nothing still passes a buffer
    s["send_ptrs"] = _ptrs(send)
    s["recv_ptrs"] = [t.data_ptr() or t.untyped_storage().data_ptr() for t in recv]
    _comm_stream().wait_stream(torch.cuda.current_stream())
    return s


def run(s):
    case, dtype, stream, send, recv = s["case"], s["dtype"], s["stream"], s["send_ptrs"], s["recv_ptrs"]
    kind, n = case["kind"], case["ranks"]
    if kind == "moe":
        send_counts, sdispls, recv_counts, rdispls = s["count_ptrs"]
        hidden, topk = case["hidden"], case["topk"]
        hcclx.moe_route(s["dest_ptrs"], s["entries"], hidden, send_counts, sdispls, recv_counts, rdispls, s["perm_ptrs"],
                        s["workspace"].data_ptr(), stream=stream)
        hcclx.moe_dispatch(send, s["dest_ptrs"], s["perm_ptrs"], s["entries"], topk, hidden, dtype, sdispls, rdispls, recv,
                           stream=stream)
        # the experts would work here, in place, on the rows that arrived
        hcclx.moe_gather_combine(recv, s["dest_ptrs"], s["perm_ptrs"], case["tokens"], topk, hidden, dtype, sdispls, rdispls,
                                 s["out_ptrs"], stream=stream)
        return {"arrived": s["arrived"], "out": s["out"], "tables": s["counts"], "perm": s["perm"]}
    w, ranks = s["world"], range(n)
    if kind == "all_reduce":
        count, op = case["count"], OPS[case["op"]]
        for r in ranks:
            api.check(w.all_reduce(r, send[r], recv[r], count, dtype, op, stream))
    elif kind == "reduce_scatter":
        count, op = case["count"], OPS[case["op"]]
        for r in ranks:
            api.check(w.reduce_scatter(r, send[r], recv[r], count, dtype, op, stream))
    elif kind == "all_gather":
        count = case["count"]
        for r in ranks:
            api.check(w.all_gather(r, send[r], recv[r], count, dtype, stream))
    elif kind == "all_gather_v":
        counts, (table, displs) = s["counts"], s["tables"]
        for r in ranks:
            api.check(w.all_gather_v(r, send[r], counts[r], recv[r], table, displs, dtype, stream))
    elif kind == "all_to_all_v":
        for r in ranks:
            sc, sd, rc, rd = s["tables"][r]
            api.check(w.all_to_all_v(r, send[r], sc, sd, recv[r], rc, rd, dtype, stream))
        return s["arrived"]
    else:
        count = case["count"]
        for r in ranks:
            api.check(w.all_to_all(r, send[r], count, recv[r], dtype, stream))
    return s["recv"]


def work(case):
    """Every input byte read once, every output byte written once; one operation per element and source folded in."""
    n, size = case["ranks"], DTYPES[case["dtype"]][2]
    kind = case["kind"]
    if kind == "all_reduce":
        return {"bytes": 2 * n * case["count"] * size, "flops": (n - 1) * case["count"]}
    if kind == "reduce_scatter":
        return {"bytes": (n + 1) * n * case["count"] * size, "flops": (n - 1) * n * case["count"]}
    if kind == "all_gather":
        return {"bytes": (n + 1) * n * case["count"] * size, "flops": 0}
    if kind == "all_gather_v":
        return {"bytes": (n + 1) * sum(_ragged(case)) * size, "flops": 0}
    if kind == "all_to_all_v":
        return {"bytes": 2 * n * case["tokens"] * case["hidden"] * size, "flops": 0}
    if kind == "all_to_all":
        return {"bytes": 2 * n * n * case["count"] * size, "flops": 0}
    rows = n * case["tokens"]
    # tokens read, rows written where they arrive, read from there, results written; the destinations
    return {"bytes": (2 * rows + 2 * rows * case["topk"]) * case["hidden"] * size + rows * case["topk"] * 4,
            "flops": rows * (case["topk"] - 1) * case["hidden"]}


def tolerance(case):
    """Copies, maxima and whole numbers: the same bits.  Sums and products: four times what folding the same values in
    the opposite order in fp32 differs by among 64 ranks (fp32: 2.9e-7, at most 1.5e-6 of a value; a 16-bit result
    rounded once: one rounding, 1.8e-3 for bf16 and 2.3e-4 for fp16, at most one unit in the last place)."""
    kind = case["kind"]
    folds = kind in ("all_reduce", "reduce_scatter") and case["op"] != "max"
    if not folds and not (kind == "moe" and case["topk"] > 1):
        return "exact"
    return {"fp32": {"rel": 1.2e-6, "max": 6e-6}, "fp16": {"rel": 9e-4, "max": 2e-3}, "bf16": {"rel": 7e-3, "max": 1.6e-2},
            "int32": "exact"}[case["dtype"]]
