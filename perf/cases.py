"""The work that users of this package have it do, as cases that can be timed.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges.  ``prepare(case, seed)`` makes
what a program holds before the call (ranks as slices of one GPU arena, operands in the symmetric heap,
plan objects), ``run(state)`` is one pass through the public entry points and returns the outputs,
``work(case)`` what one pass cannot do without, and ``tolerance(case)`` how far another correct
implementation at the same precision may be off.

The kinds of case (``kind``) and what each stands for:

==================  ====================================================================================
allscatter          ``ops.gemm_allscatter`` as one rank calls it: full GEMM, its column block to every peer
gather_cols         ``GemmAllGatherPlan`` of every rank: a column-parallel linear layer whose output is
                    gathered; M = 1 .. 64 is decoding, M in the thousands is prefill or a training step
gather_rows         ``v2.FusedGemmAllGather`` (TileGroup launch, both directions of the exchange)
reduce_rows         ``v2.FusedGemmReduceScatter`` (both owners' reductions), 16-bit and fp8 inputs
reduce_cols         ``GemmReduceScatterPlan`` of one rank, its peers' partials resident: a row-parallel
                    linear layer
chained             ``AllGatherGemmReduceScatterPlan``: gather the input's column shards, multiply, scatter
allreduce           ``ops.allreduce`` of every rank: gradients or activations, from latency-bound up
allreduce_staged    ``primitives.allreduce_staged``: all ranks' roles in one launch, one gradient bucket
sharded_step        ``ops.reduce_scatter`` of the gradients and ``ops.allgather`` of the parameters on every
                    rank: the traffic of one bucket of a sharded optimiser
==================  ====================================================================================
"""

from __future__ import annotations

import math

import torch

import tileccl_amd
from tileccl_amd import ops, v2
from tileccl_amd.primitives import allreduce_staged

_DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32, "f8": torch.float8_e4m3fn}
_SIZES = {"f16": 2, "bf16": 2, "f32": 4, "f8": 1}
_GEMM_KINDS = ("allscatter", "gather_cols", "gather_rows", "reduce_rows", "reduce_cols", "chained")


def listed():
    return [
        # The smallest problem of the benchmark configurations: a call is launches and host work.
        {"name": "allscatter small", "kind": "allscatter", "M": 512, "N": 512, "K": 256, "world": 2, "dtype": "f16", "layout": "kn"},
        # One decoding step of a column-parallel layer: 16 rows, the weight held as (N, K).
        {"name": "gather cols decode", "kind": "gather_cols", "M": 16, "N": 4096, "K": 4096, "world": 2, "dtype": "bf16", "layout": "nk"},
        # The same layer over a long prompt or a training batch; the largest case.
        {"name": "gather cols prefill", "kind": "gather_cols", "M": 8192, "N": 8192, "K": 4096, "world": 2, "dtype": "bf16", "layout": "nk"},
        # The headline configuration: local 4096x1024 @ 1024x4096 fp16, gathered to 8192x4096.
        {"name": "gather rows", "kind": "gather_rows", "M": 4096, "N": 4096, "K": 1024, "world": 2, "dtype": "f16", "layout": "kn"},
        # The reduce-scatter configurations: fp16 with fp32 partials, and fp8 with bf16 partials.
        {"name": "reduce rows", "kind": "reduce_rows", "M": 8192, "N": 4096, "K": 2048, "world": 2, "dtype": "f16", "layout": "kn"},
        {"name": "reduce rows fp8", "kind": "reduce_rows", "M": 16384, "N": 4096, "K": 2048, "world": 2, "dtype": "f8", "layout": "kn"},
        # A row-parallel layer on four ranks over a short prompt.
        {"name": "reduce cols", "kind": "reduce_cols", "M": 1024, "N": 4096, "K": 2048, "world": 4, "dtype": "bf16", "layout": "kn"},
        # The chained benchmark: two shards of 1024 input columns.
        {"name": "chained", "kind": "chained", "M": 4096, "N": 4096, "K": 2048, "world": 2, "dtype": "f16", "layout": "kn"},
        # Nothing divides: rows, columns and an odd K, A a transposed view.
        {"name": "allscatter ragged", "kind": "allscatter", "M": 1000, "N": 2064, "K": 1003, "world": 2, "dtype": "bf16", "layout": "any"},
        # A small all-reduce on four ranks: launches and latency.
        {"name": "allreduce small", "kind": "allreduce", "elems": 65536, "world": 4, "dtype": "bf16"},
        # A gradient bucket of 64 MiB.
        {"name": "allreduce staged", "kind": "allreduce_staged", "elems": 1 << 25, "world": 2, "dtype": "f16"},
        # One bucket of a sharded optimiser on eight ranks, fp32.
        {"name": "sharded step", "kind": "sharded_step", "elems": 1 << 22, "world": 8, "dtype": "f32"},
    ]


def _spread(rng, lo, hi, step=1):
    """A multiple of ``step`` in [lo, hi], evenly spread over the logarithm."""
    value = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi // step, max(-(-lo // step), round(value / step))) * step


def draw(rng):
    largest = max(_cost(c) for c in listed())
    while True:
        case = _draw_one(rng)
        if _cost(case) <= largest:
            return case


def _draw_one(rng):
    kind = rng.choice(("allscatter", "gather_cols", "gather_rows", "reduce_rows", "reduce_cols", "chained",
                       "allreduce", "allreduce_staged", "sharded_step"))
    world = rng.choice((2, 2, 4, 8))
    half = rng.choice(("f16", "bf16"))
    if kind in ("allreduce", "allreduce_staged", "sharded_step"):
        top = {"allreduce": 1 << 24, "allreduce_staged": 1 << 25, "sharded_step": 1 << 24}[kind]
        dtype = "f32" if kind == "sharded_step" else rng.choice((half, half, "f32"))
        return {"kind": kind, "elems": _spread(rng, 8192, top, 8 * world), "world": world, "dtype": dtype}
    layout = rng.choice(("kn", "nk"))
    if kind == "allscatter":
        layout = rng.choice(("kn", "nk", "any"))
        k = _spread(rng, 64, 4096, 1 if layout == "any" else 8)
        return {"kind": kind, "M": _spread(rng, 16, 8192), "N": _spread(rng, 256, 8192, 8 * world), "K": k, "world": world,
                "dtype": half, "layout": layout}
    if kind == "gather_cols":
        return {"kind": kind, "M": _spread(rng, 1, 8192), "N": _spread(rng, 512, 8192, 8 * world), "K": _spread(rng, 256, 8192, 8),
                "world": world, "dtype": half, "layout": layout}
    if kind == "reduce_cols":
        m = _spread(rng, 1, 8192)
        if m > 128 and rng.random() < 0.7:  # prompts and batches are mostly padded to whole tiles
            m = -(-m // 128) * 128
        return {"kind": kind, "M": m, "N": _spread(rng, 512, 8192, 8 * world), "K": _spread(rng, 256, 8192, 8), "world": world,
                "dtype": half, "layout": layout}
    if kind == "gather_rows":
        return {"kind": kind, "M": _spread(rng, 128, 8192), "N": _spread(rng, 512, 8192, 8), "K": _spread(rng, 256, 4096, 8),
                "world": rng.choice((2, 2, 4)), "dtype": half, "layout": layout}
    if kind == "reduce_rows":
        world = rng.choice((2, 2, 4))
        dtype = rng.choice((half, "f8"))
        return {"kind": kind, "M": _spread(rng, 128 * world, 16384, 128 * world), "N": _spread(rng, 512, 8192, 16),
                "K": _spread(rng, 256, 4096, 16), "world": world, "dtype": dtype, "layout": layout}
    world = rng.choice((2, 2, 4))
    return {"kind": kind, "M": _spread(rng, 128, 8192), "N": _spread(rng, 512, 8192, 8), "K": _spread(rng, 512, 4096, 8 * world),
            "world": world, "dtype": half, "layout": "kn"}


# ---------------------------------------------------------------------------------------------- inputs
def _normal(gen, shape, dtype, std=1.0):
    x = torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32)
    return (x * std).to(dtype)


def _quantised(gen, shape, std):
    """e4m3 values and their per-tensor scale: one sigma is stored as 64, clipped to +-448."""
    x = torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32)
    return (x * 64).clamp(-448.0, 448.0).to(torch.float8_e4m3fn), std / 64


def _placed(heap, value):
    t = heap.allocate_tensor(tuple(value.shape), value.dtype)
    t.copy_(value)
    return t


def _weight(heap, value, layout):
    """B as the program holds it: (K, N), or the ``.t()`` view of an (N, K) weight."""
    return _placed(heap, value) if layout != "nk" else _placed(heap, value.t().contiguous()).t()


def _activations(heap, value, layout):
    return _placed(heap, value) if layout != "any" else _placed(heap, value.t().contiguous()).t()


def _heap_bytes(case):
    """One rank's slice: every tensor of the case, what its operation keeps beside them, and some room."""
    if case["kind"] in _GEMM_KINDS:
        M, N, K, w = case["M"], case["N"], case["K"], case["world"]
        need = 4 * M * N * (3 if case["kind"].startswith("reduce") else 1) + 2 * (w if case["kind"] == "gather_rows" else 1) * M * N
        need += 2 * (2 * M * K + K * N)
    else:
        need = 4 * case["elems"] * _SIZES[case["dtype"]]
    return need + (96 << 20)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    make = globals()["_prepare_" + case["kind"]]
    return make(case, gen)


def _prepare_allscatter(case, gen):
    M, N, K, dtype = case["M"], case["N"], case["K"], _DTYPES[case["dtype"]]
    ctxs = tileccl_amd.init_local(world_size=case["world"], heap_size=_heap_bytes(case))
    outputs = [c.zeros(M, N, dtype=dtype) for c in ctxs]
    heap = ctxs[0].require_heap()
    A = _activations(heap, _normal(gen, (M, K), dtype), case["layout"])
    B = _weight(heap, _normal(gen, (K, N), dtype, K**-0.5), case["layout"])
    return {"kind": case["kind"], "ctxs": ctxs, "A": A, "B": B, "C": outputs}


def _prepare_gather_cols(case, gen):
    M, N, K, world, dtype = case["M"], case["N"], case["K"], case["world"], _DTYPES[case["dtype"]]
    ctxs = tileccl_amd.init_local(world_size=world, heap_size=_heap_bytes(case))
    x = _normal(gen, (M, K), dtype)
    ranks = []
    for ctx in ctxs:
        heap = ctx.require_heap()
        C = ctx.zeros(M, N, dtype=dtype)
        A = _placed(heap, x)
        B = _weight(heap, _normal(gen, (K, N // world), dtype, K**-0.5), case["layout"])
        ranks.append((ops.build_gemm_allgather_plan(A, B, C, ctx=ctx), A, B, C))
    return {"kind": case["kind"], "ctxs": ctxs, "ranks": ranks}


def _prepare_gather_rows(case, gen):
    M, N, K, dtype = case["M"], case["N"], case["K"], _DTYPES[case["dtype"]]
    heaps = v2.SymmetricHeap.create_all(_heap_bytes(case), case["world"])
    gathers = [v2.FusedGemmAllGather(h, M, N, dtype, directions="both") for h in heaps]
    for r, op in enumerate(gathers):  # the peers' blocks are there, as they are once their launches have ended
        op.out.zero_()
        if r:
            op.local_block.copy_(_normal(gen, (M, N), dtype))
    A = _placed(heaps[0], _normal(gen, (M, K), dtype))
    B = _weight(heaps[0], _normal(gen, (K, N), dtype, K**-0.5), case["layout"])
    gathers[0].mark_peers_ready()
    return {"kind": case["kind"], "heaps": heaps, "op": gathers[0], "A": A, "B": B,
            "outs": [op.out for op in gathers]}


def _prepare_reduce_rows(case, gen):
    M, N, K = case["M"], case["N"], case["K"]
    fp8 = case["dtype"] == "f8"
    partial, out = (torch.bfloat16, torch.bfloat16) if fp8 else (torch.float32, _DTYPES[case["dtype"]])
    heaps = v2.SymmetricHeap.create_all(_heap_bytes(case), case["world"])
    reducers = [v2.FusedGemmReduceScatter(h, M, N, partial_dtype=partial, out_dtype=out, own_rows_in_registers=True) for h in heaps]
    for op in reducers[1:]:
        op.partial.copy_(_normal(gen, (M, N), partial))
    if fp8:
        (a, scale_a), (b, scale_b) = _quantised(gen, (M, K), 1.0), _quantised(gen, (K, N), K**-0.5)
    else:
        a, b = _normal(gen, (M, K), out), _normal(gen, (K, N), out, K**-0.5)
        scale_a = scale_b = 1.0
    reducers[0].mark_peers_ready()
    return {"kind": case["kind"], "heaps": heaps, "op": reducers[0], "A": _placed(heaps[0], a), "B": _weight(heaps[0], b, case["layout"]),
            "scales": (scale_a, scale_b), "outs": [op.out for op in reducers]}


def _prepare_reduce_cols(case, gen):
    M, N, K, world, dtype = case["M"], case["N"], case["K"], case["world"], _DTYPES[case["dtype"]]
    ctxs = tileccl_amd.init_local(world_size=world, heap_size=_heap_bytes(case))
    ranks = []
    for ctx in ctxs:
        heap = ctx.require_heap()
        C = ctx.zeros(M, N // world, dtype=dtype)
        A = _placed(heap, _normal(gen, (M, K), dtype))
        B = _weight(heap, _normal(gen, (K, N), dtype, K**-0.5), case["layout"])
        ranks.append((ops.build_gemm_reducescatter_plan(A, B, C, ctx=ctx), A, B, C))
    for plan, A, B, C in ranks[1:]:  # the peers' calls: their partials are there before this rank's
        plan.execute(A, B, C)
    return {"kind": case["kind"], "ctxs": ctxs, "rank": ranks[0]}


def _prepare_chained(case, gen):
    M, N, K, world, dtype = case["M"], case["N"], case["K"], case["world"], _DTYPES[case["dtype"]]
    ctxs = tileccl_amd.init_local(world_size=world, heap_size=_heap_bytes(case))
    shards, outputs = [], []
    for ctx in ctxs:
        shards.append(_placed(ctx.require_heap(), _normal(gen, (M, K // world), dtype)))
        outputs.append(ctx.zeros(M, N, dtype=dtype))
    W = _placed(ctxs[0].require_heap(), _normal(gen, (K, N), dtype, K**-0.5))
    plan = ops.build_allgather_gemm_reducescatter_plan(shards[0], W, outputs[0], ctx=ctxs[0])
    return {"kind": case["kind"], "ctxs": ctxs, "plan": plan, "shard": shards[0], "W": W, "outs": outputs}


def _prepare_allreduce(case, gen):
    ctxs = tileccl_amd.init_local(world_size=case["world"], heap_size=_heap_bytes(case))
    tensors = [_placed(c.require_heap(), _normal(gen, (case["elems"],), _DTYPES[case["dtype"]])) for c in ctxs]
    return {"kind": case["kind"], "ctxs": ctxs, "tensors": tensors}


def _prepare_allreduce_staged(case, gen):
    heaps = v2.SymmetricHeap.create_all(_heap_bytes(case), case["world"])
    return {"kind": case["kind"], "heaps": heaps,
            "tensors": [_placed(h, _normal(gen, (case["elems"],), _DTYPES[case["dtype"]])) for h in heaps]}


def _prepare_sharded_step(case, gen):
    elems, world, dtype = case["elems"], case["world"], _DTYPES[case["dtype"]]
    ctxs = tileccl_amd.init_local(world_size=world, heap_size=_heap_bytes(case))
    ranks = []
    for ctx in ctxs:
        heap = ctx.require_heap()
        gradient = _placed(heap, _normal(gen, (elems,), dtype))
        reduced = ctx.zeros(elems // world, dtype=dtype)
        shard = _placed(heap, _normal(gen, (elems // world,), dtype))
        parameters = ctx.zeros(elems, dtype=dtype)
        ranks.append((ops.build_reduce_scatter_plan(gradient, reduced, ctx=ctx), gradient, reduced,
                      ops.build_allgather_plan(shard, parameters, ctx=ctx), shard, parameters))
    return {"kind": case["kind"], "ctxs": ctxs, "ranks": ranks}


# ------------------------------------------------------------------------------------------- one pass
def run(state):
    kind = state["kind"]
    if kind == "allscatter":
        ops.gemm_allscatter(state["A"], state["B"], state["C"][0], ctx=state["ctxs"][0])
        return state["C"]
    if kind == "gather_cols":
        return [plan.execute(A, B, C) for plan, A, B, C in state["ranks"]]
    if kind == "gather_rows":
        state["op"](state["A"], state["B"])
        return state["outs"]
    if kind == "reduce_rows":
        state["op"](state["A"], state["B"], scale_a=state["scales"][0], scale_b=state["scales"][1])
        return state["outs"]
    if kind == "reduce_cols":
        plan, A, B, C = state["rank"]
        return plan.execute(A, B, C)
    if kind == "chained":
        state["plan"].execute(state["shard"], state["W"], state["outs"][0])
        return state["outs"]
    if kind == "allreduce":
        for ctx, t in zip(state["ctxs"], state["tensors"]):
            ops.allreduce(t, ctx=ctx)
        return state["tensors"]
    if kind == "allreduce_staged":
        allreduce_staged(state["tensors"], state["heaps"])
        return state["tensors"]
    outputs = []
    for scatter, gradient, reduced, _, _, _ in state["ranks"]:
        outputs.append(scatter.execute(gradient, reduced))
    for _, _, _, gather, shard, parameters in state["ranks"]:
        outputs.append(gather.execute(shard, parameters))
    return outputs


# ------------------------------------------------------------------------------- what a pass stands for
def work(case):
    """Each input read once and each output written once, on all ranks that the pass serves."""
    w, e = case["world"], _SIZES[case["dtype"]]
    kind = case["kind"]
    if kind not in _GEMM_KINDS:
        size = case["elems"] * e
        if kind == "sharded_step":  # gradients and shards read, shards and parameters written
            return {"bytes": w * size + size + size + w * size, "flops": (w - 1) * case["elems"]}
        return {"bytes": 2 * w * size, "flops": (w - 1) * case["elems"]}
    M, N, K = case["M"], case["N"], case["K"]
    flops = 2 * M * N * K
    operands = (M * K + K * N) * e
    if kind == "allscatter":  # the whole C here, this rank's column block at the peers
        return {"bytes": operands + M * N * e + (w - 1) * M * (N // w) * e, "flops": flops}
    if kind == "gather_cols":  # every rank reads the input and its weight; the full C on every rank
        return {"bytes": w * M * K * e + K * N * e + w * M * N * e, "flops": flops}
    if kind == "gather_rows":  # own block to every rank, the peers' blocks read and written here
        return {"bytes": operands + (w + 2 * (w - 1)) * M * N * e, "flops": flops}
    if kind == "reduce_rows":  # the peers' partials read, the sums written
        partial, out = (2, 2) if case["dtype"] == "f8" else (4, 2)
        return {"bytes": operands + (w - 1) * M * N * partial + M * N * out, "flops": flops + (w - 1) * M * N}
    if kind == "reduce_cols":  # the other ranks' blocks written as partials, the own columns reduced
        block = M * (N // w)
        return {"bytes": operands + (w - 1) * block * 4 + (w - 1) * block * 4 + block * e, "flops": flops + (w - 1) * block}
    # chained: the shards read, the gathered input and every rank's output written
    return {"bytes": 2 * M * K * e + K * N * e + w * M * N * e, "flops": flops}


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def tolerance(case):
    """fp16 and bf16 outputs are sums in fp32 rounded once: half a unit in the last place and the few
    values that another order of summation rounds the other way; fp32 sums differ in their last bits."""
    if case["dtype"] == "f32":
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": 1e-3, "max": 4e-3} if case["dtype"] == "f16" else {"rel": 6e-3, "max": 2e-2}
