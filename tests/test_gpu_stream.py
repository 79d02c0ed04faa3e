"""The streaming GEMM for small outputs: every tile shape at its edges (one row, rows and columns that end inside
a tile, K that ends inside a 64-element block), alone and inside the fused operations.  References: fp32 products on
the CPU; what is moved or reduced, byte for byte against the oracle."""

import ctypes as C

import pytest
import torch

from oracle import collectives as oracle
from tests.gpu_util import assert_gemm_close, bits, into_heap, seeded

pytestmark = pytest.mark.gpu

# M, N, K: shapes that the cost rule gives the tiles 16x16, 16x16, 16x16, 16x32, 32x32, 32x64 and 64x64
SHAPES = [(1, 24, 8), (17, 1000, 520), (33, 264, 1096), (100, 1032, 2008), (190, 1000, 1000), (250, 2000, 456), (1000, 1000, 200)]


def weight(heap, B, layout):
    return into_heap(heap, B) if layout == "kn" else into_heap(heap, B.t().contiguous()).t()


@pytest.mark.parametrize("layout", ["kn", "nk"])
@pytest.mark.parametrize("dtype,out", [(torch.float16, torch.float16), (torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_gemm_alone(lib, M, N, K, dtype, out, layout):
    from tileccl_amd import _launch, _lib
    from tileccl_amd.v2 import SymmetricHeap

    with SymmetricHeap.create_all(64 << 20, 1)[0] as heap:
        A, B = seeded((M, K), 1, dtype), seeded((K, N), 2, dtype, scale=K**-0.5)
        got = torch.full((M + 1, N), 7.0, dtype=out, device="cuda")  # one row more: nothing lands beyond M
        d = _launch.gemm_desc(into_heap(heap, A), weight(heap, B, layout), got[:M], alpha=0.5)
        _lib.check(lib.tccl_gemm(C.byref(d), _launch.stream_ptr()), "tccl_gemm")
        torch.cuda.synchronize()
        tight = {torch.float16: 0.004, torch.bfloat16: 0.032, torch.float32: 1e-3}[out]
        assert_gemm_close(got[:M], 0.5 * (A.float() @ B.float()), tight=tight)
        assert bool((got[M] == 7.0).all())


@pytest.mark.parametrize("layout", ["kn", "nk"])
@pytest.mark.parametrize("M,N,K", [(1, 16, 16), (17, 1008, 528), (100, 1040, 2000), (190, 1008, 1008), (250, 2000, 464), (1000, 1040, 208),
                                   (1500, 2000, 400)])
def test_gemm_alone_e4m3(lib, M, N, K, layout):
    """The same shapes with e4m3 inputs (128 k per block), the last one in two 64 x 64 tiles per CU."""
    from tileccl_amd import _launch, _lib
    from tileccl_amd.v2 import SymmetricHeap

    with SymmetricHeap.create_all(64 << 20, 1)[0] as heap:
        A, B = (seeded(s, k, torch.float32, scale=64.0).clamp(-448, 448).to(torch.float8_e4m3fn) for s, k in (((M, K), 1), ((K, N), 2)))
        got = torch.full((M + 1, N), 7.0, dtype=torch.float32, device="cuda")
        d = _launch.gemm_desc(into_heap(heap, A), weight(heap, B, layout), got[:M], alpha=K**-0.5 / 4096)
        _lib.check(lib.tccl_gemm(C.byref(d), _launch.stream_ptr()), "tccl_gemm")
        torch.cuda.synchronize()
        assert_gemm_close(got[:M], (A.float() @ B.float()) * (K**-0.5 / 4096), tight=1e-3)
        assert bool((got[M] == 7.0).all())


@pytest.mark.parametrize("variant", ["s1", "s2"])
@pytest.mark.parametrize("world,layout", [(2, "kn"), (3, "nk")])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_all_gather_pushes_pulls_and_publishes(lib, M, N, K, world, layout, variant):
    """Three launches in a row: the arrival counters start over by themselves and the published words reach every launch's
    number.  The peers are resident: their words are preset and they launch nothing.  (Waits for words that another launch
    writes: ``test_gpu_stream_live.py``.)"""
    from tileccl_amd.v2 import FusedGemmAllGather, SymmetricHeap

    heaps = SymmetricHeap.create_all(128 << 20, world)
    try:
        ops = [FusedGemmAllGather(h, M, N, torch.float16, directions="both", tau_min_bytes=1) for h in heaps]
        puller = ops[1]
        blocks = {p: seeded((M, N), 50 + p) for p in range(1, world)}
        for launch in range(3):
            for p, op in enumerate(ops):
                op.out.zero_()
                if p:
                    op.local_block.copy_(blocks[p])
            A, B = seeded((M, K), 3 * launch), seeded((K, N), 3 * launch + 1, scale=K**-0.5)
            for peer in range(1, world):
                for words in (ops[0].signals.counter, ops[0].locks):
                    heaps[0].peer_view(words, peer).fill_(1 << 30)
            ops[0](into_heap(heaps[0], A), weight(heaps[0], B, layout), variant)
            ops[0].check_faults()
            assert_gemm_close(ops[0].local_block, A.float() @ B.float(), tight=0.004)
            for p in range(1, world):
                assert torch.equal(bits(ops[p].out[:M]), bits(ops[0].local_block))
                assert torch.equal(bits(ops[0].out[p * M:(p + 1) * M]).cpu(), bits(blocks[p]))
            n = ops[0].words.epoch if variant == "s2" else ops[0].words.lock_epoch
            assert n == launch + 1
            if variant == "s2":
                assert ops[0].signals.counter.tolist() == [n * t for t in ops[0].plan.tile_counts()]
            else:
                assert ops[0].locks.tolist() == [n] * ops[0].locks.numel()
            assert not ops[0].words.arrivals.any()
        assert puller.words.epoch == 0
    finally:
        for h in heaps:
            h.cleanup()


@pytest.mark.parametrize("own,emulate,partial", [(True, True, torch.float32), (False, False, torch.float32), (True, False, torch.float16)])
@pytest.mark.parametrize("M,N,K", [(256, 104, 72), (256, 1000, 520), (512, 520, 1000), (768, 776, 200)])
def test_reduce_scatter_rows(lib, M, N, K, own, emulate, partial):
    from tileccl_amd.v2 import FusedGemmReduceScatter, SymmetricHeap

    heaps = SymmetricHeap.create_all(64 << 20, 2)
    try:
        ops = [FusedGemmReduceScatter(h, M, N, partial_dtype=partial, emulate_peer=emulate, own_rows_in_registers=own) for h in heaps]
        peer = seeded((M, N), 9, partial)
        ops[1].partial.copy_(peer)
        ops[0].mark_peers_ready()
        A, B = seeded((M, K), 3), seeded((K, N), 4, scale=K**-0.5)
        for _ in range(2):
            for op in ops:
                op.out.zero_()
            ops[0].partial.zero_()
            ops[0](into_heap(heaps[0], A), into_heap(heaps[0], B))
            ops[0].check_faults()
            mine = A.float() @ B.float()
            for owner in ((0, 1) if emulate else (0,)):
                want = oracle.reduce_rows([mine.to(partial), peer], owner, torch.float16)
                assert_gemm_close(ops[owner].out, want.float(), tight=0.008)
            stored = ops[0].partial.cpu().float()
            assert_gemm_close(stored[M // 2:], mine[M // 2:], tight=0.004)  # the other owner's rows
            assert bool((stored[:M // 2] == 0).all()) == own
            if not emulate:
                assert not ops[1].out.any()
            assert not ops[0].words.arrivals.any()
    finally:
        for h in heaps:
            h.cleanup()


@pytest.mark.parametrize("world,M,N,K", [(2, 1, 512, 264), (4, 62, 1088, 1032), (8, 5, 2048, 520), (3, 200, 504, 104), (2, 1500, 4096, 64)])
@pytest.mark.parametrize("layout", ["kn", "nk"])
def test_reduce_scatter_columns_of_any_row_count(lib, world, M, N, K, layout):
    """Row counts that are no whole plan tiles: one launch (the last shape: a GEMM per column block)."""
    import tileccl_amd as tileccl

    ctxs = tileccl.init_local(world_size=world, heap_size=96 << 20)
    try:
        A = [seeded((M, K), 10 + r) for r in range(world)]
        B = [seeded((K, N), 20 + r, scale=K**-0.5) for r in range(world)]
        Cs = [c.zeros(M, N // world, dtype=torch.float16) for c in ctxs]
        for _ in range(2):  # the second round finds every peer's partials
            for r, c in enumerate(ctxs):
                tileccl.ops.gemm_reducescatter(into_heap(c.heap, A[r]), weight(c.heap, B[r], layout), Cs[r], ctx=c)
        torch.cuda.synchronize()
        total = sum(a.float() @ b.float() for a, b in zip(A, B))
        for r in range(world):
            assert_gemm_close(Cs[r], total[:, r * (N // world):(r + 1) * (N // world)], tight=0.016)
    finally:
        for c in ctxs:
            c.heap.cleanup()


@pytest.mark.parametrize("variant", ["s1", "s2"])
def test_counts_of_overlapping_launches_stay_apart(lib, variant):
    """Launches that overlap share the arrival words.  What stands in those that other launches count in (here beyond what any
    plan tile has: counted into, they would never publish) neither disturbs a launch nor is touched by it."""
    from tileccl_amd import _lib
    from tileccl_amd.v2 import FusedGemmAllGather, SymmetricHeap

    M, N, K = 200, 600, 256
    with SymmetricHeap.create_all(64 << 20, 1)[0] as heap:
        op = FusedGemmAllGather(heap, M, N, torch.float16, directions="push", tau_min_bytes=1)
        A, B = into_heap(heap, seeded((M, K), 1)), into_heap(heap, seeded((K, N), 2, scale=K**-0.5))
        half = _lib.ARRIVAL_STRIDE // 2
        for launch in range(1, 2 * half + 2):
            words = op.words.arrivals.view(-1, _lib.ARRIVAL_STRIDE)
            words.fill_(1 << 30)
            words[:, launch % half + (half if variant == "s1" else 0)] = 0
            before = words.clone()
            op(A, B, variant)
            op.check_faults()
            assert torch.equal(words, before)
            if variant == "s2":
                assert op.signals.counter.tolist() == [launch * t for t in op.plan.tile_counts()]
            else:
                assert op.locks.tolist() == [launch] * op.locks.numel()


def test_launches_of_different_tiles_on_two_streams_leave_no_counts(lib):
    """One context's tile-by-tile calls share their words by the number of plan tiles: 16 here, of 16 tiles each in one
    call and of 8 in the other."""
    import tileccl_amd as tileccl

    ctx = tileccl.init_local(world_size=1, heap_size=64 << 20)[0]
    try:
        K = 1024
        calls = []
        for M, N, stream in ((512, 512, torch.cuda.Stream()), (1, 2048, torch.cuda.Stream())):
            A, B = seeded((M, K), M), seeded((K, N), N, scale=K**-0.5)
            calls.append((into_heap(ctx.heap, A), into_heap(ctx.heap, B), ctx.zeros(M, N, dtype=torch.float16), A.float() @ B.float(), stream))
        torch.cuda.synchronize()
        for _ in range(30):
            for A, B, C_out, _, stream in calls:
                with torch.cuda.stream(stream):
                    tileccl.ops.gemm_allscatter(A, B, C_out, ctx=ctx, pattern="wg_specialized")
        torch.cuda.synchronize()
        for _, _, C_out, want, _ in calls:
            assert_gemm_close(C_out, want, tight=0.004)
        words = [w for k, w in ctx._workspace_cache.items() if "locks" in k]
        assert len(words) == 1 and words[0].lock_epoch == 60 and not words[0].arrivals.any()
    finally:
        ctx.heap.cleanup()


@pytest.mark.parametrize("pattern", ["wg_specialized", "tile_group"])
def test_words_made_on_a_busy_stream_are_clear_for_another(lib, pattern):
    """The first call of a shape makes its words, on a stream that is still at work; the next call comes on another one.  The
    memory that the words are made in is not clear by itself."""
    import tileccl_amd as tileccl
    from tileccl_amd import _lib

    ctx = tileccl.init_local(world_size=1, heap_size=64 << 20)[0]
    try:
        M, N, K = 300, 520, 264
        A, B = seeded((M, K), 1), seeded((K, N), 2, scale=K**-0.5)
        a, b, outs = into_heap(ctx.heap, A), into_heap(ctx.heap, B), [ctx.zeros(M, N, dtype=torch.float16) for _ in range(2)]
        ctx.heap.get_peer_buffer(0)[ctx.heap.bytes_allocated:].fill_(5)
        busy, other = torch.cuda.Stream(), torch.cuda.Stream()
        big = torch.randn(4096, 4096, device="cuda", dtype=torch.float16)
        torch.cuda.synchronize()
        tiles = 3 * 5
        with torch.cuda.stream(busy):
            dirty = [torch.full((tiles * _lib.ARRIVAL_STRIDE,), 5, dtype=torch.int32, device="cuda") for _ in range(4)]
            del dirty
            for _ in range(200):  # some 20 ms
                big @ big
            tileccl.ops.gemm_allscatter(a, b, outs[0], ctx=ctx, pattern=pattern)
        with torch.cuda.stream(other):
            tileccl.ops.gemm_allscatter(a, b, outs[1], ctx=ctx, pattern=pattern)
            (words,) = [w for k, w in ctx._workspace_cache.items() if isinstance(k, tuple) and k[0] == "tileccl_amd.sync"]
            assert not words.arrivals.any()
            other.synchronize()
            assert_gemm_close(outs[1], A.float() @ B.float(), tight=0.004)
        torch.cuda.synchronize()
        assert_gemm_close(outs[0], A.float() @ B.float(), tight=0.004)
        assert not words.arrivals.any()
        if pattern == "wg_specialized":
            assert set(words.locks.tolist()) <= {1, 2}
        else:
            assert words.counter.tolist() == [2 * t for t in words.host_plan.tile_counts()]
    finally:
        ctx.heap.cleanup()
