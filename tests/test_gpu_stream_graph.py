"""Launches of the streaming kernel, and calls that pack their operands, recorded into a HIP graph: replays interleaved with
eager work and eager launches equal the eager bytes."""

import pytest
import torch

from tests.gpu_util import assert_gemm_close, bits, into_heap, seeded
from tests.test_gpu_stream_live import E4M3, TIGHT, operands, out_type, small_tiles_ran

pytestmark = pytest.mark.gpu


def record(call):
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    return graph


def eager_work():
    assert (torch.randn(256, 256, device="cuda") @ torch.randn(256, 256, device="cuda")).isfinite().all()


@pytest.mark.parametrize("variant", ["s0", "s1", "s2"])
@pytest.mark.parametrize("M,N,K,dtype", [(256, 1000, 520, torch.float16), (512, 512, 512, torch.bfloat16), (1536, 2048, 1024, E4M3)])
def test_all_gather(lib, M, N, K, dtype, variant):
    from tileccl_amd.v2 import FusedGemmAllGather, SymmetricHeap

    heaps = SymmetricHeap.create_all(192 << 20, 2)
    try:
        ops = [FusedGemmAllGather(h, M, N, out_type(dtype), directions="both") for h in heaps]
        op = ops[0]
        op.mark_peers_ready()
        each = [operands(heaps[0], M, N, K, dtype, 10 * i) for i in range(3)]
        alpha = each[0][3]
        A, B = heaps[0].allocate_tensor((M, K), dtype), heaps[0].allocate_tensor((K, N), dtype)

        def load(i):
            A.copy_(each[i][0])
            B.copy_(each[i][1])
            op.out.zero_()
            ops[1].out[:M].zero_()
            ops[1].out[M:].copy_(seeded((M, N), 50 + i, out_type(dtype)))

        def check(i):
            torch.cuda.synchronize()
            op.check_faults()
            assert_gemm_close(op.local_block, each[i][2], tight=TIGHT[out_type(dtype)])
            assert torch.equal(bits(op.out), bits(ops[1].out))
            assert not op.words.arrivals.any()
            return op.out.clone()

        load(0)
        op(A, B, variant, alpha)
        eager = check(0)
        graph = record(lambda: op(A, B, variant, alpha))
        for i in (1, 2, 0, 0):
            load(i)
            graph.replay()
            got = check(i)
            eager_work()
        assert torch.equal(bits(got), bits(eager))
        for i in (1, 0):
            load(i)
            op(A, B, variant, alpha)
            got = check(i)
        load(2)
        graph.replay()
        check(2)
        assert torch.equal(bits(got), bits(eager))
        if variant != "s0":
            assert small_tiles_ran(op, A, B, variant, alpha)
    finally:
        for h in heaps:
            h.cleanup()


@pytest.mark.parametrize("variant", ["s1", "s2"])
@pytest.mark.parametrize("M,N,K,dtype", [(512, 512, 512, torch.bfloat16), (2048, 512, 512, E4M3)])
def test_reduce_scatter(lib, M, N, K, dtype, variant):
    from tileccl_amd.v2 import FusedGemmReduceScatter, SymmetricHeap

    partial = torch.bfloat16 if dtype is E4M3 else torch.float32
    heaps = SymmetricHeap.create_all(192 << 20, 2)
    try:
        ops = [FusedGemmReduceScatter(h, M, N, partial_dtype=partial, out_dtype=out_type(dtype), own_rows_in_registers=True) for h in heaps]
        op = ops[0]
        op.mark_peers_ready()
        ops[1].partial.copy_(seeded((M, N), 9, partial))
        each = [operands(heaps[0], M, N, K, dtype, 10 * i) for i in range(2)]
        alpha = each[0][3]
        A, B = heaps[0].allocate_tensor((M, K), dtype), heaps[0].allocate_tensor((K, N), dtype)

        def outcome(i, call):
            A.copy_(each[i][0])
            B.copy_(each[i][1])
            for o in ops:
                o.out.zero_()
            call()
            torch.cuda.synchronize()
            op.check_faults()
            assert not op.words.arrivals.any()
            return torch.cat([bits(o.out) for o in ops])

        eager = [outcome(i, lambda: op(A, B, variant, alpha)) for i in range(2)]
        graph = record(lambda: op(A, B, variant, alpha))
        for i in (0, 1, 0):
            assert torch.equal(outcome(i, graph.replay), eager[i])
            eager_work()
        assert torch.equal(outcome(1, lambda: op(A, B, variant, alpha)), eager[1])
        assert torch.equal(outcome(0, graph.replay), eager[0])
    finally:
        for h in heaps:
            h.cleanup()


@pytest.mark.parametrize("warm", [False, True])
def test_packed_operands_of_a_recorded_call(lib, warm):
    """The dense copy that a recorded call reads is the graph's own: calls that drop the kept buffers, and tensors made from
    their memory, neither change a replay nor are changed by one."""
    import tileccl_amd as tileccl
    from tileccl_amd import _launch

    ctx = tileccl.init_local(world_size=1, heap_size=64 << 20)[0]
    try:
        M, N, K = 200, 264, 136

        def make(seed, n=N):
            A, B = seeded((M, K), seed), seeded((K, n), seed + 1, scale=K**-0.5)
            return into_heap(ctx.heap, A.t().contiguous()).t(), into_heap(ctx.heap, B), ctx.zeros(M, n, dtype=torch.float16), A.float() @ B.float()

        A, B, out, want = make(0)
        side = torch.cuda.Stream()
        call = lambda: tileccl.ops.gemm_allscatter(A, B, out, ctx=ctx, pattern="wg_specialized")  # noqa: E731
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(side):
            if warm:  # on the stream that is recorded, as torch advises: the kept buffer is this stream's
                call()
            torch.cuda.synchronize()
            with torch.cuda.graph(graph, stream=side):
                call()
            torch.cuda.synchronize()
            for k in range(1, 12):  # other shapes take the places of the kept buffers
                x = torch.zeros(M + k, K, dtype=torch.float16, device="cuda").t()
                _launch._pack([(x, K, M + k, "A")])
            guards = [torch.full((n,), 7.0, dtype=torch.float16, device="cuda") for n in [M * K] * 16]
            torch.cuda.synchronize()
            for _ in range(3):
                out.zero_()
                graph.replay()
                torch.cuda.synchronize()
                assert_gemm_close(out, want, tight=0.004)
                eager_work()
            assert all(bool((g == 7.0).all()) for g in guards)
    finally:
        ctx.heap.cleanup()
