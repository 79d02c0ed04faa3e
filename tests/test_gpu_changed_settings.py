"""What is set on an operation between two calls holds from the next call on, whatever the calls before it have kept."""

import pytest
import torch

from tests.gpu_util import assert_gemm_close, bits, into_heap, seeded

pytestmark = pytest.mark.gpu

M, N, K = 512, 768, 256


def operands(heap):
    A, B = seeded((M, K), 1), seeded((K, N), 2, scale=K**-0.5)
    return into_heap(heap, A), into_heap(heap, B), A.float() @ B.float()


def test_gather_output_block_sizes_and_words(lib):
    from tileccl_amd.v2 import FusedGemmAllGather, SymmetricHeap

    heaps = SymmetricHeap.create_all(64 << 20, 2)
    try:
        op = FusedGemmAllGather(heaps[0], M, N, directions="push")
        A, B, want = operands(heaps[0])
        first = op.out
        op(A, B)
        first.zero_()
        other = heaps[0].allocate_tensor((2 * M, N), torch.float16)
        other.fill_(7.0)
        op.out, op.local_block = other, other[:M]
        for _ in range(2):
            assert op(A, B) is other
        op.check_faults()
        assert_gemm_close(other[:M], want, tight=0.004)
        assert torch.equal(bits(heaps[0].peer_view(other, 1)[:M]), bits(other[:M]))
        assert bool((other[M:] == 7.0).all()) and not first.any()
        op.words.trace_ready_clock = op.signals.trace_ready_clock
        op(A, B)
        op.check_faults()
        assert bool((op.signals.trace_ready_clock != 0).all())
        fault = op.words.fault = torch.zeros(1, dtype=torch.int64, device="cuda")
        op.words.trace_ready_clock = None
        op.directions, op.words.spin_limit_ns = 3, 100_000  # a pull from a peer that has not produced anything
        op(A, B)
        torch.cuda.synchronize()
        assert int(fault.item()) == 1
        fault.zero_()
        op.local_block = other[M:]  # not this rank's rows of `out`
        with pytest.raises(ValueError, match="rank"):
            op(A, B)
        op.local_block = other[:M]
        for name in ("block_m", "block_n"):
            setattr(op, name, 96)
            with pytest.raises(ValueError, match="plan tile"):
                op(A, B)
            setattr(op, name, 128)
        # Refused launches were none: the counters, which a traced launch waits for itself, are still in step.
        op.directions, op.words.spin_limit_ns, op.words.trace_ready_clock = 1, 2_000_000_000, op.signals.trace_ready_clock
        op(A, B)
        op.check_faults()
    finally:
        for h in heaps:
            h.cleanup()


def test_reduction_tensors(lib):
    from tileccl_amd.v2 import FusedGemmReduceScatter, SymmetricHeap

    heaps = SymmetricHeap.create_all(64 << 20, 2)
    try:
        op = FusedGemmReduceScatter(heaps[0], M, N, emulate_peer=False)
        A, B, want = operands(heaps[0])
        op.mark_peers_ready()
        op(A, B)
        old = op.partial, op.out
        for t in old:
            t.zero_()
        op.partial = heaps[0].allocate_tensor((M, N), torch.float32)
        op.out = heaps[0].allocate_tensor((M // 2, N), torch.bfloat16)  # and of another type
        heaps[0].peer_view(op.partial, 1).fill_(2.0)
        for _ in range(2):
            assert op(A, B) is op.out
        op.check_faults()
        assert_gemm_close(op.out, want[:M // 2] + 2.0, tight=0.032)
        assert not old[0].any() and not old[1].any()
    finally:
        for h in heaps:
            h.cleanup()


@pytest.mark.parametrize("kind", ["all-scatter", "chained"])
def test_pattern_settings(lib, kind):
    import tileccl_amd as tileccl
    from tileccl_amd.patterns import TileGroupPattern
    from tileccl_amd.patterns.chained_ag_gemm_rs import ChainedAGGemmRSPattern

    ctx = tileccl.init_local(world_size=1, heap_size=64 << 20)[0]
    try:
        A, B, want = operands(ctx.heap)
        out = ctx.zeros(M, N, dtype=torch.float16)
        pattern = (TileGroupPattern if kind == "all-scatter" else ChainedAGGemmRSPattern)(ctx)
        pattern.execute(A, B, out)
        pattern.BLOCK_M = 256
        out.zero_()
        pattern.execute(A, B, out)
        pattern.check_faults()
        assert_gemm_close(out, want, tight=0.004)
        pattern.BLOCK_M = 96
        with pytest.raises(ValueError, match="plan tile"):
            pattern.execute(A, B, out)
    finally:
        ctx.heap.cleanup()
