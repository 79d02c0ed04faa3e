"""A context whose heap is replaced by one at the same address: patterns, plans and operations kept from before must not go on
with what they had in the old heap, whose place is someone else's now."""

import pytest
import torch

from tests.gpu_util import assert_gemm_close, seeded

pytestmark = pytest.mark.gpu

M, N, K, WORLD = 256, 512, 128, 2


def put(heap, cpu):
    t = heap.allocate_tensor(tuple(cpu.shape), cpu.dtype)
    t.copy_(cpu)
    return t


@pytest.mark.parametrize("kind", ["bulk_sync", "wg_specialized", "tile_group", "chained", "reduce"])
def test_calls_and_words_go_with_the_heap(lib, kind):
    import tileccl_amd as tileccl
    from tileccl_amd.memory.symmetric_heap import SymmetricHeap
    from tileccl_amd.patterns import BulkSyncPattern, TileGroupPattern, WGSpecializedPattern
    from tileccl_amd.patterns.chained_ag_gemm_rs import ChainedAGGemmRSPattern

    size = 32 << 20
    ctxs = tileccl.init_local(world_size=WORLD, heap_size=size)
    old = [c.heap for c in ctxs]
    A, B = seeded((M, K), 1), seeded((K, N), 2, scale=K**-0.5)
    made = {"bulk_sync": BulkSyncPattern, "wg_specialized": WGSpecializedPattern, "tile_group": TileGroupPattern,
            "chained": ChainedAGGemmRSPattern}
    patterns = [made[kind](c) for c in ctxs] if kind in made else None

    def run(guarded):
        calls = []
        for c in ctxs:
            mine = A[:, c.rank * (K // WORLD):(c.rank + 1) * (K // WORLD)].contiguous() if kind == "chained" else A
            out = c.heap.allocate_tensor((M, N // WORLD if kind == "reduce" else N), torch.float16)
            calls.append((put(c.heap, mine), put(c.heap, B), out))
        # What the first run allocates behind its tensors (words, workspaces) is where these lie in the second one.
        guards = [c.heap.allocate_tensor((1 << 20,), torch.int32).fill_(7) for c in ctxs] if guarded else []
        for _ in range(2):  # (a reduction finds its peer's partials in the second turn)
            for r, c in enumerate(ctxs):
                if kind == "reduce":
                    tileccl.ops.gemm_reducescatter(*calls[r], ctx=c)
                elif kind == "chained":
                    patterns[r].execute(*calls[r])
                else:
                    patterns[r].execute(*calls[r], full_N=N, b_layout="full", c_layout="full")
        torch.cuda.synchronize()
        want = A.float() @ B.float()
        for r, (_, _, out) in enumerate(calls):
            if kind == "reduce":
                assert_gemm_close(out, 2 * want[:, r * (N // WORLD):(r + 1) * (N // WORLD)], tight=0.008)
            else:
                assert_gemm_close(out, want, tight=0.004)
        assert all(bool((g == 7).all()) for g in guards)

    try:
        run(guarded=False)
        assert all(h.bytes_allocated < (4 << 20) for h in old)
        new = [SymmetricHeap(size, r, WORLD, _arena=h._arena) for r, h in enumerate(old)]  # the same slices once more
        assert [h.local_base for h in new] == [h.local_base for h in old]
        assert len({h.live_id for h in old + new}) == 2 * WORLD
        for c, h in zip(ctxs, new):
            c.attach_heap(h)
        run(guarded=True)
    finally:
        for h in old:
            h.cleanup()
        assert all(h.live_id == 0 for h in old)


@pytest.mark.parametrize("kind", ["bulk_sync", "wg_specialized", "tile_group", "chained"])
def test_the_old_heap_is_given_back(lib, kind):
    """A pattern that has gone on to another heap holds nothing of the one before: its device memory is freed."""
    import gc
    import weakref

    import tileccl_amd as tileccl
    from tileccl_amd.memory.symmetric_heap import SymmetricHeap
    from tileccl_amd.patterns import BulkSyncPattern, TileGroupPattern, WGSpecializedPattern
    from tileccl_amd.patterns.chained_ag_gemm_rs import ChainedAGGemmRSPattern

    made = {"bulk_sync": BulkSyncPattern, "wg_specialized": WGSpecializedPattern, "tile_group": TileGroupPattern,
            "chained": ChainedAGGemmRSPattern}
    (ctx,) = tileccl.init_local(world_size=1, heap_size=32 << 20)
    pattern = made[kind](ctx)

    def run():
        A, B = put(ctx.heap, seeded((M, K), 1)), put(ctx.heap, seeded((K, N), 2, scale=K**-0.5))
        out = ctx.heap.allocate_tensor((M, N), torch.float16)
        for _ in range(2):
            pattern.execute(A, B, out)
        torch.cuda.synchronize()

    run()
    old = ctx.heap
    arena = weakref.ref(old._arena)
    new = SymmetricHeap(32 << 20, 0, 1)
    ctx.attach_heap(new)
    old.cleanup()
    del old
    run()
    gc.collect()
    assert arena() is None
    new.cleanup()
