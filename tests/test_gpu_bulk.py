"""The stand-alone copies and reductions at the edges of how they are split: a workgroup's 256 threads, the
units per thread of each instantiation (worlds of 2, 4 and 8), shares of more than one task, and sizes
beyond the grid's first pass."""

import pytest
import torch

from oracle import collectives as oracle
from tests.gpu_util import bits, into_heap, seeded

pytestmark = pytest.mark.gpu


def heaps_of(world, size):
    from tileccl_amd.memory.symmetric_heap import SymmetricHeap

    return SymmetricHeap.create_all(size=size, world_size=world)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("world,units", [(2, 1023), (2, 1025), (3, 511), (4, 513), (5, 255), (8, 256), (8, 257), (2, 2 * 1024 * 1024 + 3)])
def test_allreduce_calls_and_one_launch(lib, world, units, dtype):
    """Rank by rank (owner first) and all roles at once (ascending): exactly the oracle's bits."""
    from tileccl_amd.primitives import allreduce, allreduce_staged

    numel = 8 * (units // world * world if units > 4096 else units * world)
    heaps = heaps_of(world, 2 * numel * 4 + (4 << 20))
    try:
        cpu = [seeded((numel,), 5 + r, dtype) for r in range(world)]
        ts = [into_heap(h, c) for h, c in zip(heaps, cpu)]
        us = [into_heap(h, c) for h, c in zip(heaps, cpu)]
        for t, h in zip(ts, heaps):
            allreduce(t, h)
        allreduce_staged(us, heaps)
        torch.cuda.synchronize()
        for got, want in ((ts, oracle.allreduce(cpu)), (us, oracle.allreduce_staged(cpu))):
            for r in range(world):
                assert torch.equal(bits(got[r]).cpu(), bits(want[r])), r
    finally:
        for h in heaps:
            h.cleanup()


@pytest.mark.parametrize("world,rows,cols,ld", [(2, 3, 4104, 4112), (3, 257, 40, 48), (4, 1024, 520, 520), (8, 33, 2056, 2064), (2, 4099, 2048, 2056)])
def test_exchange_and_gather_with_pitched_rows(lib, world, rows, cols, ld):
    """Every transfer of an exchange and of a column gather lands where it belongs, and nothing else is written."""
    import ctypes as C

    from tileccl_amd import _launch, _lib

    heaps = heaps_of(world, 4 * world * rows * (world * cols + ld) + (8 << 20))
    try:
        outs = [h.allocate_tensor((world * rows, ld), torch.float16) for h in heaps]
        shards = [into_heap(h, seeded((rows, ld), 30 + r)) for r, h in enumerate(heaps)]
        gathered = [h.allocate_tensor((rows, world * cols), torch.float16) for h in heaps]
        for r in range(world):
            outs[r].copy_(seeded((world * rows, ld), r))
        before = [o.cpu() for o in outs]
        me = world - 1
        view = _launch.heap_view(heaps[me].get_heap_bases(), me, world)
        transport = _launch.transport_desc(_lib.DIR_PUSH | _lib.DIR_PULL, 16384, None, 0)
        _lib.check(lib.tccl_exchange_rows(_launch.ptr(outs[me]), rows, cols, ld, 2, C.byref(view), C.byref(transport),
                                          _launch.stream_ptr()), "exchange")
        _lib.check(lib.tccl_gather_cols(_launch.ptr(gathered[me]), world * cols, _launch.ptr(shards[me]), ld, rows, cols, 2,
                                        C.byref(view), None, _launch.stream_ptr()), "gather")
        torch.cuda.synchronize()
        for r in range(world):
            want = before[r].clone()
            blocks = range(world) if r == me else (me,)
            for b in blocks:
                if b != r:
                    want[b * rows:(b + 1) * rows, :cols] = before[b][b * rows:(b + 1) * rows, :cols]
            assert torch.equal(bits(outs[r].cpu()), bits(want)), r
        assert torch.equal(bits(gathered[me].cpu()), bits(torch.cat([s[:, :cols].cpu() for s in shards], dim=1)))
    finally:
        for h in heaps:
            h.cleanup()
