"""A refused AllGather -> GEMM -> scatter call takes nothing from the heap, which gives nothing back: the ranks' allocations
stay at the same offsets."""

from types import SimpleNamespace

import pytest
import torch

from tileccl_amd import TileCCLContext
from tileccl_amd.patterns.chained_ag_gemm_rs import ChainedAGGemmRSPattern


class Heap:
    local_base, live_id, size, rank, world_size = 4096, 1, 1 << 20, 0, 2

    def __init__(self, inside):
        self.inside, self.taken = inside, []

    def owns_tensor(self, t):
        return any(t is x for x in self.inside)

    def allocate_tensor(self, shape, dtype):
        self.taken.append(shape)
        return torch.zeros(shape, dtype=dtype)


@pytest.mark.parametrize("schedule", ["bulk_sync", "wg_specialized", "tile_group"])
@pytest.mark.parametrize("refused,match", [("columns", "W rows"), ("output", "must be"), ("dtype", "dtype"), ("shard outside", "input_shard must live"),
                                           ("output outside", "output must live"), ("1-D", None), ("0-D", None), ("workspace", "gathered_workspace")])
def test_a_refused_call_allocates_nothing(lib, refused, match, schedule):
    shard, W, out = torch.zeros(8, 16), torch.zeros(32, 24), torch.zeros(8, 24)
    inside, workspace = [shard, W, out], None
    if refused == "columns":
        W = torch.zeros(40, 24)
    elif refused == "output":
        inside[2] = out = torch.zeros(8, 16)
    elif refused == "dtype":
        W = W.half()
    elif refused == "shard outside":
        inside.remove(shard)
    elif refused == "output outside":
        inside = [shard, W]
    elif refused in ("1-D", "0-D"):
        shard = shard[0] if refused == "1-D" else shard[0, 0]
    elif refused == "workspace":
        workspace = torch.zeros(8, 16)
    heap = Heap(inside)
    ctx = TileCCLContext(rank=0, world_size=2, device="cpu", backend_name="hip", backend=SimpleNamespace())
    ctx.heap = heap
    pattern = ChainedAGGemmRSPattern(ctx, schedule=schedule)
    for _ in range(2):
        with pytest.raises(ValueError, match=match):
            pattern.execute(shard, W, out, workspace)
    assert heap.taken == [] and not any(isinstance(v, torch.Tensor) for v in ctx._workspace_cache.values())
