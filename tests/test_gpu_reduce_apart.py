"""Reduce-scatters whose sums are a launch of their own behind the GEMM: shards that are no whole 256-row tiles, on every
GEMM kernel that can precede it (128-row tiles, 256-row tiles, streaming tiles beyond one per CU), and several ranks.

The sums are made in fp32 from the stored partials, owner first, the others ascending, and rounded once: bit for bit what
the oracle makes of the partial that the GEMM stored."""

import pytest
import torch

from oracle import collectives as oracle
from tests.gpu_util import assert_gemm_close, bits, into_heap, seeded

pytestmark = pytest.mark.gpu
F8 = torch.float8_e4m3fn


def run(world, M, N, K, macro, in_dtype, partial, out, variant, emulate, mark=True, **kw):
    from tileccl_amd.v2 import FusedGemmReduceScatter, SymmetricHeap

    heaps = SymmetricHeap.create_all(128 << 20, world)
    try:
        ops = [FusedGemmReduceScatter(h, M, N, partial_dtype=partial, out_dtype=out, emulate_peer=emulate, macro_tile=macro, **kw)
               for h in heaps]
        half = torch.float16 if in_dtype == F8 else in_dtype
        A_cpu, B_cpu = seeded((M, K), 0, half).to(in_dtype), seeded((K, N), 1, half, scale=K**-0.5).to(in_dtype)
        A, B = into_heap(heaps[0], A_cpu), into_heap(heaps[0], B_cpu)
        peers = [seeded((M, N), 10 + p, partial) * (1000.0 if world > 2 else 1.0) for p in range(1, world)]  # the order matters
        for op, peer in zip(ops[1:], peers):
            op.partial.copy_(peer)
        for op in ops:
            op.out.zero_()
        if mark:
            ops[0].mark_peers_ready()
        ops[0](A, B, variant)
        if not mark:
            with pytest.raises(Exception):
                ops[0].check_faults()
            return None, [op.out.cpu() for op in ops]
        ops[0].check_faults()
        assert_gemm_close(ops[0].partial, A_cpu.float() @ B_cpu.float())
        return [ops[0].partial.cpu(), *peers], [op.out.cpu() for op in ops]
    finally:
        for h in heaps:
            h.cleanup()


@pytest.mark.parametrize("variant", ["s1", "s2"])
@pytest.mark.parametrize("emulate", [True, False])
@pytest.mark.parametrize("world,M,N,K,macro,in_dtype,partial,out", [
    (2, 768, 264, 1048, 128, torch.float16, torch.float32, torch.float16),   # 384-row shards, 128-row tiles
    (3, 384, 264, 72, 128, torch.bfloat16, torch.float32, torch.bfloat16),   # three ranks, one tile row each
    (4, 512, 520, 136, 256, torch.float16, torch.float32, torch.float16),    # 256-row tiles across two owners
    (2, 256, 272, 144, 256, F8, torch.bfloat16, torch.bfloat16),             # one tile, two owners
    (2, 768, 2064, 272, 0, F8, torch.bfloat16, torch.bfloat16),              # streaming tiles that sum themselves, most CUs at work
    (2, 1536, 2048, 1024, 0, F8, torch.bfloat16, torch.bfloat16),            # streaming tiles, those of the own rows beyond one per CU
    (2, 1280, 3400, 1040, 0, torch.bfloat16, torch.bfloat16, torch.bfloat16),  # the kernel chosen by cost
])
def test_sums_behind_the_gemm_are_the_oracles(lib, variant, emulate, world, M, N, K, macro, in_dtype, partial, out):
    partials, outs = run(world, M, N, K, macro, in_dtype, partial, out, variant, emulate)
    for owner in range(world):
        if owner == 0 or emulate:
            assert torch.equal(bits(outs[owner]), bits(oracle.reduce_rows(partials, owner, out))), owner
        else:
            assert torch.all(outs[owner] == 0), owner


@pytest.mark.parametrize("variant", ["s1", "s2"])
def test_a_peer_that_has_not_published_is_waited_for_and_reported(lib, variant):
    """Nobody marks the peers' words: the bounded wait expires, nothing is summed, the fault is raised on the host."""
    _, outs = run(2, 768, 264, 1048, 128, torch.float16, torch.float32, torch.float16, variant, True, mark=False, spin_limit_ns=200_000)
    assert all(torch.all(o == 0) for o in outs)


@pytest.mark.parametrize("variant", ["s1", "s2"])
def test_sums_behind_a_wait_of_their_own_do_not_run_where_it_expired(lib, variant):
    """Three ranks: one workgroup per owner waits in a launch ahead of the sums."""
    _, outs = run(3, 384, 264, 72, 128, torch.bfloat16, torch.float32, torch.bfloat16, variant, True, mark=False, spin_limit_ns=200_000)
    assert all(torch.all(o == 0) for o in outs)


@pytest.mark.parametrize("variant", ["s1", "s2"])
@pytest.mark.parametrize("world,M,N,K,macro", [(2, 768, 264, 1048, 128), (3, 768, 264, 136, 128), (2, 1792, 1200, 1520, 0)])
def test_own_rows_kept_in_registers_are_never_stored(lib, variant, world, M, N, K, macro):
    """128-row tiles that wait, at most one per CU: asked to keep its own rows in registers, the launch sums in its tiles, and
    those rows of the partial keep what they held."""
    from tileccl_amd.v2 import FusedGemmReduceScatter, SymmetricHeap

    peers = [seeded((M, N), 10 + p, torch.float32) * (1000.0 if world > 2 else 1.0) for p in range(1, world)]
    A_cpu, B_cpu = seeded((M, K), 0, torch.bfloat16), seeded((K, N), 1, torch.bfloat16, scale=K**-0.5)
    got = []
    for own in (False, True):
        heaps = SymmetricHeap.create_all(128 << 20, world)
        try:
            ops = [FusedGemmReduceScatter(h, M, N, out_dtype=torch.bfloat16, macro_tile=macro, own_rows_in_registers=own) for h in heaps]
            A, B = into_heap(heaps[0], A_cpu), into_heap(heaps[0], B_cpu)
            for op, peer in zip(ops[1:], peers):
                op.partial.copy_(peer)
            ops[0].partial.fill_(-3.0)
            ops[0].mark_peers_ready()
            ops[0](A, B, variant)
            ops[0].check_faults()
            got.append((ops[0].partial.cpu(), [op.out.cpu() for op in ops]))
        finally:
            for h in heaps:
                h.cleanup()
    (stored, outs), (kept, kept_outs) = got
    shard = M // world
    for owner in range(world):
        assert torch.equal(bits(outs[owner]), bits(oracle.reduce_rows([stored, *peers], owner, torch.bfloat16))), owner
        assert torch.equal(bits(kept_outs[owner]), bits(outs[owner])), owner
    assert torch.all(kept[:shard] == -3.0) and not torch.any(stored[:shard] == -3.0)
    assert torch.equal(bits(kept[shard:]), bits(stored[shard:]))
