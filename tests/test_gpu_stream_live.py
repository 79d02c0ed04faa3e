"""The small-tile (streaming) kernel's waits against words that another rank's launch really writes.

First two ranks' launches at the same time on two streams, with the grids that the library chooses (tiles on a part of the
CUs, on all of them, and e4m3 tiles beyond what is resident at once): each pulls from, or reduces, what the other is producing.
Then one after the other: a launch finds the words of the one before it, and gives up (bounded) where they are of an
earlier launch.  Which workgroups wait, and that those waits end, is shown on the CPU in ``test_stream_grid.py``."""

import pytest
import torch

from oracle import collectives as oracle
from tests.gpu_util import assert_gemm_close, bits, into_heap, seeded
from tests.test_gpu_concurrent_ranks import SPIN_NS, both_at_once, streams  # noqa: F401
from tests.test_gpu_two_rank_readiness import SHORT_NS, expect_timeout

pytestmark = pytest.mark.gpu

E4M3 = torch.float8_e4m3fn
# tiles: 128 of 32x64, 256 of 32x32, 256 of 64x64; e4m3: 256 of 32x64, 768, 676 and 528 of 64x64
GATHERS = [(256, 1000, 520, torch.float16), (512, 512, 512, torch.float16), (1024, 1024, 1000, torch.bfloat16),
           (512, 1024, 512, E4M3), (1536, 2048, 1024, E4M3), (832, 3328, 1024, E4M3), (2112, 1024, 2048, E4M3)]
# own rows on half the tiles: 192 of 64x64, 256 of 32x32; e4m3: 256 and 512 of 64x64 (256 of them wait)
REDUCES = [(1024, 768, 1024, torch.float16), (512, 512, 512, torch.bfloat16), (2048, 512, 512, E4M3), (2048, 1024, 1024, E4M3)]


def operands(heap, M, N, K, dtype, seed):
    """(A, B on the heap, their fp32 product, the factor that the operation is called with)."""
    if dtype is E4M3:
        A, B = (seeded(s, seed + i, torch.float32, scale=64.0).clamp(-448, 448).to(E4M3) for i, s in enumerate(((M, K), (K, N))))
        alpha = K**-0.5 / 4096
    else:
        A, B, alpha = seeded((M, K), seed, dtype), seeded((K, N), seed + 1, dtype, scale=K**-0.5), 1.0
    return into_heap(heap, A), into_heap(heap, B), (A.float() @ B.float()) * alpha, alpha


def out_type(dtype):
    return torch.bfloat16 if dtype is E4M3 else dtype


TIGHT = {torch.float16: 0.004, torch.bfloat16: 0.032}  # an ulp of the largest results (below 8)


class Rank:
    """An operation and its operands in the form that ``both_at_once`` calls."""

    def __init__(self, op, A, B, alpha):
        self.op, self.A, self.B, self.alpha = op, A, B, alpha

    def __call__(self, A, B, variant):
        self.op(A, B, variant, self.alpha)

    def check_faults(self):
        self.op.check_faults()


def small_tiles_ran(op, A, B, variant, alpha):
    """Only the streaming kernel counts arrivals: from beyond what a plan tile has, its words end elsewhere.  (Nothing is
    published by this launch, which is therefore the last one of the words.)"""
    op.words.arrivals.fill_(1 << 30)
    op.words.spin_limit_ns = SHORT_NS
    op(A, B, variant, alpha)
    torch.cuda.synchronize()
    return bool((op.words.arrivals != 1 << 30).any())


@pytest.mark.parametrize("variant,directions", [("s1", "pull"), ("s2", "pull"), ("s2", "both")])
@pytest.mark.parametrize("M,N,K,dtype", GATHERS)
def test_all_gather_of_two_live_ranks(lib, streams, M, N, K, dtype, variant, directions):  # noqa: F811
    from tileccl_amd.v2 import FusedGemmAllGather, SymmetricHeap

    heaps = SymmetricHeap.create_all(192 << 20, 2)
    try:
        ops = [FusedGemmAllGather(h, M, N, out_type(dtype), directions=directions, spin_limit_ns=SPIN_NS) for h in heaps]
        for launch in range(3):
            each = [operands(heaps[r], M, N, K, dtype, 10 * launch + 2 * r) for r in range(2)]
            for op in ops:
                op.out.zero_()
            both_at_once([Rank(op, *e[:2], e[3]) for op, e in zip(ops, each)], [e[:2] for e in each], variant, streams)
            for r, op in enumerate(ops):
                assert_gemm_close(op.local_block, each[r][2], tight=TIGHT[out_type(dtype)])
                other = slice((1 - r) * M, (2 - r) * M)
                assert torch.equal(bits(op.out[other]), bits(ops[1 - r].local_block)), (launch, r)
                assert not op.words.arrivals.any()
        assert small_tiles_ran(ops[0], *each[0][:2], variant, each[0][3])
    finally:
        for h in heaps:
            h.cleanup()


@pytest.mark.parametrize("variant", ["s1", "s2"])
@pytest.mark.parametrize("own", [False, True])
@pytest.mark.parametrize("M,N,K,dtype", REDUCES)
def test_reduce_scatter_of_two_live_ranks(lib, streams, M, N, K, dtype, own, variant):  # noqa: F811
    from tileccl_amd.v2 import FusedGemmReduceScatter, SymmetricHeap

    partial = torch.bfloat16 if dtype is E4M3 else torch.float32
    heaps = SymmetricHeap.create_all(192 << 20, 2)
    try:
        ops = [FusedGemmReduceScatter(h, M, N, partial_dtype=partial, out_dtype=out_type(dtype), emulate_peer=False,
                                      own_rows_in_registers=own, spin_limit_ns=SPIN_NS) for h in heaps]
        for launch in range(2):
            each = [operands(heaps[r], M, N, K, dtype, 20 * launch + 2 * r) for r in range(2)]
            for op in ops:
                op.out.zero_()
            both_at_once([Rank(op, *e[:2], e[3]) for op, e in zip(ops, each)], [e[:2] for e in each], variant, streams)
            got = [op.out.clone() for op in ops]
            for r, op in enumerate(ops):  # the bulk variant stores whole partials, added up in the same order
                op(*each[r][:2], "s0", each[r][3])
                op.check_faults()
            for r, op in enumerate(ops):
                want = oracle.reduce_rows([o.partial.cpu() for o in ops], r, out_type(dtype))
                assert torch.equal(bits(got[r]).cpu(), bits(want)), (launch, r)
                assert not op.words.arrivals.any()
        assert small_tiles_ran(ops[0], *each[0][:2], variant, each[0][3])
    finally:
        for h in heaps:
            h.cleanup()


@pytest.mark.parametrize("variant", ["s1", "s2"])
@pytest.mark.parametrize("M,N,K,dtype", [GATHERS[0], GATHERS[1], GATHERS[4]])
def test_pulls_follow_the_peers_own_launch(lib, M, N, K, dtype, variant):
    from tileccl_amd.v2 import FusedGemmAllGather, SymmetricHeap

    heaps = SymmetricHeap.create_all(192 << 20, 2)
    try:
        puller, peer = (FusedGemmAllGather(h, M, N, out_type(dtype), directions=d) for h, d in zip(heaps, ("pull", "push")))
        A, B, want, alpha = operands(heaps[0], M, N, K, dtype, 0)
        for launch in range(2):
            A1, B1, _, _ = operands(heaps[1], M, N, K, dtype, 10 * (launch + 1))
            # Alone: the peer's words are those of the launch before.
            limit, puller.words.spin_limit_ns = puller.words.spin_limit_ns, SHORT_NS
            puller.out[M:].fill_(7.0)
            puller(A, B, variant, alpha)
            expect_timeout(puller)
            assert bool((puller.out[M:] == 7.0).all())
            assert_gemm_close(puller.local_block, want, tight=TIGHT[out_type(dtype)])
            puller.words.spin_limit_ns = limit
            peer(A1, B1, variant, alpha)
            peer.check_faults()
            puller.out[M:].zero_()
            puller.words.epoch = puller.words.lock_epoch = launch  # the same launch once more
            if variant == "s2":  # whose tiles have counted already
                puller.signals.counter.copy_(torch.tensor([launch * t for t in puller.plan.tile_counts()], dtype=torch.int32))
            puller(A, B, variant, alpha)
            puller.check_faults()
            assert torch.equal(bits(puller.out[M:]), bits(peer.local_block))
    finally:
        for h in heaps:
            h.cleanup()


@pytest.mark.parametrize("variant", ["s1", "s2"])
@pytest.mark.parametrize("M,N,K,dtype", [REDUCES[0], REDUCES[1], REDUCES[3]])
def test_reductions_wait_for_the_peers_own_launch(lib, M, N, K, dtype, variant):
    from tileccl_amd.v2 import FusedGemmReduceScatter, SymmetricHeap

    partial = torch.bfloat16 if dtype is E4M3 else torch.float32
    heaps = SymmetricHeap.create_all(192 << 20, 2)
    try:
        mine, peer = (FusedGemmReduceScatter(h, M, N, partial_dtype=partial, out_dtype=out_type(dtype), emulate_peer=False,
                                             spin_limit_ns=SHORT_NS) for h in heaps)
        A, B, _, alpha = operands(heaps[0], M, N, K, dtype, 0)
        A1, B1, _, _ = operands(heaps[1], M, N, K, dtype, 10)
        peer(A1, B1, variant, alpha)  # stores and publishes its partials; nobody has produced what it would add
        expect_timeout(peer)
        mine(A, B, "s0", alpha)
        mine.check_faults()
        want = mine.out.clone()
        mine.out.zero_()
        mine.words.spin_limit_ns = SPIN_NS
        mine(A, B, variant, alpha)
        mine.check_faults()
        assert torch.equal(bits(mine.out), bits(want))
        mine.words.spin_limit_ns = SHORT_NS
        mine.out.fill_(7.0)
        mine(A, B, variant, alpha)  # launch 2: the peer's words say "launch 1"
        expect_timeout(mine)
        assert bool((mine.out == 7.0).all())
    finally:
        for h in heaps:
            h.cleanup()
