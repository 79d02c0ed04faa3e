"""Sums behind the GEMM whose words another rank's launch really writes: two ranks' launches at the same time on two streams,
then one after the other (words of an earlier launch are not taken for this one's).

Shapes whose tiles do not sum themselves: 384-row shards with more K than the tiles' epilogue takes on, 256-row tiles across
two owners, e4m3 streaming tiles beyond one per CU, and a GEMM that needs every CU while the other rank waits.  Without ``emulate`` a rank
sums its own rows, with it both owners'; either way what it adds is what the peer's launch stored."""

import pytest
import torch

from oracle import collectives as oracle
from tests.gpu_util import bits
from tests.test_gpu_concurrent_ranks import SPIN_NS, both_at_once, streams  # noqa: F401
from tests.test_gpu_stream_live import E4M3, Rank, operands, out_type, small_tiles_ran
from tests.test_gpu_two_rank_readiness import SHORT_NS, expect_timeout

pytestmark = pytest.mark.gpu

SHAPES = [(768, 264, 1048, 128, torch.float16), (768, 264, 1048, 256, torch.float16), (1536, 2048, 1024, 0, E4M3), (4352, 2056, 1040, 0, torch.bfloat16)]


def reducers(heaps, M, N, macro, dtype, **kw):
    from tileccl_amd.v2 import FusedGemmReduceScatter

    partial = torch.bfloat16 if dtype is E4M3 else torch.float32
    return [FusedGemmReduceScatter(h, M, N, partial_dtype=partial, out_dtype=out_type(dtype), macro_tile=macro, **kw) for h in heaps]


def sums(op, peer, owner, dtype):
    """What the oracle makes of the partials that the two ranks (rank 0's first) have stored."""
    return oracle.reduce_rows([op.partial.cpu(), peer.partial.cpu()], owner, out_type(dtype))


@pytest.mark.parametrize("variant", ["s1", "s2"])
@pytest.mark.parametrize("emulate", [False, True])
@pytest.mark.parametrize("M,N,K,macro,dtype", SHAPES)
def test_two_live_ranks(lib, streams, M, N, K, macro, dtype, emulate, variant):  # noqa: F811
    from tileccl_amd.v2 import SymmetricHeap

    heaps = SymmetricHeap.create_all(256 << 20, 2)
    try:
        ops = reducers(heaps, M, N, macro, dtype, emulate_peer=emulate, spin_limit_ns=SPIN_NS)
        for launch in range(3):  # launch numbers stay in step; the operands change
            each = [operands(heaps[r], M, N, K, dtype, 20 * launch + 2 * r) for r in range(2)]
            for op in ops:
                op.out.fill_(7.0)
            both_at_once([Rank(op, *e[:2], e[3]) for op, e in zip(ops, each)], [e[:2] for e in each], variant, streams)
            for r, op in enumerate(ops):
                assert torch.equal(bits(op.out).cpu(), bits(sums(*ops, r, dtype))), (launch, r)
                assert torch.allclose(op.partial.float().cpu(), each[r][2], rtol=1e-2, atol=1e-1)
        assert dtype is not E4M3 or small_tiles_ran(ops[0], *each[0][:2], variant, each[0][3])
    finally:
        for h in heaps:
            h.cleanup()


@pytest.mark.parametrize("variant", ["s1", "s2"])
@pytest.mark.parametrize("M,N,K,macro,dtype", SHAPES[:3])
def test_words_of_an_earlier_launch_do_not_end_the_wait(lib, M, N, K, macro, dtype, variant):
    from tileccl_amd.v2 import SymmetricHeap

    heaps = SymmetricHeap.create_all(192 << 20, 2)
    try:
        mine, peer = reducers(heaps, M, N, macro, dtype, emulate_peer=False, spin_limit_ns=SHORT_NS)
        A, B, _, alpha = operands(heaps[0], M, N, K, dtype, 0)
        for launch in range(2):
            mine.out.fill_(7.0)
            mine(A, B, variant, alpha)  # alone: the peer's words, if any, are those of the launch before
            expect_timeout(mine)
            assert bool((mine.out == 7.0).all())
            A1, B1, _, _ = operands(heaps[1], M, N, K, dtype, 10 * (launch + 1))
            peer(A1, B1, variant, alpha)  # finds this rank's words of the same launch
            peer.check_faults()
            assert torch.equal(bits(peer.out).cpu(), bits(sums(mine, peer, 1, dtype)))
    finally:
        for h in heaps:
            h.cleanup()
