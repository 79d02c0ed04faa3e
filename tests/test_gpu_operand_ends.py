"""Nothing behind an operand's end reaches a result: what a K step of the large-tile kernel fetches past row K of a row-major
B, or past column K of A or of a k-major B, is zero whatever the memory there holds.

Each operand is the front of a larger allocation.  Filled up with NaN, which a product with zero does not remove,
the result has the bits it has with zeros there, and these are the product's."""

import pytest
import torch

from tests.gpu_util import assert_gemm_close, bits, seeded

pytestmark = pytest.mark.gpu

F8 = torch.float8_e4m3fn
M, N = 512, 512
# A K step is 64 elements (e4m3: 128) in two halves: tails inside the first and the second half, odd and even numbers of steps.
LENGTHS = [(torch.float16, 72), (torch.float16, 104), (torch.bfloat16, 136), (torch.bfloat16, 168), (torch.float16, 264),
           (F8, 80), (F8, 144), (F8, 208), (F8, 272)]


def front_of(heap, cpu, rows, cols, behind):
    """`cpu` as the front of a (rows, cols) tensor of the heap whose other elements are `behind`."""
    whole = heap.allocate_tensor((rows, -(-cols // 16) * 16), cpu.dtype)  # rows on 16-byte boundaries
    if cpu.dtype == F8:
        whole.view(torch.uint8).fill_(0x7F if behind != 0 else 0)  # e4m3: NaN
    else:
        whole.fill_(behind)
    view = whole[: cpu.shape[0], : cpu.shape[1]]
    view.copy_(cpu)
    return view


def operands(heap, dtype, K, kmajor, behind, M=M, N=N):
    half = torch.float16 if dtype == F8 else dtype
    A_cpu, B_cpu = seeded((M, K), 0, half).to(dtype), seeded((K, N), 1, half, scale=K**-0.5).to(dtype)
    A = front_of(heap, A_cpu, M + 256, K + 512, behind)
    B = front_of(heap, B_cpu.t(), N + 256, K + 512, behind).t() if kmajor else front_of(heap, B_cpu, K + 512, N + 256, behind)
    return A, B, A_cpu.float() @ B_cpu.float()


@pytest.mark.parametrize("kmajor", [False, True])
@pytest.mark.parametrize("directions", ["push", "both"])  # the K loop of phases, the one beside a pull
@pytest.mark.parametrize("dtype,K", LENGTHS)
def test_all_gather(lib, dtype, K, directions, kmajor):
    from tileccl_amd.v2 import FusedGemmAllGather, SymmetricHeap

    heaps = SymmetricHeap.create_all(64 << 20, 2)
    try:
        out = torch.bfloat16 if dtype == F8 else dtype
        ops = [FusedGemmAllGather(h, M, N, out, directions=directions, macro_tile=256) for h in heaps]
        got = []
        for behind in (0.0, float("nan")):
            A, B, want = operands(heaps[0], dtype, K, kmajor, behind)
            for variant in ("s0", "s2"):
                ops[0].local_block.zero_()
                ops[0].mark_peers_ready()
                ops[0](A, B, variant)
                ops[0].check_faults()
                assert_gemm_close(ops[0].local_block, want)
                got.append(bits(ops[0].local_block).cpu().clone())
        assert all(torch.equal(g, got[0]) for g in got)
    finally:
        for h in heaps:
            h.cleanup()


@pytest.mark.parametrize("kmajor", [False, True])
@pytest.mark.parametrize("rows,cols", [(256 + 64, 256 + 32), (256 + 72, 256 + 40), (8, 8)])  # last tiles without and with a second half
@pytest.mark.parametrize("dtype,K", [LENGTHS[0], LENGTHS[3], LENGTHS[7]])
def test_last_tiles(lib, dtype, K, rows, cols, kmajor):
    from tileccl_amd.v2 import FusedGemmAllGather, SymmetricHeap

    heaps = SymmetricHeap.create_all(64 << 20, 2)
    try:
        out = torch.bfloat16 if dtype == F8 else dtype
        ops = [FusedGemmAllGather(h, rows, cols, out, directions="push", macro_tile=256) for h in heaps]
        got = []
        for behind in (0.0, float("nan")):
            A, B, want = operands(heaps[0], dtype, K, kmajor, behind, rows, cols)
            ops[0](A, B, "s2")
            ops[0].check_faults()
            assert_gemm_close(ops[0].local_block, want)
            got.append(bits(ops[0].local_block).cpu().clone())
        assert torch.equal(got[0], got[1])
    finally:
        for h in heaps:
            h.cleanup()


@pytest.mark.parametrize("dtype,K", LENGTHS)
def test_reduce_scatter_in_the_tiles(lib, dtype, K):
    from tileccl_amd.v2 import FusedGemmReduceScatter, SymmetricHeap

    heaps = SymmetricHeap.create_all(64 << 20, 2)
    try:
        out = torch.bfloat16 if dtype == F8 else dtype
        partial = torch.bfloat16 if dtype == F8 else torch.float32
        ops = [FusedGemmReduceScatter(h, M, N, partial_dtype=partial, out_dtype=out, macro_tile=256, own_rows_in_registers=True) for h in heaps]
        ops[1].partial.zero_()  # the sums are this rank's rows
        got = []
        for behind in (0.0, float("nan")):
            A, B, want = operands(heaps[0], dtype, K, False, behind)
            ops[0].mark_peers_ready()
            ops[0](A, B, "s2")
            ops[0].check_faults()
            assert_gemm_close(ops[0].out, want[: M // 2])
            got.append(bits(ops[0].out).cpu().clone())
        assert torch.equal(got[0], got[1])
    finally:
        for h in heaps:
            h.cleanup()


@pytest.mark.parametrize("Ks", [64, 192])
def test_gathered_input_with_a_wider_pitch(lib, Ks):
    """The kernel that reads A's column shards in place: B ends at row K, each shard at its column Ks and row M."""
    from tileccl_amd.patterns.chained_ag_gemm_rs import ChainedAGGemmRSPattern
    import tileccl_amd as tileccl

    rows, cols, world = 2048, 4096, 3
    ctxs = tileccl.init_local(world_size=world, heap_size=256 << 20)
    try:
        K = Ks * world
        shards_cpu = [seeded((rows, Ks), 10 + p) for p in range(world)]
        W_cpu = seeded((K, cols), 1, scale=K**-0.5)
        shards = []
        for c, cpu in zip(ctxs, shards_cpu):
            t = c.zeros(rows, Ks, dtype=cpu.dtype)
            t.copy_(cpu)
            shards.append(t)
        outs = [c.zeros(rows, cols, dtype=torch.float16) for c in ctxs]
        got = []
        for behind in (0.0, float("nan")):
            whole = ctxs[0].zeros(K + 512, cols, dtype=torch.float16)
            whole.fill_(behind)
            whole[:K].copy_(W_cpu)
            pattern = ChainedAGGemmRSPattern(ctxs[0], schedule="tile_group")
            pattern.execute(shards[0], whole[:K], outs[0])
            pattern.check_faults()
            torch.cuda.synchronize()
            assert_gemm_close(outs[0], torch.cat(shards_cpu, 1).float() @ W_cpu.float(), tight=0.004)
            got.append(bits(outs[0]).cpu().clone())
        assert torch.equal(got[0], got[1])
    finally:
        for c in ctxs:
            c.heap.cleanup()
