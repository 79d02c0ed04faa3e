"""The tiled kernels that ``tccl_gemm`` and the pushing launches choose from by shape: the same bits from all of them."""

import ctypes as C

import pytest
import torch

from tileccl_amd import _launch, _lib, ops
from tileccl_amd.v2 import FusedGemmAllGather, SymmetricHeap

pytestmark = pytest.mark.gpu

# Which kernel each shape gets on 256 CUs: 128 x 256 tiles (wide), 128 x 128 in steps of 64 (deep).
SHAPES = [
    (2064, 2064, 264),    # wide: remainders in rows, columns and K
    (1, 66000, 64),       # wide: one row, one K step
    (1025, 8200, 1096),   # wide, two rounds; an odd number of plan tiles across
    (130, 8328, 1032),    # deep: remainders everywhere
    (128, 128 * 256, 2048),  # deep: one tile on every CU
]


def operands(M, N, K, dtype, layout):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randn(M, K, generator=g, device="cuda").to(dtype)
    B = (torch.randn(K, N, generator=g, device="cuda") * K**-0.5).to(dtype)
    return A, B.t().contiguous().t() if layout == "nk" else B


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype,out", [(torch.float16, torch.float16), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("layout", ["kn", "nk"])
def test_chosen_tiles_against_the_oracle_and_the_small_tiles(lib, shape, dtype, out, layout):
    M, N, K = shape
    A, B = operands(M, N, K, dtype, layout)
    got = torch.full((M + 1, N), 7.0, dtype=out, device="cuda")
    small = torch.zeros(M, N, dtype=out, device="cuda")
    for d in (_launch.gemm_desc(A, B, got[:M]), _launch.gemm_desc(A, B, small, macro_tile=128)):
        _lib.check(lib.tccl_gemm(C.byref(d), _launch.stream_ptr()), "tccl_gemm")
    assert torch.equal(got[:M], small)
    assert bool((got[M] == 7).all())  # nothing past the last row
    cols = torch.cat([torch.arange(0, N, max(1, N // 257)), torch.arange(max(0, N - 40), N)]).unique().cuda()
    want = A.double() @ B[:, cols].double()
    torch.testing.assert_close(got[:M][:, cols].double(), want, rtol=4e-3, atol=4e-3)


@pytest.mark.parametrize("shape", SHAPES[:4])
@pytest.mark.parametrize("variant", ["s1", "s2"])
def test_pushes_and_signals_of_the_chosen_tiles(lib, shape, variant):
    M, N, K = shape
    A, B = operands(M, N, K, torch.float16, "kn")
    heaps = SymmetricHeap.create_all(2 * M * N * 2 + (32 << 20), 2)
    gathers = [FusedGemmAllGather(h, M, N, torch.float16, directions="push") for h in heaps]
    for launch in (1, 2):
        for op in gathers:
            op.out.zero_()
        gathers[1](A, B, variant=variant)
        full = gathers[1].local_block
        assert torch.equal(gathers[0].out[M:], full) and float(full.abs().sum()) > 0
        words = gathers[1].words
        if variant == "s1":
            assert bool((words.locks == launch).all())
        else:
            assert torch.equal(words.counter, launch * words.plan.tile_counts)


@pytest.mark.parametrize("M,N,K", [(1956, 2784, 264), (300, 4096, 1032), (129, 1088, 72)])
@pytest.mark.parametrize("layout", ["kn", "nk"])
def test_ragged_column_shards_in_one_launch(lib, M, N, K, layout):
    """Row blocks that are no whole tiles: the sums over four ranks' partials, each block's rows its own."""
    import tileccl_amd

    ctxs = tileccl_amd.init_local(world_size=4, heap_size=M * N * 8 + (64 << 20))
    data = []
    for r, ctx in enumerate(ctxs):
        heap = ctx.require_heap()
        A, B = operands(M, N, K, torch.float16, layout)
        A = A.roll(r, 0)
        data.append((A, B, heap.allocate_tensor((M, N // 4), torch.float16)))
    for _ in range(2):  # once to produce the partials, once to sum them
        for ctx, (A, B, out) in zip(ctxs, data):
            ops.gemm_reducescatter(A, B, out, ctx=ctx)
    want = sum(A.float() @ B.float() for A, B, _ in data)
    for r, (_, _, out) in enumerate(data):
        torch.testing.assert_close(out.float(), want[:, r * N // 4:(r + 1) * N // 4], rtol=4e-3, atol=8e-3)
