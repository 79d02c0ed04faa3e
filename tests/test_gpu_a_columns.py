"""A given by columns (the `.t()` view of a (K, M) tensor) read in place by the 128-row tile kernels: the bits of the same call on
A's rows, whatever lies behind the operand, on every kernel of that class and through every schedule of the all-scatter."""

import ctypes as C

import pytest
import torch

from tests.gpu_util import assert_gemm_close, bits, seeded

pytestmark = pytest.mark.gpu


def columns(cpu, pitch, behind):
    """`cpu` (M, K) given by columns `pitch` elements apart, everything around it filled with `behind`."""
    whole = torch.full((cpu.shape[1] + 80, pitch), behind, dtype=cpu.dtype, device="cuda")
    view = whole[: cpu.shape[1], : cpu.shape[0]]
    view.copy_(cpu.t())
    return view.t()


# Deep tiles, two workgroups per CU, 128 x 256 tiles; rows and K short of a tile, of a vector, one K step and less.
SHAPES = [(1000, 2064, 1003, 1000), (1544, 2056, 64, 1544), (1032, 2200, 129, 1040), (2056, 1800, 203, 2056), (3000, 2056, 330, 3000),
          (1544, 4104, 7, 1544), (2304, 1032, 1000, 2304)]


@pytest.mark.parametrize("M,N,K,pitch", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_product(lib, M, N, K, pitch, dtype):
    from tileccl_amd import _launch, _lib

    A_cpu, B_cpu = seeded((M, K), 0, dtype), seeded((K, N), 1, dtype, scale=K**-0.5)
    B = B_cpu.cuda()
    rows = torch.empty(M, N, dtype=dtype, device="cuda")
    d = _launch.gemm_desc(A_cpu.cuda(), B, rows)
    _lib.check(lib.tccl_gemm(C.byref(d), _launch.stream_ptr()), "tccl_gemm")
    for behind in (0.0, float("nan")):
        A = columns(A_cpu, pitch, behind)
        got = torch.full((M + 3, N), -7.0, dtype=dtype, device="cuda")
        d, plan = _launch._gemm_desc(A, B, got[:M], a_columns=True)
        assert not plan.pack_a and d.flags & _lib.GEMM_A_COLUMNS
        d.A, d.B = A.data_ptr(), B.data_ptr()
        _lib.check(lib.tccl_gemm(C.byref(d), _launch.stream_ptr()), "tccl_gemm")
        torch.cuda.synchronize()
        assert torch.equal(bits(got[:M]), bits(rows)) and torch.all(got[M:] == -7.0)
    assert_gemm_close(rows, A_cpu.float() @ B_cpu.float())


@pytest.mark.parametrize("schedule", ["bulk_sync", "wg_specialized", "tile_group"])
@pytest.mark.parametrize("M,N,K", [(1000, 2064, 1003), (1032, 4000, 136)])
def test_all_scatter(lib, M, N, K, schedule):
    import tileccl_amd
    from tileccl_amd import ops

    ctxs = tileccl_amd.init_local(world_size=2, heap_size=128 << 20)
    try:
        A_cpu, B_cpu = seeded((M, K), 0, torch.bfloat16), seeded((K, N), 1, torch.bfloat16, scale=K**-0.5)
        heap, outs = ctxs[0].require_heap(), [c.zeros(M, N, dtype=torch.bfloat16) for c in ctxs]
        by_columns = heap.allocate_tensor((K, M), torch.bfloat16)
        by_columns.copy_(A_cpu.t())
        A, B = heap.allocate_tensor((M, K), torch.bfloat16), heap.allocate_tensor((K, N), torch.bfloat16)
        A.copy_(A_cpu)
        B.copy_(B_cpu)
        got = []
        for a in (A, by_columns.t()):
            for o in outs:
                o.zero_()
            ops.gemm_allscatter(a, B, outs[0], ctx=ctxs[0], pattern=schedule)
            torch.cuda.synchronize()
            got.append([bits(o).cpu().clone() for o in outs])
        for x, y in zip(*got):
            assert torch.equal(x, y)
        assert_gemm_close(outs[0], A_cpu.float() @ B_cpu.float())
    finally:
        for c in ctxs:
            c.heap.cleanup()


@pytest.mark.parametrize("in_place_first", [False, True])
def test_all_scatter_into_its_own_input(lib, in_place_first):
    """``C.t() @ B`` into ``C``, beside the same call on tensors that lie apart: A is read before anything is stored."""
    import tileccl_amd
    from tileccl_amd import _launch, ops

    n, dtype = 1040, torch.bfloat16
    ctxs = tileccl_amd.init_local(world_size=2, heap_size=128 << 20)
    try:
        A_cpu, B_cpu = seeded((n, n), 0, dtype), seeded((n, n), 1, dtype, scale=n**-0.5)
        outs, spare = [c.zeros(n, n, dtype=dtype) for c in ctxs], [c.zeros(n, n, dtype=dtype) for c in ctxs]
        B = ctxs[0].zeros(n, n, dtype=dtype)
        B.copy_(B_cpu)
        assert [_launch._gemm_desc(t.t(), B, outs[0], a_columns=True)[1].pack_a for t in (spare[0], outs[0])] == [False, True]
        got = []
        for in_place in (in_place_first, not in_place_first, in_place_first):
            held = outs[0] if in_place else spare[0]
            held.copy_(A_cpu.t())
            ops.gemm_allscatter(held.t(), B, outs[0], ctx=ctxs[0])
            torch.cuda.synchronize()
            got.append([bits(o[:, : n // 2]).cpu().clone() for o in outs])
        for x in got[1:]:
            assert all(torch.equal(a, b) for a, b in zip(x, got[0]))
        assert_gemm_close(outs[0], A_cpu.float() @ B_cpu.float())
    finally:
        for c in ctxs:
            c.heap.cleanup()


def test_all_scatter_from_a_peers_copy_of_its_output(lib):
    """``C.t() @ B`` into ``C`` with the input taken from the other rank's copy, which the launch stores to."""
    import tileccl_amd
    from tileccl_amd import ops

    n, dtype = 1040, torch.bfloat16
    ctxs = tileccl_amd.init_local(world_size=2, heap_size=128 << 20)
    try:
        A_cpu, B_cpu = seeded((n, n), 0, dtype), seeded((n, n), 1, dtype, scale=n**-0.5)
        outs, spare = [c.zeros(n, n, dtype=dtype) for c in ctxs], [c.zeros(n, n, dtype=dtype) for c in ctxs]
        B = ctxs[0].zeros(n, n, dtype=dtype)
        B.copy_(B_cpu)
        assert [ctxs[0].heap.lies_with_a_peer(t) for t in (*outs, B_cpu.cuda())] == [False, True, False]
        got = []
        for held in (spare[0], outs[1], spare[0], outs[1]):
            held.copy_(A_cpu.t())
            ops.gemm_allscatter(held.t(), B, outs[0], ctx=ctxs[0])
            torch.cuda.synchronize()
            got.append([bits(o[:, : n // 2]).cpu().clone() for o in outs])
        for x in got[1:]:
            assert all(torch.equal(a, b) for a, b in zip(x, got[0]))
        assert_gemm_close(outs[0], A_cpu.float() @ B_cpu.float())
    finally:
        for c in ctxs:
            c.heap.cleanup()


@pytest.mark.parametrize("variant", ["s0", "s1", "s2"])
@pytest.mark.parametrize("world,directions,how", [(2, "pull", {}), (2, "both", {}), (2, "push", {"trace": True}), (2, "both", {"trace": True}),
                                                  (3, "push", {"num_gemm_wgs": 40}), (4, "push", {})])
@pytest.mark.parametrize("M,N,K", [(1032, 2056, 203), (1000, 2064, 1003)])
def test_all_gather(lib, monkeypatch, world, directions, how, variant, M, N, K):
    """Pulls beside the GEMM, transfers kept apart by clock stamps, pushes to several peers, workgroups counted by the caller."""
    from functools import partial

    from tileccl_amd import _launch, _lib
    from tileccl_amd.v2 import FusedGemmAllGather, SymmetricHeap

    heaps = SymmetricHeap.create_all(96 << 20, world)
    try:
        ops = [FusedGemmAllGather(h, M, N, torch.bfloat16, directions=directions, **how) for h in heaps]
        A_cpu, B_cpu = seeded((M, K), 0, torch.bfloat16), seeded((K, N), 1, torch.bfloat16, scale=K**-0.5)
        B = B_cpu.cuda()
        given, got = _launch._gemm_desc, []
        assert given(columns(A_cpu, 1040, 0.0), B, ops[0].local_block, a_columns=True)[0].flags & _lib.GEMM_A_COLUMNS
        for A, in_place in ((A_cpu.cuda(), False), (columns(A_cpu, 1040, float("nan")), True)):
            monkeypatch.setattr(_launch, "_gemm_desc", partial(given, a_columns=in_place))
            for r, op in enumerate(ops):
                op.out.zero_()
                op.local_block.copy_(seeded((M, N), 5 + r, torch.bfloat16))
            ops[0].mark_peers_ready()
            ops[0](A, B, variant)
            ops[0].check_faults()
            torch.cuda.synchronize()
            got.append([bits(op.out).cpu().clone() for op in ops])
        for x, y in zip(*got):
            assert torch.equal(x, y)
        assert_gemm_close(ops[0].local_block, A_cpu.float() @ B_cpu.float())
    finally:
        for h in heaps:
            h.cleanup()


def test_refusals(lib):
    from tileccl_amd import _launch, _lib

    A, B = torch.zeros(256, 512, device="cuda", dtype=torch.float16).t(), torch.zeros(256, 1024, device="cuda", dtype=torch.float16)
    out = torch.zeros(512, 1024, device="cuda", dtype=torch.float16)
    d, _ = _launch._gemm_desc(A, B, out, flags=_lib.GEMM_A_COLUMNS)
    d.A, d.B, d.lda = A.data_ptr(), B.data_ptr(), 512
    assert lib.tccl_gemm(C.byref(d), _launch.stream_ptr()) == 0
    for field, value in (("macro_tile", 256), ("lda", 504), ("M", 500), ("flags", d.flags | _lib.GEMM_B_KMAJOR), ("flags", d.flags | 8 << _lib.GEMM_A_SHORT_SHIFT)):
        kept = getattr(d, field)
        setattr(d, field, value)
        assert lib.tccl_gemm(C.byref(d), _launch.stream_ptr()) != 0, field
        setattr(d, field, kept)
    torch.cuda.synchronize()
