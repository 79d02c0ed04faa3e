"""Reduce-scatters of column shards whose sub-tiles run across the owners: every workgroup has a part of this rank's columns
and sums it behind its own product.

The sums are made in fp32 from the partials, owner first, the others ascending, and rounded once: bit for bit what the oracle
makes of the partials, this rank's as the launch with stored partials leaves it."""

import pytest
import torch

import tileccl_amd as tileccl
from oracle import collectives as oracle
from tests.gpu_util import assert_gemm_close, bits, seeded

pytestmark = pytest.mark.gpu


# Of fp32 partials: K roundings of sums of a few units, sqrt(6152) * 2^-24 * 5 = 2.4e-5 on either side, with room for the largest of two
# million; a product left out (K^-0.5 in size, 0.013 at the longest K) shows.
TIGHT = 1e-3


def reduce(world, rank, M, N, K, dtype, kmajor, variant, own, launches=1, spoil=None):
    """(out, this rank's partial as (world, M, N / world), A @ B, the peers' partials) after `launches` launches."""
    ctxs = tileccl.init_local(world_size=world, heap_size=128 << 20)
    try:
        A_cpu, B_cpu = seeded((M, K), 0, dtype), seeded((K, N), 1, dtype, scale=K**-0.5)
        # (every rank allocates the same things in the same order: the workspaces sit at the same offset)
        operands = [(c.zeros(M, K, dtype=dtype), c.zeros(N, K, dtype=dtype).t() if kmajor else c.zeros(K, N, dtype=dtype),
                     c.zeros(M, N // world, dtype=dtype)) for c in ctxs]
        ctx, (A, B, out) = ctxs[rank], operands[rank]
        A.copy_(A_cpu)
        B.copy_(B_cpu)
        peers = {}
        for p, c in enumerate(ctxs):  # the order of the sums matters
            part = c.workspace("gemm_reducescatter.partial", world, M, N // world, dtype=torch.float32)
            part.fill_(-7.0)
            if p != rank:
                peers[p] = seeded((world, M, N // world), 10 + p, torch.float32) * 1000.0
                if spoil is not None:
                    spoil(p, peers[p])
                part.copy_(peers[p])
        got = []
        for _ in range(launches):
            out.zero_()
            tileccl.ops.gemm_reducescatter(A, B, out, ctx=ctx, variant=variant, own_rows_in_registers=own)
            torch.cuda.synchronize()
            got.append(out.cpu().clone())
        assert all(torch.equal(bits(o), bits(got[0])) for o in got)
        partial = ctx.workspace("gemm_reducescatter.partial", world, M, N // world, dtype=torch.float32).cpu().clone()
        return got[0], partial, A_cpu.float() @ B_cpu.float(), peers
    finally:
        for c in ctxs:
            c.heap.cleanup()


# Last columns in the first and in a later run of a tile, runs of a tile that do not exist, a last tile of few rows.
SHAPES = [
    (2, 0, 1024, 2 * 776, 1160, torch.float16),
    (2, 1, 1000, 2 * 904, 1032, torch.bfloat16),
    (4, 0, 768, 4 * 648, 1160, torch.bfloat16),
    (4, 2, 640, 4 * 848, 1480, torch.float16),
    (4, 3, 700, 4 * 712, 1032, torch.float16),
    (4, 1, 513, 4 * 1024, 2048, torch.bfloat16),
    (8, 1, 256, 8 * 776, 1096, torch.float16),
    (8, 6, 330, 8 * 776, 1032, torch.bfloat16),
    # (few K steps: the costs name the five-stage kernel)
    (2, 1, 1920, 2 * 752, 264, torch.bfloat16),
    (4, 3, 512, 4 * 1568, 200, torch.float16),
    (8, 5, 1000, 8 * 504, 360, torch.bfloat16),
]


@pytest.mark.parametrize("kmajor", [False, True])
@pytest.mark.parametrize("variant", ["s1", "s2"])
@pytest.mark.parametrize("world,rank,M,N,K,dtype", SHAPES)
def test_sums_are_the_oracles(lib, world, rank, M, N, K, dtype, kmajor, variant):
    out, partial, want, peers = reduce(world, rank, M, N, K, dtype, kmajor, variant, own=False, launches=2)
    cols = N // world
    assert_gemm_close(torch.cat(list(partial), 1), want, tight=TIGHT)
    partials = [partial if p == rank else peers[p] for p in range(world)]
    tall = [p.reshape(world * M, cols) for p in partials]
    assert torch.equal(bits(out), bits(oracle.reduce_rows(tall, rank, dtype)))
    kept, registers, _, _ = reduce(world, rank, M, N, K, dtype, kmajor, variant, own=True)
    assert torch.equal(bits(kept), bits(out))
    others = [q for q in range(world) if q != rank]
    assert torch.equal(registers[others], partial[others])
    if kmajor or world < 8:  # (a row-major B on eight ranks keeps the reduction of its own, which reads a stored partial)
        assert torch.all(registers[rank] == -7.0)


@pytest.mark.parametrize("kmajor", [False, True])
@pytest.mark.parametrize("world,rank,M,N,K,dtype", [SHAPES[1], SHAPES[2], SHAPES[4], SHAPES[6], SHAPES[7]])
def test_only_this_ranks_block_is_added(lib, world, rank, M, N, K, dtype, kmajor):
    """Infinities and NaN in this rank's block of the peers' partials come out as the oracle's sums; those of the other blocks,
    right before and behind it, are never read."""

    def spoil(p, partial):
        partial[[q for q in range(world) if q != rank]] = float("nan")
        partial[rank, p % M, ::3] = float("inf")
        partial[rank, (7 * p + 64) % M, 1::3] = float("-inf")
        partial[rank, -1, p::9] = float("nan")
        partial[rank, -1, -1 - p] = float("-inf")

    out, partial, _, peers = reduce(world, rank, M, N, K, dtype, kmajor, "s2", own=False, spoil=spoil)
    want = oracle.reduce_rows([(partial if p == rank else peers[p]).reshape(world * M, N // world) for p in range(world)], rank, dtype)
    assert torch.equal(out.isnan(), want.isnan()) and 0 < int(out.isnan().sum()) < out.numel() // 8
    assert torch.equal(bits(out)[~out.isnan()], bits(want)[~want.isnan()])
    kept, _, _, _ = reduce(world, rank, M, N, K, dtype, kmajor, "s1", own=True, spoil=spoil)
    assert torch.equal(kept.isnan(), want.isnan()) and torch.equal(bits(kept)[~kept.isnan()], bits(want)[~want.isnan()])


@pytest.mark.parametrize("world,rank,M,N,K,kmajor", [(2, 1, 1000, 2 * 904, 1032, False), (4, 3, 700, 4 * 712, 1032, True), (2, 0, 1024, 2 * 776, 1160, False),
                                                     (2, 1, 24, 2 * 512, 512, True)])
def test_the_bulk_schedule_stores_every_partial(lib, world, rank, M, N, K, kmajor):
    """Whatever the shards' rows and kernel: the flag that keeps this rank's block in registers is one of the fused schedules."""
    got = {}
    for variant, own in (("s0", False), ("s0", True), ("s1", True), ("s2", True)):
        got[variant, own] = reduce(world, rank, M, N, K, torch.bfloat16, kmajor, variant, own)[:2]
    out, partial = got["s0", False]
    for kept, registers in got.values():
        assert torch.equal(bits(kept), bits(out))
    assert torch.equal(got["s0", True][1], partial)
    others = [q for q in range(world) if q != rank]
    for variant in ("s1", "s2"):
        assert torch.equal(got[variant, True][1][others], partial[others]) and torch.all(got[variant, True][1][rank] == -7.0)


@pytest.mark.parametrize("world,rank,M,cols,K,kmajor,across", [
    (4, 1, 1024, 704, 2048, False, True), (4, 1, 1024, 704, 2056, False, False), (4, 2, 700, 736, 1792, False, True),
    (4, 2, 700, 736, 1800, False, False), (4, 3, 1000, 648, 1280, False, True), (4, 3, 1000, 648, 1312, False, False),
    (4, 0, 1000, 648, 1528, False, True), (4, 0, 1000, 648, 1544, False, False), (4, 0, 1000, 648, 2048, True, True),
    (2, 1, 1000, 904, 6144, False, True), (2, 1, 1000, 904, 6152, False, False), (2, 1, 1000, 928, 6152, False, True)])
def test_longest_k_of_a_row_major_b(lib, world, rank, M, cols, K, kmajor, across):
    """Beyond it the runs of B cost more than the second launch, which reads a stored partial: the sums are the same."""
    for own in (False, True):
        out, partial, want, peers = reduce(world, rank, M, world * cols, K, torch.bfloat16, kmajor, "s2", own)
        assert torch.all(partial[rank] == -7.0) == (across and own)
        if not own:
            tall = [(partial if p == rank else peers[p]).reshape(world * M, cols) for p in range(world)]
            sums = oracle.reduce_rows(tall, rank, torch.bfloat16)
            assert_gemm_close(torch.cat(list(partial), 1), want, tight=TIGHT)
        assert torch.equal(bits(out), bits(sums))


@pytest.mark.parametrize("kmajor", [False, True])
@pytest.mark.parametrize("where", ["A", "B", "behind A", "C"])
@pytest.mark.parametrize("world,M,K", [(2, 1024, 776), (4, 700, 648)])
def test_output_in_an_operands_memory(lib, world, M, K, where, kmajor):
    """A square layer in place: nothing is stored to memory that the product still reads, nor to that of another owner's partial, which it
    still writes.  The GEMM and the reduction behind it store this rank's partial, the sums in the GEMM's epilogue do not."""
    dtype, cols = torch.bfloat16, K
    ctxs = tileccl.init_local(world_size=world, heap_size=128 << 20)
    try:
        ctx = ctxs[0]
        A_cpu, B_cpu = seeded((M, K), 0, dtype), seeded((K, world * cols), 1, dtype, scale=K**-0.5)
        room = ctx.zeros(2 * M, K, dtype=dtype)
        A, apart = room[:M], ctx.zeros(M, cols, dtype=dtype)
        B = ctx.zeros(world * cols, K, dtype=dtype).t() if kmajor else ctx.zeros(K, world * cols, dtype=dtype)
        part = ctx.workspace("gemm_reducescatter.partial", world, M, cols, dtype=torch.float32)
        stored = B.t() if kmajor else B
        out = {"A": A, "B": stored.reshape(-1)[: M * cols].view(M, cols), "behind A": room[M:], "C": part[1].view(dtype).reshape(-1)[: M * cols].view(M, cols)}[where]
        got = []
        for o in (apart, out):
            A.copy_(A_cpu)
            B.copy_(B_cpu)
            part.fill_(-7.0)
            tileccl.ops.gemm_reducescatter(A, B, o, ctx=ctx)
            torch.cuda.synchronize()
            got.append((bits(o).cpu().clone(), bool(torch.all(part[0] == -7.0))))
        assert torch.equal(got[0][0], got[1][0])
        assert got[0][1] and got[1][1] == (where == "behind A")
    finally:
        for c in ctxs:
            c.heap.cleanup()


def test_every_plan_tile_is_published_once(lib):
    """The words that the peers of the next launch look at: locks hold the launch's number, counters all tiles of every launch,
    and the arrival words are zero again."""
    from tileccl_amd import ops_collective

    M, cols, K, world = 384, 904, 1032, 4
    ctxs = tileccl.init_local(world_size=world, heap_size=128 << 20)
    try:
        A, B = ctxs[0].zeros(M, K, dtype=torch.float16), ctxs[0].zeros(world * cols, K, dtype=torch.float16).t()
        out = ctxs[0].zeros(M, cols, dtype=torch.float16)
        words = ops_collective._reduce_scatter_words(ctxs[0], world, M, cols)
        counts = words.host_plan.tile_counts()
        for launch in (1, 2, 3):
            for variant in ("s1", "s2"):
                tileccl.ops.gemm_reducescatter(A, B, out, ctx=ctxs[0], variant=variant)
            torch.cuda.synchronize()
            assert torch.all(words.locks == launch)
            assert words.counter.tolist() == [launch * int(c) for c in counts]
            assert torch.all(words.arrivals == 0)
    finally:
        for c in ctxs:
            c.heap.cleanup()


@pytest.mark.parametrize("variant", ["s1", "s2"])
@pytest.mark.parametrize("world,kmajor", [(4, False), (8, True)])
def test_two_streams_and_a_recorded_graph(lib, world, kmajor, variant):
    """Launches that overlap count in the same lines of arrival words; a recorded launch counts in the word it was recorded with,
    between eager ones.  All leave the words zero, every plan tile published once by each, and the sums of one launch alone."""
    from tileccl_amd import ops_collective

    M, cols, K = 384, 904, 1032
    ctxs = tileccl.init_local(world_size=world, heap_size=128 << 20)
    try:
        ctx = ctxs[0]
        A = ctx.zeros(M, K, dtype=torch.float16)
        B = ctx.zeros(world * cols, K, dtype=torch.float16).t() if kmajor else ctx.zeros(K, world * cols, dtype=torch.float16)
        A.copy_(seeded((M, K), 0))
        B.copy_(seeded((K, world * cols), 1, scale=K**-0.5))
        outs = [ctx.zeros(M, cols, dtype=torch.float16) for _ in range(3)]
        for p, c in enumerate(ctxs):
            c.workspace("gemm_reducescatter.partial", world, M, cols, dtype=torch.float32).copy_(seeded((world, M, cols), 10 + p, torch.float32))
        call = lambda out: tileccl.ops.gemm_reducescatter(A, B, out, ctx=ctx, variant=variant)
        call(outs[2])
        torch.cuda.synchronize()
        alone = outs[2].clone()
        words = ops_collective._reduce_scatter_words(ctx, world, M, cols)

        def check(launches, which):
            torch.cuda.synchronize()
            assert all(torch.equal(bits(outs[i]), bits(alone)) for i in which)
            assert not words.arrivals.any()
            if variant == "s2":
                assert words.counter.tolist() == [launches * int(c) for c in words.host_plan.tile_counts()]
            for o in outs:
                o.zero_()
            torch.cuda.synchronize()

        streams = [torch.cuda.Stream() for _ in range(2)]
        for _ in range(20):
            for out, stream in zip(outs, streams):
                with torch.cuda.stream(stream):
                    call(out)
        check(41, (0, 1))
        graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
            call(outs[0])
        for _ in range(4):  # (from here on every launch starts from cleared counters: SyncWords)
            graph.replay()
            call(outs[1])
            check(1, (0, 1))
            assert (torch.randn(256, 256, device="cuda") @ torch.randn(256, 256, device="cuda")).isfinite().all()
    finally:
        for c in ctxs:
            c.heap.cleanup()
