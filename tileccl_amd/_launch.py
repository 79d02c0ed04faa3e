"""Marshalling between torch tensors and the C ABI descriptors.

Everything here is host bookkeeping: it validates what the kernels assume (contiguity,
dtypes, device) and hands raw device pointers down.  The launches go to torch's current
stream, like the reference's Triton launches do.
"""

from __future__ import annotations

import ctypes as C
import sys
from dataclasses import dataclass, replace
from functools import partial

import torch

from tileccl_amd import _lib

_DTYPE_CODES = {
    torch.float16: _lib.F16,
    torch.bfloat16: _lib.BF16,
    torch.float32: _lib.F32,
}
if hasattr(torch, "float8_e4m3fn"):
    _DTYPE_CODES[torch.float8_e4m3fn] = _lib.F8E4M3

VARIANTS = {"s0": _lib.S0_BULK, "s1": _lib.S1_TILE, "s2": _lib.S2_TILEGROUP}
DEFAULT_SPIN_LIMIT_NS = 2_000_000_000


def dtype_code(dtype: torch.dtype) -> int:
    try:
        return _DTYPE_CODES[dtype]
    except KeyError:
        raise ValueError(f"dtype {dtype} is not supported by the HIP kernels") from None


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def stream_ptr() -> int:
    """torch's current stream on the heap's device as a ``hipStream_t`` value.  The raw accessor
    costs well under a microsecond; building a ``torch.cuda.Stream`` object costs ~9 us, a fifth
    of a c1-sized launch."""
    if _raw_stream is not None:
        return int(_raw_stream(0))  # every emulated rank lives on device 0
    return int(torch.cuda.current_stream().cuda_stream)


def ptr(t: torch.Tensor | None) -> int | None:
    return None if t is None else int(t.data_ptr())


def _row_major(t: torch.Tensor, name: str) -> int:
    """Leading dimension of a 2-D tensor whose rows are contiguous."""
    if t.ndim != 2:
        raise ValueError(f"{name} must be 2-D, got {t.ndim}-D")
    if t.shape[1] > 1 and t.stride(1) != 1:
        raise ValueError(
            f"{name} must have contiguous rows (stride(1) == 1), got strides {tuple(t.stride())}; "
            "call .contiguous() first"
        )
    return int(t.stride(0)) if t.shape[0] > 1 else int(t.shape[1])


def _vector_elems(t: torch.Tensor) -> int:
    return 16 // t.element_size()


def _rows_vectorised(t: torch.Tensor, ld: int) -> bool:
    """Rows of pitch ``ld`` start on 16-byte boundaries (what the kernels' row vectors need)."""
    return t.data_ptr() % 16 == 0 and ld % _vector_elems(t) == 0


def _b_layout(B: torch.Tensor) -> tuple[int, int] | None:
    """(ldb, flag bits) of a B operand the kernels read in place: rows contiguous, or the ``.t()``
    view of a tensor whose rows are contiguous (k-major: the layout of a linear layer's weight).
    ``None`` for every other layout; the reference's kernels take any strides
    (``/root/reference/tileccl/kernels/gemm.py:139-151``) and these are the two forms with 16-byte
    vector access."""
    K, N = B.shape
    if N == 1 or B.stride(1) == 1:
        ld = int(B.stride(0)) if K > 1 else int(N)
        return (ld, 0) if ld >= N and _rows_vectorised(B, ld) else None
    if K == 1 or B.stride(0) == 1:
        ld = int(B.stride(1)) if N > 1 else int(K)
        return (ld, _lib.GEMM_B_KMAJOR) if ld >= K and _rows_vectorised(B, ld) else None
    return None


_PACKED: dict[tuple, torch.Tensor] = {}
_PACKED_LIMIT = 8


def _pack_buffer(t: torch.Tensor, rows: int, cols: int, role: str, stream: int) -> torch.Tensor:
    """A dense ``rows x cols`` buffer, kept per (role, shape, dtype, stream) and reused by the next call with that key, which
    the stream orders behind this one's GEMM, unless a descriptor that has not been dropped yet still points at it.  A call that
    is being recorded into a graph takes one from the graph's memory: a kept one might be dropped, and its memory be someone
    else's, while the graph goes on writing it."""
    if torch.cuda.is_current_stream_capturing():
        return torch.empty((rows, cols), dtype=t.dtype, device=t.device)
    key = (role, rows, cols, t.dtype, t.device, stream)
    out = _PACKED.pop(key, None)
    if out is not None and sys.getrefcount(out) > 2:  # this name and the call's argument
        out = None
    if out is None:
        while len(_PACKED) >= _PACKED_LIMIT:
            _PACKED.pop(next(iter(_PACKED)))
        out = torch.empty((rows, cols), dtype=t.dtype, device=t.device)
    _PACKED[key] = out  # most recently used last
    return out


def _pack(jobs: "list[tuple[torch.Tensor, int, int, str]]") -> "list[torch.Tensor]":
    """Each (tensor, rows, cols, role) as a dense ``rows x cols`` matrix, zero beyond the tensor's own shape: one
    launch on the current stream."""
    stream = stream_ptr()
    descs = (_lib.PackDesc * len(jobs))()
    outs = []
    for d, (t, rows, cols, role) in zip(descs, jobs):
        out = _pack_buffer(t, rows, cols, role, stream)
        d.src, d.dst = t.data_ptr(), out.data_ptr()
        d.stride_row, d.stride_col = t.stride()
        d.ld_dst = cols
        d.rows, d.cols = t.shape
        d.dst_rows, d.dst_cols = rows, cols
        outs.append(out)
    rc = _lib.load().tccl_pack_matrices(descs, len(jobs), outs[0].element_size(), stream)
    if rc:
        _lib.check(rc, "tccl_pack_matrices")
    return outs


@dataclass(frozen=True, slots=True)
class OperandPlan:
    """How the kernels read A and B of one layout: in place, or from packed copies."""

    pack_a: bool
    pack_b: bool
    K: int  # zero-filled up to whole 16-byte vectors where an operand is packed
    lda: int
    ldb: int
    b_flags: int


def operand_plan(A: torch.Tensor, B: torch.Tensor) -> OperandPlan:
    """An operand the kernels can address in place (16-byte row vectors: A with contiguous rows, B with contiguous rows
    or columns, K a whole number of vectors) is passed through; any other layout the reference's pointer arithmetic accepts
    (``/root/reference/tileccl/kernels/gemm.py:63-66,139-151``: a transposed A, strided slices, odd K)
    is packed into a dense buffer first, K zero-filled up to the next whole vector, which adds exact zeros
    to every dot product."""
    for name, t in (("A", A), ("B", B)):
        if t.ndim != 2:
            raise ValueError(f"{name} must be 2-D, got {t.ndim}-D")
        if any(s < 0 for s in t.stride()):
            raise ValueError(f"{name} has negative strides {tuple(t.stride())}")
    M, K = A.shape
    vec = _vector_elems(A)
    k_pad = (K + vec - 1) // vec * vec
    lda = int(A.stride(0)) if M > 1 else int(K)
    pack_a = k_pad != K or (K > 1 and A.stride(1) != 1) or lda < K or not _rows_vectorised(A, lda)
    layout = _b_layout(B)
    if layout is not None and k_pad != K:  # a row-major B need not have the rows that A is filled up with
        layout = (layout[0], (k_pad - K) << _lib.GEMM_B_SHORT_SHIFT) if not layout[1] else None
    ldb, flags = layout or (int(B.shape[1]), 0)
    # A packed A's rows start on 64-byte boundaries, as its chunks are fetched (1000 x 2064 x 1003, A transposed: 22.3 us with
    # rows of 1008 elements, 20.7 with 1024; whole 128-byte lines give the same).
    line = 4 * vec
    return OperandPlan(pack_a, layout is None, int(k_pad), -(-k_pad // line) * line if pack_a else lda, ldb, flags)


def planned_operands(plan: OperandPlan, A: torch.Tensor, B: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """(A, B) with the operands that ``plan`` says so packed on the current stream."""
    if plan.pack_a and plan.pack_b:
        return tuple(_pack([(A, A.shape[0], plan.lda, "A"), (B, plan.K, B.shape[1], "B")]))
    if plan.pack_a:
        (A,) = _pack([(A, A.shape[0], plan.lda, "A")])
    if plan.pack_b:
        (B,) = _pack([(B, plan.K, B.shape[1], "B")])
    return A, B


def gemm_operands(A: torch.Tensor, B: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor, int, int, int, int]:
    """(A, B, K, lda, ldb, flag bits) as the kernels read them (``operand_plan``), packed where need be."""
    plan = operand_plan(A, B)
    A, B = planned_operands(plan, A, B)
    return A, B, plan.K, plan.lda, plan.ldb, plan.b_flags


def _apart(a: torch.Tensor, b: torch.Tensor) -> bool:
    """No byte from the first to the last element of ``a`` lies among those of ``b``."""
    (a_first, a_end), (b_first, b_end) = (
        (t.data_ptr(), t.data_ptr() + (1 + sum((n - 1) * s for n, s in zip(t.shape, t.stride()))) * t.element_size()) for t in (a, b)
    )
    return a_end <= b_first or b_end <= a_first


def _gemm_desc(
    A: torch.Tensor,
    B: torch.Tensor,
    C_out: torch.Tensor,
    *,
    block_m: int = 128,
    block_n: int = 128,
    group_m: int = 8,
    alpha: float = 1.0,
    num_wgs: int = 0,
    macro_tile: int = 0,
    flags: int = 0,
    column_shards: int = 0,
    a_columns: bool = False,
) -> tuple[_lib.GemmDesc, OperandPlan]:
    """The descriptor without its operands' addresses, and how those are to be read.  ``a_columns``: the operation takes an A
    that is given by columns (a transposed view) where it lies, if C lies elsewhere (``C.t() @ B`` into ``C`` takes a copy of A
    before it stores anything); the kernels that would run decide."""
    if not (A.is_cuda and B.is_cuda and C_out.is_cuda):
        raise ValueError("GEMM operands must be device tensors")
    if A.dtype != B.dtype:
        raise ValueError(f"A and B must share a dtype, got {A.dtype} and {B.dtype}")
    M, K = A.shape
    K2, N = B.shape
    if K2 != K:
        raise ValueError(f"B.shape[0] must equal A.shape[1]: got {K2} vs {K}")
    if column_shards > 1:  # C stacks the column blocks of A @ B as row blocks
        if N % column_shards:
            raise ValueError(f"B.shape[1]={N} must be divisible by column_shards={column_shards}")
        M, N = M * column_shards, N // column_shards
    if tuple(C_out.shape) != (M, N):
        raise ValueError(f"C shape mismatch: expected ({M}, {N}), got {tuple(C_out.shape)}")
    plan = operand_plan(A, B)
    d = _lib.GemmDesc()
    d.C = ptr(C_out)
    d.M, d.N, d.K = int(M), int(N), plan.K
    d.lda, d.ldb, d.ldc = plan.lda, plan.ldb, _row_major(C_out, "C")
    d.in_dtype, d.out_dtype = dtype_code(A.dtype), dtype_code(C_out.dtype)
    d.alpha = float(alpha)
    d.block_m, d.block_n, d.group_m = int(block_m), int(block_n), int(group_m)
    d.num_wgs = int(num_wgs)
    d.macro_tile = int(macro_tile)
    d.flags = int(flags) | plan.b_flags
    d.column_shards = int(column_shards)
    if a_columns and plan.pack_a and not plan.pack_b and M > 1 and A.stride(0) == 1 and _apart(A, C_out):
        pitch = int(A.stride(1)) if K > 1 else int(M)
        if pitch >= M and _rows_vectorised(A, pitch):
            kept = d.lda, d.flags, d.A, d.B
            d.lda, d.flags = pitch, d.flags | _lib.GEMM_A_COLUMNS | (plan.K - K) << _lib.GEMM_A_SHORT_SHIFT
            d.A, d.B = A.data_ptr(), B.data_ptr()
            taken = _lib.load().tccl_gemm_reads_columns(C.byref(d))
            d.A, d.B = kept[2:]
            if taken:
                plan = replace(plan, pack_a=False, lda=pitch)
            else:
                d.lda, d.flags = kept[:2]
    return d, plan


def gemm_desc(A: torch.Tensor, B: torch.Tensor, C_out: torch.Tensor, **how) -> _lib.GemmDesc:
    """The descriptor of ``C_out = A @ B`` (keywords: ``_gemm_desc``), operands packed where need be."""
    d, plan = _gemm_desc(A, B, C_out, **how)
    A, B = planned_operands(plan, A, B)
    d.operands = (A, B)  # a packed operand lives as long as the descriptor
    d.A, d.B = ptr(A), ptr(B)
    return d


_ENTRIES: dict[str, tuple] = {}  # an operation's entry point and its address
SYNC = object()  # stands for the sync descriptor in the arguments of a bound call


def call_table(owner: dict):
    """The bound calls kept with ``owner`` (a heap's or an operation's ``__dict__``, a context's workspaces): at most 1024, some
    2 KiB each.  A program that goes round more layouts than that (of row counts, of gradient buckets) binds every call anew."""
    table = owner.get("tileccl_amd.calls")
    if table is None:
        table = owner["tileccl_amd.calls"] = _lib.host().Table(1024)
    return table


def bind(table, key: tuple, tensors: tuple, fn, args: tuple, what: str, *, gemm: _lib.GemmDesc | None = None,
         plan: "OperandPlan | None" = None, words: "SyncWords | None" = None, variant: str = "s0", tag=None, c=None, heap=None,
         on_heap: int | None = None, bases=None) -> None:
    """Keep a checked call for tensors laid out like ``tensors``: ``table.launch(key, alpha, *tensors)`` issues ``fn(*args, stream)``
    and returns ``tag`` (``True`` by default); it returns ``None`` where no call of the table fits.

    In ``args``, ``gemm`` stands for a copy of that descriptor with the addresses of the first two tensors as A and B (packed
    first where ``plan`` says so) and, with ``c=(i, offset)``, tensor ``i``'s as C; ``SYNC`` for ``words``' descriptor with
    the launch's number; ``(i, offset)`` for the address of tensor ``i``; other descriptors are passed as they are.
    The tensors of the bit mask ``on_heap`` (default: all) must start inside ``heap``; with ``bases`` all tensors must lie at
    one distance from their base.  An A that is read by columns lies apart from C and, with ``heap``, in no other rank's.
    Tensors for which that does not hold find no call."""
    host = _lib.host()
    entry = _ENTRIES.get(what)
    if entry is None or entry[0] is not fn:
        entry = _ENTRIES[what] = fn, C.cast(fn, C.c_void_p).value
    keep = [words]  # what the descriptors point at lives as long as the call
    passed = []
    for a in args:
        if a is gemm and a is not None:
            a = host.GEMM
        elif a is SYNC:
            a = None if words is None else host.SYNC
        elif isinstance(a, C.Structure):
            keep.append(a)
            a = C.addressof(a)
        passed.append(a)
    sync = None if words is None else words.desc(variant)
    packs = plan is not None and (plan.pack_a or plan.pack_b)
    by_columns = gemm is not None and gemm.flags & _lib.GEMM_A_COLUMNS
    table.add(host.Call(
        entry[1], what, tuple(passed), tensors, key, tag=tag, gemm=0 if gemm is None else C.addressof(gemm), c=c,
        sync=0 if sync is None else C.addressof(sync), words=words, variant=variant, on_heap=on_heap,
        heap=None if heap is None else (heap.local_base, heap.size, *(heap.all_ranks if by_columns else ())), bases=bases,
        prepare=partial(planned_operands, plan) if packs else None, keep=keep,
    ))


def issue(table, key: tuple, alpha, *tensors):
    """Launch a call that has just been bound."""
    tag = table.launch(key, alpha, *tensors)
    if tag is None:
        raise RuntimeError(f"the call bound as {key} does not fit the tensors it was made for")
    return tag


def view_of(heap) -> _lib.HeapView:
    """The heap's view descriptor, built once per heap (kernels only read it)."""
    view = heap.__dict__.get("_view_desc")
    bases = heap.get_heap_bases()  # raises once the heap has been cleaned up
    if view is None:
        view = heap.__dict__["_view_desc"] = heap_view(bases, heap.rank, heap.world_size)
        view.bases = bases  # lives as long as a descriptor that names it
    return view


def heap_view(heap_bases: torch.Tensor, rank: int, world_size: int) -> _lib.HeapView:
    v = _lib.HeapView()
    v.heap_bases = ptr(heap_bases)
    v.rank, v.world_size = int(rank), int(world_size)
    return v


def transport_desc(directions: int, copy_elems: int, reduce_elems: int | None, num_comm_wgs: int) -> _lib.TransportDesc:
    t = _lib.TransportDesc()
    t.directions = int(directions)
    t.copy_elems = int(copy_elems)
    t.reduce_elems = int(reduce_elems or 0)
    t.num_comm_wgs = int(num_comm_wgs)
    return t


@dataclass(frozen=True)
class DevicePlan:
    """Device-resident copy of a ``TileGroupPlan``'s vectors (uploaded once per plan)."""

    n_groups: int
    group_table: torch.Tensor
    row_starts: torch.Tensor
    row_ends: torch.Tensor
    tile_counts: torch.Tensor

    @classmethod
    def upload(cls, plan, device: str = "cuda:0") -> "DevicePlan":
        def dev(values) -> torch.Tensor:
            return torch.tensor(list(values), dtype=torch.int32, device=device)

        return cls(
            n_groups=plan.n_groups,
            group_table=plan.group_table.to(device=device, dtype=torch.int32).contiguous(),
            row_starts=dev(plan.row_starts()),
            row_ends=dev(plan.row_ends()),
            tile_counts=dev(plan.tile_counts()),
        )


@dataclass(init=False)
class SyncWords:
    """Signal words of one fused operation plus the launch epoch.

    Counters grow monotonically: TileGroup launch ``e`` (1-based) treats group ``g`` as ready
    at ``counter[g] >= e * tile_counts[g]``, and tile-by-tile launch ``e`` stores ``e`` into
    ``locks[tile]`` and treats a tile as ready at ``locks[tile] >= e``, so repeated launches
    need no reset kernel and a flag of an earlier launch is never mistaken for this one's.
    The two kinds of launch count separately (``epoch`` / ``lock_epoch``): each numbers the
    launches that wrote its own words.  Ranks that wait on each other's words must have issued
    the same number of launches.  ``reset()`` zeroes the words and restarts both numbers,
    which is also what happens automatically before the 32-bit words could overflow.

    A launch recorded into a HIP graph replays with the arguments it was recorded with, so
    its epoch cannot advance.  A TileGroup launch issued while the stream is capturing is
    therefore preceded by fill kernels that clear the counters (recorded with it; never a
    memset node) and runs as epoch 1; from then on every launch of these words does the
    same, captured or not, so replays and eager launches can alternate freely (one after the
    other: what clears the words for one launch takes them from another that is still running).

    Launches that overlap on two streams count their tiles in arrival words of their own
    (``ARRIVAL_STRIDE / 2`` launch numbers in turn).
    """

    locks: torch.Tensor | None = None
    counter: torch.Tensor | None = None
    barrier: torch.Tensor | None = None
    plan: DevicePlan | None = None
    host_plan: object | None = None  # the TileGroupPlan `plan` was uploaded from
    trace_comm_counter: torch.Tensor | None = None
    trace_start_clock: torch.Tensor | None = None
    trace_ready_clock: torch.Tensor | None = None
    trace_done_clock: torch.Tensor | None = None
    fault: torch.Tensor | None = None  # made by the constructor unless it is given one
    epoch: int = 0
    lock_epoch: int = 0
    spin_limit_ns: int = DEFAULT_SPIN_LIMIT_NS
    max_tasks_per_tile: int = 1 << 16
    arrivals: torch.Tensor | None = None  # counters, zero between launches (tccl_sync_desc_arrivals)
    arrivals_from_capture: bool = False  # zeroed by a recorded fill only: every launch has to clear them itself
    clear_every_launch: bool = False  # set by the first launch recorded into a graph
    revision: int = 0  # grows with every change of what the descriptor holds: calls bound with an earlier one are built again

    _DESCRIBED = frozenset(("locks", "counter", "barrier", "plan", "fault", "arrivals", "trace_comm_counter", "trace_start_clock",
                            "trace_ready_clock", "trace_done_clock"))

    def __init__(self, **given) -> None:
        unknown = given.keys() - self.__dataclass_fields__.keys()
        if unknown:
            raise TypeError(f"SyncWords has no {', '.join(sorted(unknown))}")
        if given.get("fault") is None:
            given["fault"] = torch.zeros(1, dtype=torch.int64, device="cuda:0")
        mine = self.__dict__  # (field by field, counting changes, it took 8 us)
        mine.update(epoch=0, lock_epoch=0, spin_limit_ns=DEFAULT_SPIN_LIMIT_NS, max_tasks_per_tile=1 << 16, clear_every_launch=False, revision=0)
        mine.update(given)

    def __setattr__(self, name: str, value) -> None:
        self.__dict__[name] = value
        if name in SyncWords._DESCRIBED:
            self.__dict__["revision"] = self.revision + 1

    def reset(self) -> None:
        for t in (self.locks, self.counter, self.barrier, self.arrivals, self.trace_comm_counter, self.trace_start_clock,
                  self.trace_ready_clock, self.trace_done_clock, self.fault):
            if t is not None:
                t.zero_()
        self.epoch = 0
        self.lock_epoch = 0

    def next_epoch(self, variant: str = "s2") -> int:
        """Number the launch about to be issued: ``"s2"`` advances ``epoch``, ``"s1"`` ``lock_epoch``."""
        tile_by_tile = variant == "s1"
        if self.clear_every_launch or torch.cuda.is_current_stream_capturing():
            self.clear_every_launch = True
            for t in (self.locks, self.counter, self.barrier, self.arrivals if self.arrivals_from_capture else None):
                if t is not None:
                    t.zero_()
            self.epoch = self.lock_epoch = 0
        elif max(self.epoch, self.lock_epoch) >= (1 << 30) // self.max_tasks_per_tile:
            torch.cuda.current_stream().synchronize()
            self.reset()
        if tile_by_tile:
            self.lock_epoch += 1
            return self.lock_epoch
        self.epoch += 1
        return self.epoch

    @classmethod
    def made(cls, host_plan=None, **words) -> "SyncWords":
        """Words cleared on the current stream (``words``), with what goes with them.  Another stream's launch may use them
        next: they are clear for every stream when this returns (but for words made while a stream is capturing)."""
        made = cls(host_plan=host_plan, **words)
        made.tile_arrivals()
        if host_plan is not None:
            made.plan = DevicePlan.upload(host_plan)  # copies from host memory, which wait for the stream
        elif not torch.cuda.is_current_stream_capturing():
            torch.cuda.current_stream().synchronize()
        return made

    def tile_arrivals(self) -> torch.Tensor:
        """The arrival counters, made on first use for every plan tile these words have signals for."""
        if self.arrivals is None:
            plan = self.plan or self.host_plan
            tiles = max(int(t.numel()) for t in (self.locks, plan.group_table if plan is not None else None) if t is not None)
            self.arrivals_from_capture = torch.cuda.is_current_stream_capturing()
            self.arrivals = torch.zeros(tiles * _lib.ARRIVAL_STRIDE, dtype=torch.int32, device="cuda:0")
        return self.arrivals

    def desc(self, variant: str = "s2") -> _lib.SyncDescArrivals:
        s = _lib.SyncDescArrivals()
        s.arrivals = ptr(self.tile_arrivals())
        s.locks = ptr(self.locks)
        s.counter = ptr(self.counter)
        s.barrier = ptr(self.barrier)
        if self.plan is not None:
            s.group_table = ptr(self.plan.group_table)
            s.row_starts = ptr(self.plan.row_starts)
            s.row_ends = ptr(self.plan.row_ends)
            s.tile_counts = ptr(self.plan.tile_counts)
            s.n_groups = self.plan.n_groups
        s.epoch = max(self.lock_epoch if variant == "s1" else self.epoch, 1)
        s.trace_comm_counter = ptr(self.trace_comm_counter)
        s.trace_start_clock = ptr(self.trace_start_clock)
        s.trace_ready_clock = ptr(self.trace_ready_clock)
        s.trace_done_clock = ptr(self.trace_done_clock)
        s.fault = ptr(self.fault)
        s.spin_limit_ns = int(self.spin_limit_ns)
        return s

    def raise_if_faulted(self) -> None:
        """Synchronises the stream; raises if a device-side wait ran into its deadline."""
        torch.cuda.current_stream().synchronize()
        if int(self.fault.item()) != 0:
            self.fault.zero_()
            raise RuntimeError(
                "a communication workgroup gave up waiting for a tile/TileGroup signal "
                f"(spin limit {self.spin_limit_ns} ns); the output of this launch is incomplete"
            )


def byref(x):
    return C.byref(x) if x is not None else None
