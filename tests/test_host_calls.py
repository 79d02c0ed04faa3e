"""Bound calls (``_launch.bind`` / ``_host.Table``): which tensors find a call, and what the entry point is given."""

import ctypes as C

import pytest
import torch

from tileccl_amd import _launch, _lib

ENTRY = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_int32, C.c_void_p, C.c_void_p)


@pytest.fixture
def table(lib):
    host = _lib.host()
    capturing = []
    host.setup(lambda device: 0x5000 + device, lambda: bool(capturing), _lib.check)
    yield host.Table(), capturing
    _lib._host = None
    _lib.host()  # torch's stream again


class Heap:
    def __init__(self, t, size):
        self.local_base, self.size = t.data_ptr(), size


def bound(table, key, tensors, returns=0, **how):
    seen = []

    @ENTRY
    def entry(a, b, c, stream):
        seen.append((a, b, c, stream))
        return returns

    _launch.bind(table, key, tensors, entry, ((0, 64), -3, (1, 0)), "entry", **how)
    return seen, entry


@pytest.mark.parametrize("change", ["none", "moved", "shape", "strides", "dtype", "alignment", "outside", "key", "count"])
def test_which_tensors_find_a_call(table, change):
    table, _ = table
    buf = torch.zeros(4096, dtype=torch.float32)
    a, b = buf[:64].view(8, 8), buf[64:128].view(8, 8)
    seen, keep = bound(table, ("op", 1, a), (a, b), heap=Heap(buf, 1024), tag="tag")
    key, found = ("op", 1, a), (a, b)
    if change == "moved":
        found = (b, a)
    elif change == "shape":
        found = (a, b[:7])
    elif change == "strides":
        found = (a.t(), b)
    elif change == "dtype":
        found = (a, b.view(torch.int32))
    elif change == "alignment":
        found = (a, buf[65:129].view(8, 8))
    elif change == "outside":
        found = (a, buf[256:320].view(8, 8))  # starts at byte 1024: just past the heap
    elif change == "key":
        key = ("op", 1, a.clone())  # anything but plain values counts by identity
    elif change == "count":
        found = (a,)
    hit = change in ("none", "moved")
    assert table.launch(key, None, *found) == ("tag" if hit else None)
    assert seen == ([(found[0].data_ptr() + 64, -3, found[1].data_ptr(), 0x5000)] if hit else [])
    assert table.launch(("op", 1, a), None, a, "no tensor") is None


def test_one_offset_on_every_rank_and_reported_errors(table):
    table, _ = table
    buf = torch.zeros(256, dtype=torch.float32)
    a, b, off = buf[:64], buf[128:192], buf[132:196]
    seen, keep = bound(table, ("op",), (a, b), bases=[a.data_ptr(), b.data_ptr()])
    assert table.launch(("op",), None, a, off) is None and table.launch(("op",), None, a, b) is True and len(seen) == 1
    _, keep2 = bound(table, ("bad",), (a, b), returns=_lib.ERR_INVALID)
    with pytest.raises(ValueError, match="entry"):
        table.launch(("bad",), None, a, b)


def test_the_table_is_bounded(table):
    table, _ = table
    a = torch.zeros(8)
    keep = [bound(table, ("op", i), (a, a)) for i in range(70)]
    assert len(table) == 64
    assert table.launch(("op", 5), None, a, a) is None and table.launch(("op", 6), None, a, a) is True


@pytest.mark.parametrize("variant,attr", [("s2", "epoch"), ("s1", "lock_epoch"), ("s0", None)])
def test_descriptors_and_launch_numbers(table, variant, attr):
    """The GEMM descriptor gets the operands' addresses and alpha, the sync descriptor the number ``next_epoch`` would give."""
    table, capturing = table

    class Words:
        epoch = lock_epoch = 0
        clear_every_launch = False
        max_tasks_per_tile = 1 << 16
        spin_limit_ns = 77
        asked = 0

        def desc(self, _variant):
            return _lib.SyncDescArrivals(locks=0x1230)

        def next_epoch(self, which):
            assert which == variant
            self.asked += 1
            return 40

    words, seen = Words(), []

    @C.CFUNCTYPE(C.c_int, C.POINTER(_lib.GemmDesc), C.POINTER(_lib.SyncDescArrivals), C.c_void_p)
    def entry(gemm, sync, stream):
        seen.append((gemm[0].A, gemm[0].B, gemm[0].C, gemm[0].M, gemm[0].alpha, sync[0].locks, sync[0].epoch, sync[0].spin_limit_ns))
        return 0

    a, b, c = (torch.zeros(16) for _ in range(3))
    gemm = _lib.GemmDesc(M=5, alpha=1.0)
    _launch.bind(table, ("g",), (a, b, c), entry, (gemm, _launch.SYNC), "g", gemm=gemm, words=words, variant=variant, c=(2, 32))

    def numbers():
        assert table.launch(("g",), 0.5, a, b, c) is True
        assert seen[-1][:6] == (a.data_ptr(), b.data_ptr(), c.data_ptr() + 32, 5, 0.5, 0x1230) and seen[-1][7] == 77
        return seen[-1][6]

    if attr is None:
        assert numbers() == 0 and words.epoch == words.lock_epoch == words.asked == 0
        return
    assert [numbers(), numbers()] == [1, 2] and getattr(words, attr) == 2 and words.asked == 0
    setattr(words, attr, (1 << 14))  # max_tasks_per_tile leaves room for 2**14 launches
    assert numbers() == 40 and words.asked == 1
    setattr(words, attr, 3)
    capturing.append(1)
    assert numbers() == 40 and words.asked == 2


def test_an_a_by_columns_lies_apart_from_c(table):
    """The launch reads it while it stores C: tensors that share memory find no such call (and one that packs A is built for them)."""
    table, _ = table
    buf = torch.zeros(4096, dtype=torch.float16)
    M, N, K, pitch = 8, 16, 24, 32
    base = buf.data_ptr() + (-buf.data_ptr()) % 16 - buf.data_ptr()
    at = lambda first, rows, cols, ld: buf.as_strided((rows, cols), (ld, 1), base // 2 + first)
    a = at(0, K, M, pitch).t()  # 23 * 32 + 8 elements
    b, c = at(2048, K, N, N), at(1024, M, N, N)
    gemm = _lib.GemmDesc(M=M, N=N, K=K, lda=pitch, ldb=N, ldc=N, in_dtype=_lib.F16, out_dtype=_lib.F16, flags=_lib.GEMM_A_COLUMNS)
    seen = []

    @C.CFUNCTYPE(C.c_int, C.POINTER(_lib.GemmDesc), C.c_void_p)
    def entry(g, stream):
        seen.append((g[0].A, g[0].C))
        return 0

    _launch.bind(table, ("columns",), (a, b, c), entry, (gemm,), "columns", gemm=gemm, c=(2, 0))
    for first, fits in ((1024, True), (0, False), (736, False), (744, True)):
        out = at(first, M, N, N)
        assert table.launch(("columns",), None, a, b, out) == (True if fits else None), first
        assert _launch._apart(a, out) == fits, first
    moved = at(128, K, M, pitch).t()  # C right before A, and one vector into it
    assert table.launch(("columns",), None, moved, b, at(0, M, N, N)) is True and _launch._apart(moved, at(0, M, N, N))
    assert table.launch(("columns",), None, moved, b, at(8, M, N, N)) is None and not _launch._apart(moved, at(8, M, N, N))
    assert len(seen) == 3
    # Three ranks' heaps, this one's in the middle: an A that starts in another's may be what the launch stores to that rank.
    heap = Heap(at(1024, 1, 1, 1), 2048)
    heap.all_ranks = (heap.local_base - 2048, 3 * 2048)
    _launch.bind(table, ("peers",), (at(1024, K, M, pitch).t(), b, c), entry, (gemm,), "columns", gemm=gemm, c=(2, 0), heap=heap, on_heap=0)
    behind = torch.zeros(8192, dtype=torch.float16)
    for first, fits in ((1024, True), (1016, None), (0, None), (2048, None), (3064, None), (3072, True)):
        out = behind.as_strided((M, N), (N, 1), -(behind.data_ptr() // 2) % 8)
        assert table.launch(("peers",), None, at(first, K, M, pitch).t(), b, out) == fits, first


@pytest.mark.parametrize("kind", ["sparse", "nested", "jagged", "vmap", "grad", "meta"])
def test_tensors_without_an_address_find_no_call(table, kind):
    """They throw when asked for one; that is "no call", and an ordinary error where a call is built for them."""
    table, _ = table
    a = torch.zeros(8, 8)
    seen, keep = bound(table, ("op",), (a, a), heap=Heap(a, 256))

    def asks(t):
        assert table.launch(("op",), None, a, t) is None
        assert table.launch(("op",), None, t, a) is None
        if kind != "meta":  # (whose address is zero)
            with pytest.raises(RuntimeError):
                bound(table, ("op",), (t, a))
        return t.sum() if kind in ("vmap", "grad") else None

    if kind == "sparse":
        asks(a.to_sparse())
    elif kind == "nested":
        asks(torch.nested.nested_tensor([a, a[:3]], layout=torch.strided))
    elif kind == "jagged":
        assert table.launch(("op",), None, a, torch.nested.nested_tensor([a, a[:3]], layout=torch.jagged)) is None
    elif kind == "vmap":
        torch.vmap(asks)(torch.zeros(3, 8, 8))
    elif kind == "grad":
        torch.func.grad(asks)(a)
    else:
        asks(torch.empty(8, 8, device="meta"))
    assert seen == [] and table.launch(("op",), None, a, a) is True


def test_operands_packed_into_something_without_an_address(table):
    table, _ = table
    a = torch.zeros(8, 8)
    host = _lib.host()

    @ENTRY
    def entry(*_):
        raise AssertionError("not reached")

    for packed in (a.to_sparse(), None):
        t = host.Table()
        t.add(host.Call(C.cast(entry, C.c_void_p).value, "entry", ((0, 0), 1, (1, 0)), (a, a), ("op",), prepare=lambda *_: (packed, a)))
        with pytest.raises((RuntimeError, TypeError)):
            t.launch(("op",), None, a, a)


def test_changed_signal_words_are_seen(table):
    """A bound call copies the words' descriptor; after a change of what that holds the call is built again, not launched."""
    table, _ = table
    fault = torch.zeros(1, dtype=torch.int64)
    words = _launch.SyncWords(locks=torch.zeros(4, dtype=torch.int32), arrivals=torch.zeros(4), fault=fault)
    seen = []

    @C.CFUNCTYPE(C.c_int, C.POINTER(_lib.SyncDescArrivals), C.c_void_p)
    def entry(sync, stream):
        seen.append((sync[0].locks, sync[0].trace_done_clock, sync[0].epoch))
        return 0

    a = torch.zeros(8)

    def call():
        if table.launch(("w",), None, a) is None:
            _launch.bind(table, ("w",), (a,), entry, (_launch.SYNC,), "w", words=words, variant="s1")
            return _launch.issue(table, ("w",), None, a) and "bound"
        return "known"

    assert [call(), call()] == ["bound", "known"] and len(table) == 1
    words.spin_limit_ns = 5  # read at every launch, like the launch number
    assert call() == "known" and seen[-1] == (words.locks.data_ptr(), None, 3)
    words.trace_done_clock = torch.zeros(4, dtype=torch.int64)
    assert [call(), call()] == ["bound", "known"] and len(table) == 1
    assert seen[-1] == (words.locks.data_ptr(), words.trace_done_clock.data_ptr(), 5)
    words.locks = torch.zeros(4, dtype=torch.int32)
    assert call() == "bound" and seen[-1] == (words.locks.data_ptr(), words.trace_done_clock.data_ptr(), 6)
    with pytest.raises(AttributeError):  # a plan's vectors are only changed with the plan
        _launch.DevicePlan(1, a, a, a, a).tile_counts = a


@pytest.mark.parametrize("variant,attr", [("s2", "epoch"), ("s1", "lock_epoch")])
def test_a_refused_launch_takes_no_number(table, variant, attr):
    table, _ = table
    words = _launch.SyncWords(locks=torch.zeros(4, dtype=torch.int32), arrivals=torch.zeros(4), fault=torch.zeros(1, dtype=torch.int64))
    numbers, answers = [], [0, _lib.ERR_UNSUPPORTED, _lib.ERR_INVALID, 0, 700, 0]

    @C.CFUNCTYPE(C.c_int, C.POINTER(_lib.SyncDescArrivals), C.c_void_p)
    def entry(sync, stream):
        numbers.append(sync[0].epoch)
        return answers[len(numbers) - 1]

    a = torch.zeros(8)
    _launch.bind(table, ("n",), (a,), entry, (_launch.SYNC,), "n", words=words, variant=variant)
    for rc in answers:
        if rc:
            with pytest.raises(ValueError if rc < 0 else RuntimeError):
                table.launch(("n",), None, a)
        else:
            assert table.launch(("n",), None, a) is True
    assert numbers == [1, 2, 2, 2, 3, 4]  # a HIP error may come after the launch: its number is gone
    assert getattr(words, attr) == 4 and words.epoch + words.lock_epoch == 4


def test_the_call_unused_for_longest_goes_first(table):
    host = _lib.host()
    table, keep = host.Table(3), []
    a = torch.zeros(8)

    def found(n):
        return table.launch(("op", n), None, a) is True

    with pytest.raises(ValueError):
        host.Table(0)
    for n in range(3):
        keep.append(bound_to(table, n, a))
    assert found(0)
    keep.append(bound_to(table, 3, a))
    assert [found(n) for n in range(4)] == [True, False, True, True]


def bound_to(table, n, t):
    @ENTRY
    def entry(*_):
        return 0

    _launch.bind(table, ("op", n), (t,), entry, ((0, 0), 1, 2), "entry")
    return entry


def test_a_program_that_goes_round_many_layouts_finds_its_calls(table):
    """Gradient buckets of 500 sizes, several times round: bound once each."""
    made = _launch.call_table({})
    buf = torch.zeros(1 << 12)
    keep = []
    for turn in range(3):
        for n in range(1, 501):
            t = buf[:n]
            if made.launch(("op", 0), None, t) is None:
                keep.append(bound_to(made, 0, t))
    assert len(keep) == len(made) == 500
