"""Which workgroups of a small-tile launch wait for another rank, and whether ranks that wait for each other always finish.

``finishes`` plays the launches of ranks through on the CUs they share (one rank: a GPU of its own): a workgroup is started
in the order of its number as soon as a CU of its XCD is free, one with a tile ends by itself, one that pulls ends
once every rank has finished its tiles.  The start order among the ranks is the worst one: whoever is first takes all it can."""

import ctypes as C

import pytest

CUS, XCDS = 256, 8


def grid(lib, tiles, world, pulls=1):
    first, wgs = C.c_int32(), C.c_int32()
    assert lib.tccl_stream_grid(tiles, pulls, CUS, world, C.byref(first), C.byref(wgs)) == 0
    return first.value, wgs.value


def finishes(launches, per_cu):
    """``launches``: per rank (workgroups, number of the first that waits, tiles); all on one device."""
    slots = CUS * per_cu // XCDS
    for_xcd = [[list(range(x, wgs, XCDS)) for x in range(XCDS)] for wgs, _, _ in launches]
    free = [slots] * XCDS
    tiles_left = [tiles for _, _, tiles in launches]
    waiting = [0] * XCDS
    while True:
        moved = False
        for r, (_, first, tiles) in enumerate(launches):
            for x in range(XCDS):
                while for_xcd[r][x] and free[x]:
                    wg = for_xcd[r][x].pop(0)
                    free[x] -= 1
                    if wg < tiles:  # its tile is done and published whether or not it then waits
                        tiles_left[r] -= 1
                    if wg >= first:
                        waiting[x] += 1
                    else:
                        free[x] += 1
                    moved = True
        if not any(tiles_left):
            return True  # what the others wait for is there
        if not moved:
            return False


@pytest.mark.parametrize("world", [2, 3, 4, 8])
def test_ranks_that_pull_from_each_other_finish(lib, world):
    for tiles in (*range(8, 264, 8), 328, 512, 520, 768, 1024):
        first, wgs = grid(lib, tiles, world)
        assert first == tiles < wgs  # no workgroup with a tile waits
        live = min(world, 4)  # launches of one process that can run at a time
        assert (wgs - first) * (live - 1) < CUS
        per_cu = 1 if tiles <= CUS else 2
        assert finishes([(wgs, first, tiles)] * live, per_cu), tiles
        assert grid(lib, tiles, world, pulls=0) == (tiles, tiles)


def test_what_the_rule_rules_out():
    """Workgroups that wait behind their own tile: not resident together (one rank's own GPU), and no place for a peer."""
    assert finishes([(512, 0, 512)], 2) and not finishes([(520, 0, 520)], 2)
    assert finishes([(224, 0, 224)], 1) and not finishes([(256, 0, 256)] * 2, 1)


@pytest.mark.parametrize("bad", [(0, 1, 256, 2), (8, 1, 0, 2), (8, 1, 256, 0), (8, 1, 256, 9)])
def test_bad_arguments(lib, bad):
    first, wgs = C.c_int32(), C.c_int32()
    assert lib.tccl_stream_grid(*bad, C.byref(first), C.byref(wgs)) != 0
    assert lib.tccl_stream_grid(8, 1, 256, 2, None, C.byref(wgs)) != 0
