"""The slab entries that the row-finishing query-gradient kernel asks for, walked on the host with the kernel's own arithmetic
(smx_measure_slab_walk): an entry that is asked for is used as a row's address, so each has to be one of the slab's 64."""
import ctypes
import random

import pytest

from smore_amd import _lib


def walk(cnt, singles, rif):
    place, taken = (ctypes.c_int * 64)(), (ctypes.c_int * 64)()
    low, high = ctypes.c_int(), ctypes.c_int()
    rc = _lib.load().smx_measure_slab_walk(cnt, singles, rif, place, taken, ctypes.byref(low), ctypes.byref(high))
    assert rc == 0
    return list(place), [t for t in taken if t >= 0], low.value, high.value


@pytest.mark.parametrize("rif", [1, 2, 4])
def test_every_entry_asked_for_exists(rif):
    rng = random.Random(rif)
    for cnt in range(1, 65):
        for n in range(cnt + 1):
            front = (1 << n) - 1
            drawn = sum(1 << i for i in rng.sample(range(cnt), n))
            for singles in {front, front << (cnt - n), drawn}:
                place, taken, low, high = walk(cnt, singles, rif)
                assert sorted(place) == list(range(64)) and place[cnt:] == list(range(cnt, 64))
                lane_of = {p: lane for lane, p in enumerate(place)}
                others = [lane for lane in range(cnt) if not singles >> lane & 1]
                assert [lane_of[t] for t in taken] == others, "each of the others once, in pair order"
                ones = [lane for lane in range(cnt) if singles >> lane & 1]
                assert [lane_of[p] for p in range(cnt - n, cnt)] == ones, "the rows to finish are the last n, in pair order"
                if others:
                    assert low == 0 and high < 64
