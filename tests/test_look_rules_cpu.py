"""The rules of the kNN search's looks (tgmm_amd/csrc/tgmm_device.h), built for
the host: when an iteration looks, when its list is searched by waves, and when
a look was futile, at the edges of each line. Runs without a GPU."""
import ctypes
import os

import pytest

SO = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "libdevmath_host.so")
if not os.path.exists(SO):
    pytest.skip("tests/native/libdevmath_host.so not built", allow_module_level=True)
D = ctypes.CDLL(SO)
_ll = ctypes.c_longlong
D.dm_look_due.argtypes = [ctypes.c_int, ctypes.c_int, _ll, _ll]
D.dm_look_few.argtypes = [_ll, _ll]
D.dm_look_futile.argtypes = [_ll, _ll]


def test_a_look_is_due():
    assert D.dm_look_due(1, 0, 0, 1000) == 0  # the first iteration searches whole
    assert D.dm_look_due(2, 0, 0, 1000) == 1
    assert D.dm_look_due(2, 0, 10, 1280) == 1
    assert D.dm_look_due(2, 0, 11, 1280) == 0
    assert D.dm_look_due(2, 1, 0, 1280) == 0  # an earlier one was futile


@pytest.mark.parametrize("ns", [1, 15, 16, 17, 1600, 1 << 27])
def test_looks_stop_where_the_unmoved_alone_are_too_many(ns):
    """Queries listed whatever moved stay listed: past the line a look ends in
    the whole search, and so would every later one."""
    line = ns // 16
    assert D.dm_look_few(line, ns) == 1 and D.dm_look_few(line + 1, ns) == 0
    assert D.dm_look_futile(line, ns) == 0 and D.dm_look_futile(line + 1, ns) == 1


def iterations_that_look(stuck, moved, ng, ns):
    """The frame's iterations as the kernels step the state: the look lists the
    stuck queries and 2K = 16 of a moved mean's."""
    blind, looks = 0, []
    for it, mv in enumerate(moved, 1):
        if not D.dm_look_due(it, blind, mv, ng):
            continue
        looks.append(it)
        if D.dm_look_futile(stuck, ns):
            blind = 1
    return looks


def test_a_frame_of_small_cells_looks_once():
    moved = [60000, 9000, 3000, 400, 100] + [20] * 20
    assert iterations_that_look(200000, moved, 60000, 660000) == [4]
    assert iterations_that_look(2000, moved, 60000, 660000) == list(range(4, 26))
