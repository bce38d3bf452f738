"""The launch shapes chosen where none are set (tgmm::tiles_for), through the
library on the CPU: the sizes on either side of each line, and that every
choice is a valid one."""
import ctypes
import itertools
import os

import pytest

SO = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "tgmm_amd",
                  "libtgmm_em.so")
if not os.path.exists(SO):
    pytest.skip("libtgmm_em.so not built", allow_module_level=True)
L = ctypes.CDLL(SO)
FIELDS = ("ll_gw", "ll_u", "ms_lanes", "sv_block", "knn_block", "knn_chunk", "knn_cell",
          "knn_lanes")


class Tiles(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int) for n in FIELDS]


tiles_for = getattr(L, "_ZN4tgmm9tiles_forExxib")
tiles_for.restype = Tiles
tiles_for.argtypes = [ctypes.c_longlong, ctypes.c_longlong, ctypes.c_int, ctypes.c_bool]
tiles_valid = getattr(L, "_ZN4tgmm11tiles_validERKNS_5TilesE")
tiles_valid.restype = ctypes.c_bool


def test_lines():
    ms = lambda S, G: tiles_for(S, G, 5, False).ms_lanes
    assert [ms(S, 1000) for S in (0, 5999, 6000, 31999, 32000)] == [4, 4, 8, 8, 16]
    knn = lambda S, K: tiles_for(S, 1000, K, False).knn_lanes
    assert [knn(S, 5) for S in (900, 12288, 12289, 65536, 65537, 299999, 300000)] == [
        64, 64, 4, 4, 2, 2, 1]
    assert [knn(S, 8) for S in (12289, 16384, 16385)] == [64, 64, 4]
    assert tiles_for(7359, 640, 5, False).ms_lanes == 8  # 32 frames of 20 Gaussians


def test_every_choice_is_valid():
    for S, G, K, v in itertools.product((0, 1, 900, 13000, 70000, 200000, 1 << 26),
                                        (0, 1, 200, 60000), (1, 5, 8, 16), (False, True)):
        t = tiles_for(S, G, K, v)
        assert tiles_valid(ctypes.byref(t)), (S, G, K, v)
