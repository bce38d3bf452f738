"""A server's workspace keeps to its budget: the capacity rule against the sum
of the workspace's arrays, through the library's own functions (no GPU), and
against the capacity that the estimate without this list gave."""
import ctypes
import os

import pytest

SO = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "tgmm_amd",
                  "libtgmm_em.so")
if not os.path.exists(SO):
    pytest.skip("libtgmm_em.so not built", allow_module_level=True)
L = ctypes.CDLL(SO)
_ll = ctypes.c_longlong


class Shape(ctypes.Structure):
    _fields_ = [("V", _ll), ("S", _ll), ("G", _ll), ("C", _ll), ("F", ctypes.c_int)]


ws_bytes = getattr(L, "_Z8ws_bytesRK7WsShapei")
ws_bytes.restype = _ll
ws_bytes.argtypes = [ctypes.POINTER(Shape), ctypes.c_int]
server_shape = getattr(L, "_Z12server_shapexii")
server_shape.restype = Shape
server_shape.argtypes = [_ll, ctypes.c_int, ctypes.c_int]


def _shape(V, F, K):
    up = lambda x, a: (x + a - 1) // a * a
    S, G = up(V // 8 + 256 * F, 256), up(V // 32 + 256 * F, 256)
    S = min(S, min((2 ** 31 - 1) >> 4, (2 ** 31 - 1) // K) // 256 * 256)
    return Shape(V, S, G, up(G // 2 + 128 * F, 64), F)


def _estimate(s, K):
    """The workspace's bytes by the sums of element sizes used before."""
    return (24 * s.V + s.S * (241 + 16 * K) + s.G * 1030 + 8 * s.C + 64 * s.F)


@pytest.mark.parametrize("K", [1, 5, 8, 16])
@pytest.mark.parametrize("F", [1, 4, 64, 4096])
def test_within_the_budget_and_hardly_smaller(K, F):
    least = 1 << 20
    floor = ws_bytes(ctypes.byref(_shape(least, F, K)), K)
    for b in range(28, 39):
        for part in (1.0, 1.1, 1.31, 1.66, 1.9):
            budget = int(part * (1 << b))
            s = server_shape(budget, F, K)
            assert (s.S, s.G, s.C) == tuple(getattr(_shape(s.V, F, K), n) for n in "SGC")
            took = ws_bytes(ctypes.byref(s), K)
            assert took <= max(budget, floor), (budget, s.V, took)
            V = least
            while 2 * V <= 1 << 31 and _estimate(_shape(2 * V, F, K), K) <= budget:
                V *= 2
            # no smaller than that, or than the budget allows (in steps of V/128)
            nxt = _shape(s.V + V // 128, F, K)
            assert s.V >= V or ws_bytes(ctypes.byref(nxt), K) > budget, (budget, s.V, V)
            if F <= 64:  # (with more slots their padding is most of a small workspace)
                assert s.V >= V * 15 // 16, (budget, s.V, V)


@pytest.mark.parametrize("K", [1, 5, 16])
@pytest.mark.parametrize("V", [22, 25, 29])
def test_just_where_a_doubling_was_accepted(K, V):
    for F in (1, 16, 512):
        t = _shape(1 << V, F, K)
        budget = _estimate(t, K)  # the doubling's arrays are a little more than this
        assert ws_bytes(ctypes.byref(t), K) > budget
        s = server_shape(budget, F, K)
        assert ws_bytes(ctypes.byref(s), K) <= budget
        assert t.V * 15 // 16 <= s.V <= t.V


@pytest.mark.parametrize("K", [1, 5, 8, 16])
@pytest.mark.parametrize("gb", [100, 150, 220, 280])
def test_indexes_stay_within_32_bits(K, gb):
    """A pair's code holds a supervoxel and a slot number, and the slots of all
    supervoxels are numbered, in 31 bits each."""
    for F in (1, 64):
        s = server_shape(gb << 30, F, K)
        assert (s.S << 4) < 1 << 31 and K * s.S < 1 << 31, s.S
        assert s.G < 1 << 31 and s.C < 1 << 31
