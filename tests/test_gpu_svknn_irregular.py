"""Neighbour searches with a few coordinates that are not finite (or beyond
1e18) among raster-ordered centroids, where the other blocks of references are
left out: in one block, in several, in the last partial one, in a query, in
both, with scales of either sign, slot for slot as the oracle's scan."""
import numpy as np
import pytest

from test_gpu_svknn import _check, _raster

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [63, 64, 65, 4161, 20000])
@pytest.mark.parametrize("where", ["ref", "refs", "query", "both"])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf, 3e18])
def test_irregular_coordinates(R, where, bad):
    rng = np.random.default_rng(R)
    span = 8.0 * R ** (1.0 / 3)
    r = _raster(rng.uniform(0, span, (3, R)) * [[1], [1], [0.2]]).astype(np.float32)
    q = _raster(rng.uniform(0, span, (3, 777)) * [[1], [1], [0.2]]).astype(np.float32)
    if where in ("ref", "both"):
        r[R % 3, R // 2] = bad
    if where == "refs":
        r[0, ::997] = bad
        r[1, R - 1] = bad
    if where in ("query", "both"):
        q[1, 300] = bad
        q[2, 776] = bad
    print("svknn irregular R=%d %s %s" % (R, where, bad), flush=True)
    q, r = np.ascontiguousarray(q).reshape(-1), np.ascontiguousarray(r).reshape(-1)
    _check(q, r, 11)
    _check(q, r, 1, scale=(-1.0, 2.0, -3.0))


@pytest.mark.parametrize("Q", [65535, 65536, 65601])
def test_both_sides_of_the_kernel_choice(Q):
    rng = np.random.default_rng(Q)
    q = rng.uniform(0, 40, (3, Q)).astype(np.float32)
    r = _raster(rng.uniform(0, 40, (3, 300))).astype(np.float32)
    r[2, 130] = np.nan
    q[0, Q - 1] = np.inf
    print("svknn irregular Q=%d" % Q, flush=True)
    _check(q.reshape(-1), np.ascontiguousarray(r).reshape(-1), 4)
