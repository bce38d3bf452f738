"""Neighbour searches of more queries than are searched for together: a partial
second piece, and a call of 2^30 queries, which one launch with four lanes a
query cannot cover."""
import os

import numpy as np
import pytest

from tgmm_amd import em
from test_gpu_svknn import SCALE, _check

pytestmark = pytest.mark.gpu

PIECE = 1 << 22


@pytest.mark.parametrize("extra", [-1, 1, 70001])
@pytest.mark.parametrize("bad", [False, True])
def test_around_a_piece(extra, bad):
    Q = PIECE + extra
    rng = np.random.default_rng(Q)
    q = rng.uniform(0, 30, (3, Q)).astype(np.float32)
    r = rng.uniform(0, 30, (3, 37)).astype(np.float32)
    if bad:
        q[0, 5] = q[1, Q - 1] = r[2, 3] = np.nan
    print("svknn pieces Q=%d bad=%d" % (Q, bad), flush=True)
    _check(q.reshape(-1), r.reshape(-1), 2)


def test_two_to_the_thirty_queries():
    if os.sysconf("SC_PAGE_SIZE") * os.sysconf("SC_AVPHYS_PAGES") < 64 << 30:
        pytest.skip("24 GB of host arrays")
    Q = (1 << 30) + 3
    q = np.zeros(3 * Q, np.float32)  # on the x axis: 0, 1, .. 7, 0, 1, ..
    q[: Q - 3].reshape(-1, 8)[:] = np.arange(8)
    print("svknn 2^30 queries", flush=True)
    ind, dist = em.knnCUDA_(q, np.array([6, 1, 0, 0, 0, 0], np.float32), 1, SCALE,
                            with_dist=False)
    want = np.array([1, 1, 1, 1, 0, 0, 0, 0])  # the nearer of x = 6 and x = 1
    got = ind[: Q - 3].reshape(-1, 8)
    assert np.array_equal(ind[Q - 3:], [1, 1, 1]) and dist is None
    assert all((got[a: a + (1 << 20)] == want).all() for a in range(0, len(got), 1 << 20))
