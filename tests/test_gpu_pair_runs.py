"""Pair lists past the LDS sort's length in many short runs: run counts around
a tile and a pass of the ranking, and lists with as many runs as pairs, whose
cost is bounded too."""
import time

import numpy as np
import pytest

import oracle_lib as O
from helpers import record_errors, records_equal
from tgmm_amd import em, synth
from test_gpu_pairlists import TOL, _frame

pytestmark = pytest.mark.gpu


def _alternating(a, n):
    """Two Gaussians far apart whose voxels alternate, `a` of one and `a` of
    the other, n times: n runs of `a` pairs each (a divides a wave)."""
    rng = np.random.default_rng(a * 100000 + n)
    i = np.arange(a * n)
    side = int(np.ceil((a * n) ** (1.0 / 3.0)))
    p = np.stack([i % side, i // side % side, i // (side * side) // 5], 1) + 50.0
    gm = np.zeros(2, synth.GMM_DTYPE)
    v = np.empty((2 * a * n, 3))
    for k in range(2):
        own = p + 400 * k
        v.reshape(n, 2, a, 3)[:, k] = own[rng.permutation(a * n)].reshape(n, a, 3)
        gm["m_o"][k] = gm["m_k"][k] = own.mean(0) + 0.3
    for f in ("alpha", "beta"):
        gm[f + "_o"] = gm[f + "_k"] = 1.0
    gm["nu_o"] = gm["nu_k"] = 4.0
    gm["W_o"] = gm["W_k"] = np.array([0.04, 0, 0, 0.04, 0, 0.04])
    q = np.ascontiguousarray(v.T.reshape(-1), np.float32)
    img = rng.uniform(0.2, 1.0, len(v)).astype(np.float32)
    return synth.Frame(q, img, q.copy(), np.arange(len(v) + 1, dtype=np.int64), gm)


@pytest.mark.parametrize("a,n", [(4, 2047), (4, 2048), (2, 2049), (2, 4096), (2, 4097), (1, 6001)])
def test_run_counts(a, n):
    f = _alternating(a, n)
    print("runs a=%d n=%d" % (a, n), flush=True)
    outs = []
    for lanes in (16, 4):
        with em.Batch([f], em.make_opts(K=2, max_iter=2, voxel=True)) as b:
            b.set_tiles(dict(b.get_tiles(), mstep_lanes=lanes))
            b.solve(em.SOLVE_GRAPH)
            outs.append(b.fetch()[0])
    gm_o = O.em_run(f, O.make_opts(K=2, max_iter=2, voxel=True))[0]
    e = record_errors(outs[0]["gm"], gm_o)
    assert max(e.values()) < TOL, e
    assert records_equal(outs[0]["gm"], outs[1]["gm"])


def test_scattered_lists_are_not_ranked_from_memory():
    """Four lists of 20,000 single-pair runs, five iterations: 20,000^2 / 256
    comparisons a thread. From memory these took 100 ms an iteration; through
    LDS, eight runs a thread and 24 instructions an entry, they are bounded by
    about 10. The line lies a factor of five above that."""
    f = _frame((20000,) * 4, True)
    print("scattered lists", flush=True)
    with em.Batch([f], em.make_opts(K=5, max_iter=5, voxel=True)) as b:
        best = 1e9
        for _ in range(3):
            b.reset()
            t = time.perf_counter()
            b.solve(em.SOLVE_GRAPH)
            best = min(best, time.perf_counter() - t)
    assert best < 5 * 0.05, best
