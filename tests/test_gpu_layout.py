"""The slot layout formed after the last iteration and the supervoxel lists of
the returned records: the lane-per-query and the wave-per-query replay against
the oracle's slots at Gaussian counts around a word of the mark bitmap, a
collected 64 and the first scan phase; the lists against a scan of the slots."""
import numpy as np
import pytest

import oracle_lib as O
from tgmm_amd import em, synth

pytestmark = pytest.mark.gpu


def _frame(G, S, seed):
    """S two-voxel supervoxels among G Gaussians, some of them alone with
    hundreds, some with none."""
    rng = np.random.default_rng(seed)
    span = 12.0 * max(G, 8) ** (1.0 / 3)
    gm = np.zeros(G, synth.GMM_DTYPE)
    m = rng.uniform(0, span, (G, 3)) * np.array([1, 1, 0.2])
    gm["m_o"] = gm["m_k"] = m
    for a in ("alpha", "beta"):
        gm[a + "_o"] = gm[a + "_k"] = 1.0
    gm["nu_o"] = gm["nu_k"] = 4.0
    gm["W_o"] = gm["W_k"] = np.array([0.02, 0, 0, 0.02, 0, 0.02])
    c = rng.uniform(0, span, (S, 3)) * np.array([1, 1, 0.2])
    near = rng.choice(G, min(G, 3), replace=False)  # long lists
    c[: S // 2] = m[near[rng.integers(0, len(near), S // 2)]] + rng.normal(0, 1.5, (S // 2, 3)) * [
        1, 1, 0.2]
    c = np.round(c * 64) / 64
    q = np.repeat(c, 2, 0)
    q[0::2, 0] -= 0.5
    q[1::2, 0] += 0.5
    img = rng.uniform(0.3, 1.0, 2 * S).astype(np.float32)
    return synth.Frame(np.ascontiguousarray(q.T.reshape(-1), np.float32), img,
                       np.ascontiguousarray(c.T.reshape(-1), np.float32),
                       2 * np.arange(S + 1, dtype=np.int64), gm)


def _lists(ind, rnk, G, cap):
    """The slot-major scan: per Gaussian, slot by slot, the supervoxels in
    increasing order with this candidate and r > 0.5."""
    out = [[] for _ in range(G)]
    for j in range(ind.shape[0]):
        for s in np.flatnonzero((rnk[j] > 0.5) & (ind[j] >= 0)):
            k = int(ind[j, s])
            if len(out[k]) < cap:
                out[k].append(int(s))
    return out


@pytest.mark.parametrize("K", [1, 5, 8, 11])
@pytest.mark.parametrize("G", [1, 63, 65, 1024, 1300])
def test_layout_and_lists(G, K):
    f = _frame(G, 1000, seed=31 * G + K)
    iters, cap = 6, {1: 16, 5: 10, 8: 1, 11: 0}[K]
    opts = em.make_opts(K=K, max_iter=iters, scale=(1.0, 1.0, 5.0), cap=cap)
    outs = []
    for n in (1, 25):  # 1,024 supervoxel places: a wave each; 25,600: a lane each
        print("layout G=%d K=%d frames=%d" % (G, K, n), flush=True)
        with em.Batch([f] * n, opts) as b:
            b.solve(em.SOLVE_GRAPH)
            assert b.stats()["layout_mismatches"] == 0
            got = b.fetch()
            outs += [got[0], got[-1]]
    ind_o = O.em_run(f, O.make_opts(K=K, max_iter=iters))[2]
    for o in outs:
        ind, rnk = np.asarray(o["ind"]).reshape(K, -1), np.asarray(o["rnk"]).reshape(K, -1)
        assert np.array_equal(ind, np.asarray(ind_o).reshape(K, -1))
        for k, want in enumerate(_lists(ind, rnk, G, cap)):
            r = o["gm"][k]
            assert r["supervoxelNum"] == len(want)
            assert list(r["supervoxelIdx"][: len(want)]) == want
