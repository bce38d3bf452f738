"""Iterations that search again only where a mean moved: frames on which most
means come to rest early while a few keep moving, through every form of the
search, bitwise alike and with the oracle's candidate slots after the last
iteration."""
import numpy as np
import pytest

import oracle_lib as O
from helpers import record_errors, records_equal
from tgmm_amd import em, synth

pytestmark = pytest.mark.gpu

TOL = 1e-5
SHAPES = [dict(knn_lanes=64), dict(knn_lanes=0, knn_block=128), dict(knn_lanes=1, knn_block=64),
          dict(knn_lanes=2, knn_cell=2), dict(knn_lanes=4, knn_chunk=4, knn_cell=4)]


def _resting():
    """1,200 cells, most of them alone, and eight with a second Gaussian close
    by, which share their supervoxels for many iterations."""
    f = synth.config1(seed=77, n_cells=1200, target_voxels=150000)
    extra = f.gm[100:900:100].copy()
    extra["m_k"] += np.array([1.2, -0.9, 0.2])
    extra["m_o"] = extra["m_k"]
    f.gm = np.concatenate([f.gm, extra]).astype(f.gm.dtype)
    return f


def _lattice():
    """Fixed Gaussians on a lattice (ties at the K-th distance for centroids
    between them) and six that move among them."""
    rng = np.random.default_rng(5)
    m = np.stack(np.meshgrid(*[np.arange(10.0) * 8] * 3, indexing="ij"), -1).reshape(-1, 3)
    gm = np.zeros(len(m), synth.GMM_DTYPE)
    gm["m_o"] = gm["m_k"] = m * np.array([1, 1, 0.2])
    for a in ("alpha", "beta"):
        gm[a + "_o"] = gm[a + "_k"] = 1.0
    gm["nu_o"] = gm["nu_k"] = 4.0
    gm["W_o"] = gm["W_k"] = np.array([0.04, 0, 0, 0.04, 0, 0.04])
    gm["fixed"] = 1
    moving = rng.choice(len(m), 6, replace=False)
    gm["fixed"][moving] = 0
    gm["m_k"][moving] += rng.normal(0, 1.0, (6, 3))
    S = 2500  # two-voxel supervoxels, most centroids midway between means
    c = rng.integers(0, 18, (S, 3)) * 4.0 * np.array([1, 1, 0.2])
    q = np.repeat(c, 2, 0)
    q[0::2, 0] -= 0.5
    q[1::2, 0] += 0.5
    img = rng.uniform(0.3, 1.0, 2 * S).astype(np.float32)
    return synth.Frame(np.ascontiguousarray(q.T.reshape(-1), np.float32), img,
                       np.ascontiguousarray(c.T.reshape(-1), np.float32),
                       2 * np.arange(S + 1, dtype=np.int64), gm)


@pytest.mark.parametrize("name", ["resting", "lattice"])
@pytest.mark.parametrize("K", [1, 5, 8, 11])
def test_look_iterations(name, K):
    f = _resting() if name == "resting" else _lattice()
    iters = 24
    outs = []
    for t in SHAPES:
        print("look %s K=%d %s" % (name, K, t), flush=True)
        with em.Batch([f, f], em.make_opts(K=K, max_iter=iters, scale=(1.0, 1.0, 5.0))) as b:
            b.set_tiles(dict(b.get_tiles(), **t))
            b.solve(em.SOLVE_GRAPH)
            b.reset()  # nothing of the first solve may be taken for the second
            b.solve(em.SOLVE_GRAPH)
            assert b.stats()["layout_mismatches"] == 0
            outs += b.fetch()
    for o in outs[1:]:
        assert records_equal(o["gm"], outs[0]["gm"]) and o["ll"] == outs[0]["ll"]
        assert np.array_equal(o["ind"], outs[0]["ind"])
        assert np.array_equal(o["rnk"], outs[0]["rnk"])
    gm_o, rnk_o, ind_o, hist, it, ll = O.em_run(f, O.make_opts(K=K, max_iter=iters))
    assert np.array_equal(outs[0]["ind"], ind_o)
    # (a lattice mean at the origin has no relative error: means compared here)
    assert np.allclose(outs[0]["gm"]["m_k"], gm_o["m_k"], rtol=TOL, atol=0)
    with np.errstate(invalid="ignore"):
        e = record_errors(outs[0]["gm"], gm_o)
    e.pop("m")
    assert max(e.values()) < TOL, e
