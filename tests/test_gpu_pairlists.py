"""The M-step's pair lists at the lengths where their ordering changes form:
single pairs, the edges of the short and the long sort and of the LDS
capacity, with the voxels of a Gaussian in one run or scattered over the
frame. The oracle's tolerance is that of the per-voxel parity tests."""
import numpy as np
import pytest

import oracle_lib as O
from helpers import record_errors, records_equal, rel_err
from tgmm_amd import em, synth

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _frame(sizes, shuffled):
    rng = np.random.default_rng(11)
    pts, gm = [], np.zeros(len(sizes), synth.GMM_DTYPE)
    for k, n in enumerate(sizes):  # compact clusters 400 apart
        side = int(np.ceil(n ** (1.0 / 3.0)))
        c = np.array([(400 * (k % 4)), 400 * (k // 4 % 4), 80 * (k // 16)]) + 50
        i = np.arange(n)
        p = np.stack([i % side, i // side % side, i // (side * side) // 5], 1) + c
        pts.append(p)
        gm["m_o"][k] = gm["m_k"][k] = p.mean(0) + rng.normal(0, 0.5, 3)
    for a in ("alpha", "beta"):
        gm[a + "_o"] = gm[a + "_k"] = 1.0
    gm["nu_o"] = gm["nu_k"] = 4.0
    gm["W_o"] = gm["W_k"] = np.array([0.04, 0, 0, 0.04, 0, 0.04])
    p = np.concatenate(pts).astype(np.float32)
    if shuffled:
        p = p[rng.permutation(len(p))]
    q = np.ascontiguousarray(p.T.reshape(-1))
    img = rng.uniform(0.2, 1.0, len(p)).astype(np.float32)
    return synth.Frame(q, img, q.copy(), np.arange(len(p) + 1, dtype=np.int64), gm)


@pytest.mark.parametrize("sizes", [(1, 2, 15, 16, 17, 127, 128, 129, 511, 512, 513, 1025),
                                   (5, 300, 4095, 4096, 4097, 6000)])
@pytest.mark.parametrize("shuffled", [False, True])
def test_pair_list_lengths(sizes, shuffled):
    f = _frame(sizes, shuffled)
    print("pair lists %s shuffled=%d N=%d" % (sizes, shuffled, f.N), flush=True)
    outs = []
    for lanes in (16, 4):
        with em.Batch([f], em.make_opts(K=5, max_iter=2, voxel=True)) as b:
            b.set_tiles(dict(b.get_tiles(), mstep_lanes=lanes))
            b.solve(em.SOLVE_GRAPH)
            outs.append(b.fetch()[0])
    gm_o, rnk_o, ind_o, hist, it, ll = O.em_run(f, O.make_opts(K=5, max_iter=2, voxel=True))
    e = record_errors(outs[0]["gm"], gm_o)
    assert max(e.values()) < TOL, e
    assert rel_err(outs[0]["ll"], ll) < TOL
    assert np.max(np.abs(outs[0]["rnk"] - rnk_o)) < 2e-6
    assert records_equal(outs[0]["gm"], outs[1]["gm"])
