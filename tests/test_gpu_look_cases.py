"""Iterations that look for queries to search again, in two situations: a
Gaussian dies while few means move, so that the look finds its place left; and
frames served together at different iterations, of which some look and others
search whole."""
import numpy as np
import pytest

import oracle_lib as O
from helpers import record_errors, records_equal
from tgmm_amd import em, synth
from tgmm_amd.records import is_dead
from test_gpu_knn_look import _resting

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _starving():
    """500 settled cells of one-voxel supervoxels, held fixed but one, and a
    second Gaussian on that one, which loses its voxels over five iterations
    and dies; at most three means move in an iteration."""
    f = synth.config1(seed=77, n_cells=500, target_voxels=25000)
    f = synth.Frame(f.query, f.img, f.query.copy(), np.arange(f.N + 1, dtype=np.int64), f.gm)
    gm = O.em_run(f, O.make_opts(K=5, max_iter=6))[0]
    gm["fixed"] = 1
    gm["fixed"][180] = 0
    extra = gm[180:181].copy()
    extra["alpha_o"] = extra["beta_o"] = 1e-9
    extra["alpha_k"] = 12.0
    f.gm = np.concatenate([gm, extra]).astype(f.gm.dtype)
    return f


@pytest.mark.parametrize("lanes", [0, 1, 2, 4, 64])
def test_a_gaussian_dies_during_looks(lanes):
    f, iters = _starving(), 12
    early = O.em_run(f, O.make_opts(K=5, max_iter=3))[0]
    gm_o, rnk_o, ind_o, hist, it, ll = O.em_run(f, O.make_opts(K=5, max_iter=iters))
    assert not is_dead(early)[-1] and is_dead(gm_o)[-1]
    print("death, lanes %d" % lanes, flush=True)
    with em.Batch([f], em.make_opts(K=5, max_iter=iters)) as b:
        b.set_tiles(dict(b.get_tiles(), knn_lanes=lanes))
        if lanes != 64:  # it dies in an iteration that looks
            S, G = f.S, f.G
            assert b.time_kernel("knn", iters)[1] < 0.5 * (S * (16 + 8 * 5) + 32 * G)
            b.reset()
        b.solve(em.SOLVE_GRAPH)
        assert b.stats()["layout_mismatches"] == 0
        o = b.fetch()[0]
    assert is_dead(o["gm"])[-1] and np.array_equal(o["ind"], ind_o)
    assert not (o["ind"] == f.G - 1).any()
    e = record_errors(o["gm"], gm_o)
    assert max(e.values()) < TOL, e


@pytest.mark.parametrize("lanes,cell", [(2, 6), (4, 2), (64, 6)])
def test_served_frames_at_different_iterations(lanes, cell):
    opts = em.make_opts(K=8, max_iter=20)
    fs = [_resting(), synth.config1(seed=12, n_cells=300, target_voxels=60000), _resting()]
    fs[2].gm["m_k"] += 0.5
    print("served looks lanes %d cell %d" % (lanes, cell), flush=True)
    with em.Server(opts, hbm_budget_bytes=1 << 30, max_frames_in_flight=3) as s:
        s.set_tiles(dict(em.DEFAULT_TILES, knn_lanes=lanes, knn_cell=cell))
        tickets = []
        for f in fs:  # seven iterations apart
            tickets.append(s.submit(f))
            for _ in range(7):
                s.step()
        s.wait(-1)
        got = [s.fetch(t, f.G) for t, f in zip(tickets, fs)]
    for f, o in zip(fs, got):
        with em.Batch([f], opts) as b:
            b.solve(em.SOLVE_GRAPH)
            want = b.fetch()[0]
        assert records_equal(o["gm"], want["gm"]) and o["ll"] == want["ll"]
        assert np.array_equal(o["ind"], want["ind"]) and np.array_equal(o["rnk"], want["rnk"])
