"""Frames on which looking for queries to search again stops paying: many slots
on grids of small cells, where a query's K nearest reach past its block of
cells, beside a frame in the same batch that goes on looking. Bitwise as the
wave-per-query form, which looks query by query, and as the oracle's slots."""
import numpy as np
import pytest

import oracle_lib as O
from helpers import records_equal
from tgmm_amd import em, synth
from test_gpu_knn_look import _resting

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [8, 16])
@pytest.mark.parametrize("lanes", [0, 1, 2, 4])
def test_looks_that_stop(K, lanes):
    fs = [_resting(), synth.config1(seed=3, n_cells=40, target_voxels=6000)]
    outs = []
    for t in (dict(knn_lanes=64, knn_cell=6), dict(knn_lanes=lanes, knn_cell=2)):
        print("look stop K=%d %s" % (K, t), flush=True)
        with em.Batch(fs, em.make_opts(K=K, max_iter=24, scale=(1.0, 1.0, 5.0))) as b:
            b.set_tiles(dict(b.get_tiles(), **t))
            for mode in (em.SOLVE_GRAPH, em.SOLVE_EAGER):
                b.solve(mode)
                assert b.stats()["layout_mismatches"] == 0
                outs.append(b.fetch())
                b.reset()  # and looks again in the next solve
    for o in outs[1:]:
        for x, y in zip(o, outs[0]):
            assert records_equal(x["gm"], y["gm"]) and x["ll"] == y["ll"]
            assert np.array_equal(x["ind"], y["ind"]) and np.array_equal(x["rnk"], y["rnk"])
    for f, o in zip(fs, outs[0]):
        ind_o = O.em_run(f, O.make_opts(K=K, max_iter=24))[2]
        assert np.array_equal(o["ind"], ind_o)
