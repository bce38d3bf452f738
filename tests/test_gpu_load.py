"""The workspace's tables and state columns formed on the device: frames whose
supervoxel and Gaussian counts lie around the ranges' 256, 64 and 16, together
in one batch in several orders, with the records, flags and lists of each frame
the same as alone and as the oracle's."""
import numpy as np
import pytest

import oracle_lib as O
from helpers import record_errors, records_equal
from tgmm_amd import em
from test_gpu_layout import _frame

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (255, 16), (256, 255), (257, 256), (512, 15), (0, 5), (40, 17), (300, 64)]


def _frames():
    out = []
    for i, (S, G) in enumerate(SIZES):
        f = _frame(G, max(S, 1), seed=400 + i)
        if S == 0:
            f.query, f.img, f.centroids = (x[:0].copy() for x in (f.query, f.img, f.centroids))
            f.sv_ptr = np.zeros(1, np.int64)
        f.gm["fixed"][::3] = 1
        f.gm["supervoxelIdx"] = np.arange(16) + 100 * np.arange(G)[:, None]
        f.gm["supervoxelNum"] = np.arange(G) % 17
        out.append(f)
    return out


@pytest.mark.parametrize("voxel", [False, True])
@pytest.mark.parametrize("shift", [0, 3])
def test_frames_around_range_ends(shift, voxel):
    fs = _frames()
    fs = fs[shift:] + fs[:shift]
    opts = em.make_opts(max_iter=4, voxel=voxel)
    print("load shift %d voxel %d" % (shift, voxel), flush=True)
    with em.Batch(fs, opts) as b:
        b.solve(em.SOLVE_GRAPH)
        together = b.fetch()
    for f, got in zip(fs, together):
        with em.Batch([f], opts) as b:
            b.solve(em.SOLVE_GRAPH)
            alone = b.fetch()[0]
        assert records_equal(got["gm"], alone["gm"]) and got["ll"] == alone["ll"]
        assert np.array_equal(got["ind"], alone["ind"])
        gm_o, rnk_o, ind_o, hist, it, ll = O.em_run(f, O.make_opts(max_iter=4, voxel=voxel))
        assert np.array_equal(got["gm"]["fixed"], f.gm["fixed"])
        if voxel:  # the lists come back as given
            assert np.array_equal(got["gm"]["supervoxelIdx"], f.gm["supervoxelIdx"])
            assert np.array_equal(got["gm"]["supervoxelNum"], f.gm["supervoxelNum"])
        if f.N > 0:
            e = record_errors(got["gm"], gm_o)
            assert max(e.values()) < 1e-5, e


@pytest.mark.parametrize("G", [4095, 4096, 8193, 33000])
def test_scans_around_a_segment(G):
    """The scans of cells and pair lists at one segment of 4,096 entries, one
    entry more, several, and a second pass of eight, beside a small frame."""
    small, f = _frame(3, 64, seed=1), _frame(G, 1500, seed=G)
    print("scan G=%d" % G, flush=True)
    with em.Batch([small, f], em.make_opts(max_iter=3)) as b:
        b.solve(em.SOLVE_GRAPH)
        got = b.fetch()[1]
    gm_o, rnk_o, ind_o, hist, it, ll = O.em_run(f, O.make_opts(max_iter=3))
    assert np.array_equal(got["ind"], ind_o)
    e = record_errors(got["gm"], gm_o)
    assert max(e.values()) < 1e-5, e
