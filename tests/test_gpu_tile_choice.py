"""The launch shapes a batch and a server start with: chosen by what the frames
hold, not by the padded ranges; shapes set on a server stay when its ranges
grow; results are bitwise the same with either."""
import numpy as np
import pytest

from helpers import records_equal
from tgmm_amd import em, synth

pytestmark = pytest.mark.gpu


def _frames(n):
    out = [synth.config1(seed=70 + i, n_cells=20, target_voxels=10000) for i in range(n)]
    assert all(9 < f.S / f.G < 14 for f in out)  # 256-padded they seem to hold 1 to 2
    return out


def test_small_frames_are_not_taken_for_their_padding():
    with em.Batch(_frames(32), em.make_opts(K=5, max_iter=2)) as b:
        assert b.get_tiles()["mstep_lanes"] == 8


@pytest.mark.parametrize("tiles", [None, dict(em.DEFAULT_TILES, mstep_lanes=16, knn_lanes=1)])
def test_server_shapes_while_ranges_grow(tiles):
    opts = em.make_opts(K=5, max_iter=6)
    fs = _frames(2) + [synth.config1(seed=5, n_cells=150, target_voxels=30000)] + _frames(1)
    print("server tiles", tiles, flush=True)
    with em.Server(opts, hbm_budget_bytes=1 << 30, max_frames_in_flight=4) as s:
        if tiles:
            s.set_tiles(tiles)
        tickets = []
        for f in fs:  # each joins while the ones before are in flight
            tickets.append(s.submit(f))
            s.step()
        s.wait(-1)
        got = [s.fetch(t, f.G) for t, f in zip(tickets, fs)]
    for f, o in zip(fs, got):
        with em.Batch([f], opts) as b:
            b.solve(em.SOLVE_GRAPH)
            want = b.fetch()[0]
        assert records_equal(o["gm"], want["gm"]) and o["ll"] == want["ll"]
        assert np.array_equal(o["ind"], want["ind"])
