"""What a batch's workspace holds on the device is what the library counts for
its shape, in both modes and for several sizes and candidate counts."""
import ctypes

import pytest

from tgmm_amd import em, synth
from test_server_budget_cpu import Shape, ws_bytes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1, 5, 16])
@pytest.mark.parametrize("voxel", [False, True])
def test_workspace_bytes(K, voxel):
    fs = [synth.config1(seed=s, n_cells=n, target_voxels=200 * n) for s, n in
          ((1, 40), (2, 300), (3, 1000))]
    up = lambda x, a: (x + a - 1) // a * a
    S = [f.N if voxel else f.S for f in fs]
    G = [f.G for f in fs]
    sh = Shape(sum(f.N for f in fs), sum(up(s, 256) for s in S), sum(up(g + 1, 256) for g in G),
               sum(up(g // 2 + 64, 64) for g in G), len(fs))
    with em.Batch(fs, em.make_opts(K=K, max_iter=1, voxel=voxel)) as b:
        assert b.stats()["workspace_bytes"] == ws_bytes(ctypes.byref(sh), K)
